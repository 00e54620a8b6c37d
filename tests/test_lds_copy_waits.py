"""Global-to-LDS copies written as inline asm take their LDS address from M0.  The hardware needs one wait state between
a scalar write of M0 and such a copy, and the compiler's hazard pass does not look inside inline asm: every asm text that
writes M0 holds the wait itself."""
import re
from pathlib import Path

import seedplane_amd

SOURCES = sorted((Path(seedplane_amd.__file__).parent / 'csrc').glob('*.h*'))


def test_every_m0_write_is_followed_by_a_wait_state():
    copies = 0
    for f in SOURCES:
        for text in re.findall(r'asm\s+volatile\s*\(\s*"([^"]*)"', f.read_text()):
            lines = [x.strip() for x in text.replace('\\t', ' ').split('\\n')]
            for i, x in enumerate(lines):
                if re.match(r's_\w+ m0\b', x):
                    copies += 1
                    assert i + 1 < len(lines) and re.match(r's_nop \d+$', lines[i + 1]), (f.name, text)
                if 'load_lds' in x:
                    assert i > 0 and lines[i - 1].startswith('s_nop'), (f.name, text)
    assert copies >= 3
