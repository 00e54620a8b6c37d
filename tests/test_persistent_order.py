"""Host bookkeeping of the persistent step (sp_order.h), compiled for the CPU: the error word is reported once per launch
even if late blocks set it again."""
import subprocess
from pathlib import Path

import seedplane_amd

CSRC = Path(seedplane_amd.__file__).parent / 'csrc'

PROGRAM = r'''
#include <cstdio>
#include "sp_order.h"

static int bad = 0;
int main() {
    // a block reports, the host looks, later blocks of the same launch report again before the stream is idle
    unsigned word = 1;
    int waits = 0;
    const bool first = sp::take_error(&word, [&] { ++waits; word = 1; });
    const bool again = sp::take_error(&word, [&] { ++waits; });
    if (!first || again || waits != 1 || word != 0) { std::printf("error word\n"); ++bad; }
    if (sp::take_error(nullptr, [&] { ++waits; }) || waits != 1) { std::printf("no word\n"); ++bad; }
    return bad;
}
'''


def test_error_word(tmp_path):
    src, exe = tmp_path / 'order.cpp', tmp_path / 'order'
    src.write_text(PROGRAM)
    subprocess.run(['g++', '-std=c++17', '-Wall', '-Werror', '-I', str(CSRC), str(src), '-o', str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
