"""The wide prefill pass (sp_engine_prefill, behind forward / generate / prefill for prompts longer than max_tokens)
against the CPU oracle: every weight format and head size, column counts at the edges of the product tiles (64 and 128
columns) and of a pass (2048), windowed rings that the prompt wraps, runs of several sequences, and the calls it
refuses.  Tolerance: the fp16-class bar, max |a - b| / max |b| < 2e-2 per row; K/V are fp16 of values of that class."""
import ctypes

import numpy as np
import pytest
import torch

from oracle.qwen_ref import RefQwen2
from seedplane_amd import _lib
from seedplane_amd.presets import preset
from seedplane_amd.qwen_engine import Qwen2Engine
from seedplane_amd.synth import make_weights, random_prompt
from tests.conftest import small_cfg
from tests.parity import TOL, check_greedy, check_rows

pytestmark = pytest.mark.gpu


def _engine(shape, fmt, max_tokens=64):
    cfg = (small_cfg(max_position_embeddings=8192) if shape == 'small' else
           preset(shape, num_hidden_layers=2, vocab_size=1000))
    cfg, w = make_weights(cfg, fmt, seed=5, scale_std=0.0005)
    return cfg, Qwen2Engine(config=cfg, tensors=w, max_tokens=max_tokens), RefQwen2(cfg, w)


def _close_kv(got, want, n, what):
    for g, r in zip(got, want):
        g, r = g[0, :n].float().cpu(), r[0, :n]
        assert float((g - r).abs().max()) < TOL * float(r.abs().max()), what


@pytest.mark.parametrize('shape,fmt,n,window', [
    ('small', 'f16', 65, None), ('small', 'q8', 127, None), ('small', 'q4', 129, None), ('small', 'q8', 640, 100),
    ('small', 'q4', 2048, 64), ('small', 'f16', 2049, 200), ('qwen2-0.5b', 'f16', 193, None),
    ('qwen2-1.5b', 'q8', 257, 65), ('qwen2-7b', 'q4', 100, None)])
def test_prompt_logits_and_cache_match_oracle(gpu_device, shape, fmt, n, window):
    print(f'prefill {shape} {fmt} n={n} window={window}', flush=True)
    cfg, eng, ref = _engine(shape, fmt)
    ids = random_prompt(n, cfg['vocab_size'], seed=n)
    rc = ref.new_cache(n + 8)
    want = ref.forward(ids, rc, all_logits=True, window=window)
    cache = eng.new_cache(n + 8, window=window)
    rows, _ = eng.forward(ids, cache, all_logits=True)
    check_rows(rows.cpu(), want, what='all logits')
    assert cache.length == n
    last, c2 = eng.forward(ids, eng.new_cache(n + 8, window=window))      # only the last column leaves the last layer
    check_rows(last.cpu(), want[-1:], what='last logits')
    first = 0 if window is None else max(0, n - window - eng.max_tokens)  # positions the ring still holds
    for c in (cache, c2):
        for l in range(cfg['num_hidden_layers']):
            _close_kv([c.keys[l][:, first:], c.values[l][:, first:]],
                      [rc.keys[l][:, first:], rc.values[l][:, first:]], n - first, f'layer {l}')
    # the cache goes on: a second prompt on top of the first, then a decode step
    more = random_prompt(70, cfg['vocab_size'], seed=1)
    c2.capacity = n + 80
    if window is not None:
        want2 = ref.forward(ids + more, ref.new_cache(n + 80), all_logits=True, window=window)
        got, _ = eng.forward(more, c2)
        check_rows(got.cpu(), want2[-1:], what='second prompt')


def test_prompts_of_several_sequences(gpu_device):
    """Ragged prompts in one call: more columns than one pass, more prompts than max_tokens, an empty prompt."""
    cfg, eng, ref = _engine('small', 'q8', max_tokens=4)
    lens = [3, 900, 1, 0, 64, 700, 65, 2, 700]
    prompts = [random_prompt(k, cfg['vocab_size'], seed=i) for i, k in enumerate(lens)]
    eng.reserve(len(lens), 960)
    caches = [eng.new_cache(950) for _ in lens]
    got = eng.prefill(prompts, caches)
    for p, c, t in zip(prompts, caches, got):
        assert c.length == len(p)
        if not p:
            assert t is None
            continue
        rc = ref.new_cache(len(p) + 1)
        row = ref.forward(p, rc)
        check_greedy([t], [row[-1]], what=f'{len(p)} tokens')
        _close_kv([c.keys[-1], c.values[-1]], [rc.keys[-1], rc.values[-1]], len(p), f'{len(p)} tokens')


def test_rotary_positions_and_rollback(gpu_device):
    cfg, eng, ref = _engine('small', 'f16')
    ids = random_prompt(150, cfg['vocab_size'], seed=9)
    a, cache = eng.forward(ids, eng.new_cache(400), positions=[p + 17 for p in range(150)])
    b, _ = eng.forward(ids, eng.new_cache(400))
    check_rows(a.cpu(), b.cpu(), what='a common shift')          # attention depends on position differences only
    c, _ = eng.forward(ids, eng.new_cache(400), positions=[3 * p for p in range(150)])
    assert float((b - c).abs().max()) > 1e-3
    cache.length = 0                                             # rolled back: the same prompt again
    d, _ = eng.forward(ids, cache)
    assert torch.equal(d, b)


def test_refused_calls(gpu_device):
    cfg, eng, _ = _engine('small', 'q8')
    eng.reserve(2, 300)
    c0, c1 = eng.new_cache(200), eng.new_cache(200)
    cols = lambda: np.concatenate([eng._prompt_columns([1] * 40, c0, 0), eng._prompt_columns([2] * 40, c1, 0)])
    out = np.array([79], dtype=np.int32)
    buf = torch.empty((1, eng.vocab), device=eng.device)

    def call(a, out=out, dst=buf, ids=None):
        return eng.lib.sp_engine_prefill(eng.h, len(a), ctypes.c_void_p(a.ctypes.data), len(out),
                                         ctypes.c_void_p(out.ctypes.data),
                                         ctypes.c_void_p(dst.data_ptr()) if dst is not None else None,
                                         ctypes.c_void_p(ids.ctypes.data) if ids is not None else None)

    def broken(field, i, v):
        a = cols()
        a[field][i] = v
        return a

    assert call(cols()) == _lib.SP_OK
    for a in (broken('ctx_hi', 5, 7), broken('slot', 5, 9), broken('ctx_lo', 5, 3), broken('tree_count', 0, 1),
              broken('token', 3, eng.vocab), broken('seq', 20, 1), broken('seq', 60, 2)):
        assert call(a) == _lib.SP_EINVAL
    assert call(cols(), out=np.array([80], dtype=np.int32)) == _lib.SP_EINVAL
    assert call(cols(), dst=None) == _lib.SP_EINVAL
    assert call(cols(), out=np.arange(65, dtype=np.int32), ids=np.zeros(65, dtype=np.int32)) == _lib.SP_EINVAL
    assert call(np.zeros(2049, dtype=_lib.TOKEN_DTYPE)) == _lib.SP_ECAPACITY
    with pytest.raises(ValueError):
        eng.forward([1] * 201, eng.new_cache(200) if eng._free else c0)


@pytest.mark.parametrize('hidden,heads,kv,n', [(128, 2, 1, 65), (1024, 8, 2, 66), (1152, 9, 3, 67), (2048, 16, 4, 65),
                                               (2176, 17, 17, 66), (4096, 32, 8, 67)])
def test_norm_widths(gpu_device, hidden, heads, kv, n):
    """Hidden sizes at both edges of the wide norm's one, two and four octets per lane, columns that leave its last
    block of four part empty."""
    print(f'hidden={hidden} n={n}', flush=True)
    cfg, w = make_weights(small_cfg(hidden_size=hidden, num_attention_heads=heads, num_key_value_heads=kv), 'q8', seed=7,
                          scale_std=0.0005)
    eng, ref = Qwen2Engine(config=cfg, tensors=w, max_tokens=64), RefQwen2(cfg, w)
    ids = random_prompt(n, cfg['vocab_size'], seed=n)
    want = ref.forward(ids, ref.new_cache(n), all_logits=True)
    rows, _ = eng.forward(ids, eng.new_cache(n), all_logits=True)
    check_rows(rows.cpu(), want, what=f'hidden {hidden}')
