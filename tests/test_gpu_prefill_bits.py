"""Prompts longer than max_tokens go through sp_engine_prefill in wide passes.  Their logits, greedy ids and cached K/V are
bit for bit those of the same columns run as steps of max_tokens columns (run(), the path of tree passes and batches):
no tolerance.  The column counts reach the wide products' tiles and both ways of forming k-slices for every format and
epilogue; head groups of 1 to 8 query heads; windowed rings that wrap inside a call; last chunks of 1, up to 16 and more
columns."""
import numpy as np
import pytest
import torch

from seedplane_amd import _lib
from seedplane_amd.presets import preset
from seedplane_amd.qwen_engine import Qwen2Engine
from seedplane_amd.synth import make_weights, random_prompt
from tests.conftest import small_cfg
from tests.parity import check_rows

pytestmark = pytest.mark.gpu


def _engine(shape, fmt, max_tokens=64, **kw):
    cfg = (small_cfg(max_position_embeddings=8192, **kw) if shape == 'small' else
           preset(shape, num_hidden_layers=2, vocab_size=1000))
    cfg, w = make_weights(cfg, fmt, seed=5, scale_std=0.0005)
    return cfg, Qwen2Engine(config=cfg, tensors=w, max_tokens=max_tokens)


def _steps(eng, queue):
    """(cache, token) columns in steps of max_tokens columns; every column's logits and greedy id.  `queue` holds each
    cache's tokens in order."""
    T, at = eng.max_tokens, {}
    rows = torch.empty((len(queue), eng.vocab), device=eng.device)
    ids = []
    for c0 in range(0, len(queue), T):
        cols = []
        for cache, t in queue[c0:c0 + T]:
            p = at.setdefault(cache.seq, cache.length)
            cols.append(eng._column(t, cache, p, p))
            at[cache.seq] = p + 1
        ids += eng.run(cols, _lib.SP_F_LOGITS, logits_out=rows[c0:c0 + T], want_ids=True).tolist()
    for cache, _ in queue:
        cache.length = at[cache.seq]
    return rows, ids


def _kv(cache, layers):
    return [t[l].clone() for l in range(layers) for t in (cache.keys, cache.values)]


def _same_kv(a, b, what):
    for x, y in zip(a, b):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16)), what


SWEEP = [
    ('small', 'f16', [65, 81, 129, 640], None), ('small', 'q8', [80, 145, 700, 2049], 100), ('small', 'q4', [96, 130, 2112], 64),
    ('qwen2-0.5b', 'f16', [193, 576, 1152, 2048], None), ('qwen2-0.5b', 'q8', [130, 705, 1500], 256),
    ('qwen2-1.5b', 'q8', [257, 700, 1100, 2048], 1024), ('qwen2-1.5b', 'q4', [128, 513, 1300], None),
    ('qwen2-7b', 'q4', [100, 360, 500, 737, 777, 1760], None), ('qwen2-7b', 'q8', [500, 1400, 1800], None),
    ('qwen2-7b', 'f16', [497, 600, 1500], None)]


@pytest.mark.parametrize('shape,fmt,counts,window', SWEEP)
def test_prompt_gives_the_bits_of_its_steps(gpu_device, shape, fmt, counts, window):
    cfg, eng = _engine(shape, fmt)
    L = cfg['num_hidden_layers']
    for n in counts:
        print(f'prefill bits {shape} {fmt} n={n} window={window}', flush=True)
        ids = random_prompt(n, cfg['vocab_size'], seed=n)
        cap = max(counts) + 160
        ref = eng.new_cache(cap, window=window)
        want, greedy = _steps(eng, [(ref, t) for t in ids])
        cache = eng.new_cache(cap, window=window)
        rows, _ = eng.forward(ids, cache, all_logits=True)
        assert torch.equal(rows, want), f'{n}: all logits'
        kv = _kv(ref, L)
        _same_kv(_kv(cache, L), kv, f'{n}: K/V')
        cache.length = 0
        last, _ = eng.forward(ids, cache)
        assert torch.equal(last, want[-1:]), f'{n}: last logits'
        _same_kv(_kv(cache, L), kv, f'{n}: K/V, last logits only')
        # a second prompt on top of the first (keys from the ring and from the call), as one call and as steps
        more = random_prompt(150, cfg['vocab_size'], seed=1)
        want2, g2 = _steps(eng, [(ref, t) for t in more])
        assert eng._prefill_greedy(more, cache) == g2[-1], f'{n}: second prompt'
        _same_kv(_kv(cache, L), _kv(ref, L), f'{n}: K/V of the second prompt')
        assert eng.decode([3], [cache]).tolist() == eng.decode([3], [ref]).tolist()
        del ref, cache


@pytest.mark.parametrize('fmt', ['f16', 'q8', 'q4'])
@pytest.mark.parametrize('max_tokens', [64, 48, 20, 17, 16, 4])
def test_prompts_of_several_sequences(gpu_device, fmt, max_tokens):
    """Ragged prompts back to back, chunks of any size, more prompts than one call can end; the decode step after them."""
    print(f'prompts bits {fmt} max_tokens={max_tokens}', flush=True)
    cfg, eng = _engine('small', fmt, max_tokens)
    lens = [3, 300, 1, 0, 64, 1, 1, 5, 400, 2, 33, 17, 130] + [1] * 70 + [90]
    prompts = [random_prompt(k, cfg['vocab_size'], seed=i) for i, k in enumerate(lens)]
    eng.reserve(2 * len(lens), 480)
    a, b = ([eng.new_cache(470) for _ in lens] for _ in range(2))
    got = eng.prefill(prompts, a)
    queue = [(b[s], t) for s, p in enumerate(prompts) for t in p]
    _, greedy = _steps(eng, queue)
    ends = np.cumsum(lens) - 1
    assert got == [greedy[e] if n else None for e, n in zip(ends, lens)]
    for x, y, n in zip(a, b, lens):
        assert x.length == y.length == n
        _same_kv(_kv(x, 2), _kv(y, 2), f'{n} tokens')
    k = min(max_tokens, 16)
    rows = [torch.empty((k, eng.vocab), device=eng.device) for _ in range(2)]
    toks = random_prompt(k, cfg['vocab_size'], seed=2)
    live = [i for i, n in enumerate(lens) if n][:k]
    i0 = eng.decode(toks, [a[i] for i in live], logits_out=rows[0])
    i1 = eng.decode(toks, [b[i] for i in live], logits_out=rows[1])
    assert i0.tolist() == i1.tolist() and torch.equal(rows[0], rows[1])


@pytest.mark.parametrize('heads,kv,hd', [(4, 4, 64), (6, 2, 64), (10, 2, 64), (6, 1, 128), (8, 1, 64), (14, 2, 128)])
def test_head_groups(gpu_device, heads, kv, hd):
    print(f'group bits heads={heads} kv={kv} hd={hd}', flush=True)
    cfg, eng = _engine('small', 'q8', hidden_size=heads * hd, num_attention_heads=heads, num_key_value_heads=kv)
    ids = random_prompt(333, cfg['vocab_size'], seed=heads)
    ref, cache = eng.new_cache(400), eng.new_cache(400)
    want, _ = _steps(eng, [(ref, t) for t in ids])
    rows, _ = eng.forward(ids, cache, all_logits=True)
    assert torch.equal(rows, want)
    _same_kv(_kv(cache, 2), _kv(ref, 2), 'K/V')


@pytest.mark.parametrize('max_tokens,n', [(64, 200), (64, 40), (8, 40)])
def test_ring_of_exactly_the_window(gpu_device, max_tokens, n):
    """A ring without the slack of a chunk (callers of the C entry): a step of several columns would overwrite keys that
    its first columns still see, a prefill call does not.  Against the ring with slack (fp16-class bar: the keys are cut
    into other blocks); the ring's content in the first layer, whose fp32 sums may be taken in another order: one fp16
    step."""
    print(f'tight ring bits max_tokens={max_tokens} n={n}', flush=True)
    W, rows, kv = 24, [], []
    ids = random_prompt(n, 1000, seed=n)
    for slots in (W, W + 64):
        cfg, eng = _engine('small', 'q8', max_tokens)
        eng.reserve(1, slots)
        cols = np.zeros(n, dtype=_lib.TOKEN_DTYPE)
        cols['token'], cols['pos'] = ids, np.arange(n)
        cols['ctx_hi'], cols['slot'] = np.arange(n), np.arange(n) % slots
        cols['ctx_lo'] = np.maximum(0, np.arange(n) - W + 1)
        rows.append(torch.empty((n, eng.vocab), device=eng.device))
        eng._wide(cols, np.arange(n), logits_out=rows[-1])
        k, v = eng._kv_pool(0)
        last = torch.arange(n - W, n, device=eng.device) % slots
        kv.append([t[0][:, last].clone() for t in (k, v)])
        del k, v
    check_rows(rows[0].cpu(), rows[1].cpu(), what='logits')
    for a, b in zip(*kv):
        a, b = a.float(), b.float()
        bound = 2.0 ** -10 * torch.maximum(a.abs(), b.abs()) + 1e-5 * float(b.abs().max())
        assert bool(((a - b).abs() <= bound).all())
