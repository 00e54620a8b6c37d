"""The work a user of this package has it do, as cases that can be timed and checked one by one.

A case is one call (or one short sequence of calls) of the public Python API or of the C ABI: decode steps, prefill,
speculative tree verification and its acceptance walk, filtered sampling, and one weight-only product.  Model cases run
the Qwen2-0.5B / 1.5B / 7B shapes of `seedplane_amd.presets` in their usual weight formats.  Two of them run every
layer and the full vocabulary; the others run a few layers over an 8192-entry vocabulary, so that the layers are what
is measured and one layer's rounding does not travel through 28 others.

Weights have the spread of a trained layer (standard deviation 0.02): fp16 normal, or uniform integer codes whose
block scales lie within a factor of three of each other.  Prompts are uniform random ids.  The K/V a step reads come
from a real prefill, except for long batches, which take the engine's own seeded fill as `bench.py` does.
"""
import ctypes
import math

import numpy as np
import torch

from seedplane_amd import _lib
from seedplane_amd.presets import head_dim, preset
from seedplane_amd.qwen_engine import Qwen2Engine
from seedplane_amd.speculative import TreeVerifier, flatten, uniforms
from seedplane_amd.synth import linear_shapes, norm_names

DEV = 'cuda'
GROUP = 32
FORMATS = {'f16': _lib.SP_FMT_F16, 'q8': _lib.SP_FMT_Q8, 'q4': _lib.SP_FMT_Q4}
BYTES_PER_WEIGHT = {'f16': 2.0, 'q8': 1.0 + 2.0 / GROUP, 'q4': 0.5 + 4.0 / GROUP}
SMALL_VOCAB = 8192
MIN_IDS = 8


def listed():
    return [
        # one token of a chat on the 1.5B int8 model, every layer, sliding window full: the interactive case
        _decode('decode_15b_int8_bs1', 'qwen2-1.5b', 'q8', 28, 1, 1500, 1500, 1024, vocab=151936),
        # the smallest whole-model call: a 0.5B fp16 drafter's token a little way into a conversation
        _decode('decode_05b_f16_bs1', 'qwen2-0.5b', 'f16', 24, 1, 61, 61, 0, vocab=151936),
        # a server's batch of 16 long conversations, the window full for all of them
        _decode('decode_15b_int8_bs16', 'qwen2-1.5b', 'q8', 8, 16, 1030, 1300, 1024),
        # a burst of 16 short requests of different lengths on the small model
        _decode('decode_05b_f16_bs16', 'qwen2-0.5b', 'f16', 8, 16, 16, 160, 0),
        # the large batch: 32 requests of 8192 cached tokens each on the 7B int4 model
        _decode('decode_7b_int4_bs32', 'qwen2-7b', 'q4', 2, 32, 8192, 8192, 0, fill=True),
        # a long prompt into a windowed cache (the ring wraps during the prefill)
        _prefill('prefill_15b_int8_2048', 'qwen2-1.5b', 'q8', 4, 2048, 1024),
        # an ordinary prompt, an odd length, full attention, the large model
        _prefill('prefill_7b_int4_777', 'qwen2-7b', 'q4', 2, 777, 0),
        # a burst's prompt phase: 16 ragged prompts in one call, then the first decode step
        {'name': 'prompts_05b_f16_16', 'kind': 'prompts', 'model': 'qwen2-0.5b', 'fmt': 'f16', 'layers': 8,
         'vocab': SMALL_VOCAB, 'batch': 16, 'lo': 16, 'hi': 128},
        # speculative verification: the root and 8 x 4 drafted tokens over 2048 cached positions
        _verify('verify_15b_int8_8x4', 'qwen2-1.5b', 'q8', 8, 8, 4, 2048),
        # the acceptance walk over that tree's logits, full vocabulary
        {'name': 'accept_8x4', 'kind': 'accept', 'vocab': 151936, 'branches': 8, 'depth': 4, 'temperature': 0.8,
         'noise': 0.3},
        # one draw for each of 16 requests with the usual filters
        {'name': 'sample_16_topk50_topp0.9', 'kind': 'sample', 'vocab': 151936, 'rows': 16, 'temperature': 0.8,
         'top_k': 50, 'top_p': 0.9},
        # a weight-only product at the widest matrix: the 1.5B model's LM head over 16 columns
        {'name': 'gemv_head_15b_int8_m16', 'kind': 'gemv', 'fmt': 'q8', 'rows': 151936, 'cols': 1536, 'm': 16},
    ]


def _decode(name, model, fmt, layers, batch, lo, hi, window, vocab=SMALL_VOCAB, fill=False):
    return {'name': name, 'kind': 'decode', 'model': model, 'fmt': fmt, 'layers': layers, 'vocab': vocab,
            'batch': batch, 'lo': lo, 'hi': hi, 'window': window, 'fill': fill}


def _prefill(name, model, fmt, layers, tokens, window, all_logits=False):
    return {'name': name, 'kind': 'prefill', 'model': model, 'fmt': fmt, 'layers': layers, 'vocab': SMALL_VOCAB,
            'tokens': tokens, 'window': window, 'all_logits': all_logits}


def _verify(name, model, fmt, layers, branches, depth, prefix):
    return {'name': name, 'kind': 'verify', 'model': model, 'fmt': fmt, 'layers': layers, 'vocab': SMALL_VOCAB,
            'branches': branches, 'depth': depth, 'prefix': prefix}


def draw(rng):
    """One more case of the same ranges."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(['decode', 'decode', 'decode', 'prefill', 'prefill', 'prompts', 'verify', 'accept', 'sample',
                       'gemv'])
    model, fmt, layers = rng.choice([('qwen2-0.5b', 'f16', 8), ('qwen2-0.5b', 'q8', 8), ('qwen2-1.5b', 'q8', 4),
                                     ('qwen2-1.5b', 'q4', 4), ('qwen2-7b', 'q4', 2)])
    window = rng.choice([0, 0, 256, 1024])
    if kind == 'decode':
        batch, hi = log(1, 33), log(16, 2048)
        c = _decode(None, model, fmt, layers, batch, max(1, int(hi * rng.uniform(0.3, 1.0))), hi, window,
                    fill=batch * hi > 20000)
        if c['fill']:
            c['window'] = 0
    elif kind == 'prefill':
        c = _prefill(None, model, fmt, 2 if model == 'qwen2-7b' else 4, log(17, 777 if model == 'qwen2-7b' else 1900),
                     window, all_logits=rng.random() < 0.25)
    elif kind == 'prompts':
        batch = log(2, 32)
        hi = log(16, min(300, (700 if model == 'qwen2-7b' else 2000) // batch))
        c = {'kind': 'prompts', 'model': model, 'fmt': fmt, 'layers': 2 if model == 'qwen2-7b' else 4,
             'vocab': SMALL_VOCAB, 'batch': batch, 'lo': max(1, hi // 8), 'hi': hi}
    elif kind == 'verify':
        depth = rng.randint(1, 5)
        c = _verify(None, model, fmt, layers, rng.randint(1, min(12, 63 // depth)), depth, log(64, 2048))
    elif kind == 'accept':
        depth = rng.randint(1, 5)
        c = {'kind': 'accept', 'vocab': rng.choice([151936, 152064, log(1000, 100000)]), 'branches': rng.randint(1, 12),
             'depth': depth, 'temperature': rng.choice([0.6, 0.8, 1.0]), 'noise': rng.choice([0.1, 0.3, 1.0])}
    elif kind == 'sample':
        c = {'kind': 'sample', 'vocab': rng.choice([151936, 152064, log(1000, 100000)]), 'rows': log(1, 32),
             'temperature': rng.choice([0.6, 0.8, 1.0]), 'top_k': rng.choice([0, 20, 50]),
             'top_p': rng.choice([1.0, 0.8, 0.9, 0.95])}
    else:
        fmt, rows, cols = rng.choice([('q8', 2048, 1536), ('q8', 1536, 8960), ('q8', 151936, 1536), ('f16', 1152, 896),
                                      ('f16', 9728, 896), ('f16', 896, 4864), ('q4', 4608, 3584), ('q4', 37888, 3584),
                                      ('q4', 3584, 18944), ('q8', 8961, 1536)])
        c = {'kind': 'gemv', 'fmt': fmt, 'rows': rows, 'cols': cols, 'm': log(1, 64)}
    c.pop('name', None)
    return c


# ------------------------------------------------------------------------------------------------ inputs from a seed
def _cfg(case):
    cfg = preset(case['model'], num_hidden_layers=case['layers'], vocab_size=case['vocab'])
    if case['fmt'] != 'f16':
        cfg['quantization_config'] = {'quant_method': 'seedplane', 'bits': 8 if case['fmt'] == 'q8' else 4,
                                      'group_size': GROUP}
    return cfg


def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + stream) % (2 ** 63))


def _quant(g, fmt, n, k):
    """Codes, scales and zeros of an n x k matrix whose values have standard deviation 0.02."""
    rnd = lambda: torch.rand((n, k // GROUP), generator=g, device=DEV)
    if fmt == 'q8':
        return (torch.randint(-127, 128, (n, k), dtype=torch.int8, generator=g, device=DEV),
                ((rnd() + 0.5) * (0.02 / 76)).half(), None)
    return (torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, generator=g, device=DEV),
            ((rnd() + 0.5) * (0.02 / 4.8)).half(), (rnd() + 7.0).half())


def _weights(case, seed):
    """Named tensors of the case's model, on the GPU."""
    cfg = _cfg(case)
    g = _gen(seed, 1)
    w = {}
    for name, n, k, has_bias in linear_shapes(cfg):
        if case['fmt'] == 'f16':
            w[name + '.weight'] = (torch.randn((n, k), generator=g, device=DEV) * 0.02).half()
        else:
            codes, scales, zeros = _quant(g, case['fmt'], n, k)
            w[name + '.qweight'], w[name + '.scales'] = codes, scales
            if zeros is not None:
                w[name + '.qzeros'] = zeros
        if has_bias:
            w[name + '.bias'] = (torch.randn(n, generator=g, device=DEV) * 0.02).half()
    for name in norm_names(cfg):
        w[name] = (1.0 + 0.1 * torch.randn(cfg['hidden_size'], generator=g, device=DEV)).half()
    return cfg, w


def _ids(rng, n, vocab):
    return rng.integers(0, vocab, n).tolist()


def _lengths(case, rng):
    return [int(x) for x in rng.integers(case['lo'], case['hi'] + 1, case['batch'])]


def _texts(case, seed):
    """The token lists of a case: prompts (or cached lengths), and the tokens fed after them."""
    rng = np.random.default_rng([seed, 2])
    if case['kind'] in ('decode', 'prompts'):
        lens = _lengths(case, rng)
        prompts = [None if case.get('fill') else _ids(rng, n, case['vocab']) for n in lens]
        return lens, prompts, _ids(rng, case['batch'], case['vocab'])
    if case['kind'] == 'prefill':
        return _ids(rng, case['tokens'], case['vocab'])
    prompt = _ids(rng, case['prefix'], case['vocab'])
    return prompt, _tree(case, rng)


def _tree(case, rng):
    """A draft tree whose branches share some first tokens, as a drafter's do."""
    firsts = _ids(rng, max(1, (case['branches'] + 1) // 2), case['vocab'])
    branches = [[firsts[int(rng.integers(len(firsts)))]] + _ids(rng, case['depth'] - 1, case['vocab'])
                if rng.random() < 0.4 else _ids(rng, case['depth'], case['vocab']) for _ in range(case['branches'])]
    return flatten(int(rng.integers(case['vocab'])), branches)


def _walk_inputs(case, seed):
    rng = np.random.default_rng([seed, 3])
    g = _gen(seed, 4)
    V = case['vocab']
    # the drafter's tokens are draws from its own distribution: give the drafted tokens of every node high logits
    tree = _tree(case, rng)
    p = torch.randn((tree.size, V), generator=g, device=DEV) * 2.0
    for i in range(tree.size):
        for c in range(tree.n_children[i]):
            p[i, tree.token[tree.first_child[i] + c]] += 12.0
    q = p + case['noise'] * torch.randn((tree.size, V), generator=g, device=DEV)
    return tree, p, q, uniforms(seed, 0, 64)


def _sample_inputs(case, seed):
    lg = torch.randn((case['rows'], case['vocab']), generator=_gen(seed, 5), device=DEV) * 3.0
    return lg, uniforms(seed, 1, case['rows'])


def _gemv_inputs(case, seed):
    g = _gen(seed, 6)
    n, k = case['rows'], case['cols']
    if case['fmt'] == 'f16':
        w = ((torch.randn((n, k), generator=g, device=DEV) * 0.02).half(), None, None)
    else:
        w = _quant(g, case['fmt'], n, k)
    return w, torch.randn((case['m'], k), generator=g, device=DEV).half()


# ------------------------------------------------------------------------------------------------ prepare / run
class _Weight:
    """A packed matrix handle of the C ABI, released with the object."""

    def __init__(self, fmt, rows, cols, arrays):
        self.lib = _lib.load()
        host = [None if a is None else a.cpu().contiguous() for a in arrays]
        ptrs = [None if a is None else ctypes.c_void_p(a.data_ptr()) for a in host]
        self.h = ctypes.c_void_p()
        _lib.check(self.lib.sp_weight_create(FORMATS[fmt], rows, cols, *ptrs, ctypes.byref(self.h)))

    def __del__(self):
        self.lib.sp_weight_destroy(self.h)


def prepare(case, seed):
    kind = case['kind']
    st = {'kind': kind, 'case': case}
    if kind == 'gemv':
        w, x = _gemv_inputs(case, seed)
        st['w'] = _Weight(case['fmt'], case['rows'], case['cols'], w)
        st['x'] = x
        st['y'] = torch.empty((case['m'], case['rows']), dtype=torch.float32, device=DEV)
        return st
    if kind == 'accept':
        tree, p, q, u = _walk_inputs(case, seed)
        st.update(tree=tree, p=p, q=q, u=u, verifier=TreeVerifier(_small_engine()))
        return st
    if kind == 'sample':
        lg, u = _sample_inputs(case, seed)
        st.update(logits=lg, u=u, eng=_small_engine(), rows=torch.arange(case['rows'], dtype=torch.int32, device=DEV))
        return st
    cfg, w = _weights(case, seed)
    eng = st['eng'] = Qwen2Engine(config=cfg, tensors=w, device=DEV, max_tokens=64)
    del w
    window = case.get('window') or None
    texts = _texts(case, seed)
    if kind == 'prefill':
        st['ids'] = texts
        st['cache'] = eng.new_cache(len(texts) + 64, window=window)
    elif kind == 'verify':
        prompt, st['tree'] = texts
        st['cache'] = eng.new_cache(len(prompt) + 128)
        eng.forward(prompt, st['cache'])
        st['verifier'] = TreeVerifier(eng)
        st['logits'] = torch.empty((st['tree'].size, case['vocab']), dtype=torch.float32, device=DEV)
    else:
        st['lens'], st['prompts'], st['tokens'] = texts
        # the caller's own logits rows (the engine's buffer goes with the engine)
        st['logits'] = torch.empty((case['batch'], case['vocab']), dtype=torch.float32, device=DEV)
        cap = max(st['lens']) + 64
        eng.reserve(case['batch'], eng.slots_for(cap, window))
        st['caches'] = [eng.new_cache(cap, window=window) for _ in st['lens']]
        if kind == 'decode':
            for b, cache in enumerate(st['caches']):
                if case['fill']:
                    eng.fill_cache(cache, st['lens'][b], seed=seed + 16 * b)
            if not case['fill']:
                eng.prefill(st['prompts'], st['caches'])
    return st


def _small_engine():
    """An engine whose model does not matter: the sampling calls take logits from anywhere."""
    case = {'model': 'tiny', 'layers': 1, 'vocab': 64, 'fmt': 'f16'}
    cfg, w = _weights(case, 0)
    return Qwen2Engine(config=cfg, tensors=w, device=DEV, max_tokens=1)


def _with_ids(st, ids, first=None):
    """Logits, and the greedy ids of batches (of a few rows, one near-tie would be a large share of the ids)."""
    out = {'logits': st['logits']}
    if len(ids) >= MIN_IDS:
        out['ids'] = ids
        if first is not None:
            out['first'] = np.asarray(first, dtype=np.int64)
    return out


def run(st):
    kind = st['kind']
    if kind == 'decode':
        for c, n in zip(st['caches'], st['lens']):
            c.length = n                                    # roll back to the same position on every pass
        ids = st['eng'].decode(st['tokens'], st['caches'], logits_out=st['logits'])
        return _with_ids(st, ids)
    if kind == 'prefill':
        cache = st['cache']
        cache.length = 0
        logits, _ = st['eng'].forward(st['ids'], cache, all_logits=st['case']['all_logits'])
        return {'logits': logits, 'k': cache.keys[-1], 'v': cache.values[-1]}
    if kind == 'prompts':
        for c in st['caches']:
            c.length = 0
        first = st['eng'].prefill(st['prompts'], st['caches'])
        ids = st['eng'].decode(st['tokens'], st['caches'], logits_out=st['logits'])
        return _with_ids(st, ids, first)
    if kind == 'verify':
        return {'logits': st['verifier'].forward(st['cache'], st['tree'], logits_out=st['logits'], ids=False)}
    if kind == 'accept':
        path, final, used, bonus = st['verifier'].accept(st['p'], st['q'], st['tree'], st['u'],
                                                         st['case']['temperature'])
        return np.asarray([len(path), *path, final, used, int(bonus)], dtype=np.int64)
    if kind == 'sample':
        c = st['case']
        ids = st['eng'].sample_gpu(st['logits'], None, st['u'], c['temperature'], c['top_k'], c['top_p'],
                                   rows_dev=st['rows'])
        return np.asarray(ids, dtype=np.int64)
    lib, c = st['w'].lib, st['case']
    _lib.check(lib.sp_op_gemv(st['w'].h, ctypes.c_void_p(st['x'].data_ptr()), c['m'],
                              ctypes.c_void_p(st['y'].data_ptr()), None,
                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return st['y']


# ------------------------------------------------------------------------------------------------ what a pass needs
def _matrix_weights(case):
    """(weights of one layer's matrices, of the head) in elements."""
    cfg = _cfg(case)
    H, I, NH, NKV, HD = (cfg['hidden_size'], cfg['intermediate_size'], cfg['num_attention_heads'],
                         cfg['num_key_value_heads'], head_dim(cfg))
    return (NH + 2 * NKV) * HD * H + H * NH * HD + 3 * H * I, case['vocab'] * H, NH * HD, NKV * HD


def work(case):
    kind = case['kind']
    if kind == 'gemv':
        n, k, m = case['rows'], case['cols'], case['m']
        return {'bytes': n * k * BYTES_PER_WEIGHT[case['fmt']] + 2 * m * k + 4 * m * n, 'flops': 2 * m * n * k}
    if kind == 'accept':
        # the rows on the accepted path: at least the root's target and drafter rows
        return {'bytes': 2 * 4 * case['vocab'], 'flops': 8 * case['vocab']}
    if kind == 'sample':
        return {'bytes': 4 * case['rows'] * case['vocab'], 'flops': 4 * case['rows'] * case['vocab']}
    layer, head, q, kv = _matrix_weights(case)
    L, W = case['layers'], case.get('window') or 0
    if kind == 'prefill':
        groups = [(case['tokens'], 0)]
        heads = case['tokens'] if case['all_logits'] else 1
    elif kind == 'verify':
        groups = [(1 + case['branches'] * case['depth'], case['prefix'])]
        heads = 1 + case['branches'] * case['depth']
    else:
        mid = (case['lo'] + case['hi']) // 2
        groups = [(1, mid) if kind == 'decode' else (mid + 1, 0)] * case['batch']
        heads = case['batch'] * (1 if kind == 'decode' else 2)
    cols = sum(n for n, _ in groups)
    read = pairs = 0
    for n, past in groups:
        read += min(past, W) if W else past
        full = n * past + n * (n + 1) // 2
        pairs += min(full, n * W) if W else full
    b = BYTES_PER_WEIGHT[case['fmt']]
    return {'bytes': (L * layer + head) * b + L * kv * 4 * (read + cols) + 4 * heads * case['vocab'],
            'flops': 2 * (L * layer * cols + head * heads) + 4 * L * q * pairs}


def tolerance(case):
    kind = case['kind']
    if kind in ('accept', 'sample'):
        return 'exact'
    if kind == 'gemv':
        return {'rel': 4e-6}          # 32-bit sums over K: about 7e-7 from the 64-bit product
    # fp16 activations and K/V between the layers: 0.6e-3 to 1.2e-3 from the 64-bit model
    return {'rel': 4e-3, 'differ': 0.15} if case.get('batch', 1) >= MIN_IDS else {'rel': 4e-3}


# ------------------------------------------------------------------------------------------------ 64-bit results
def _dense(w, name, fmt):
    """A named matrix in 64 bits."""
    if fmt == 'f16':
        return w[name + '.weight'].double()
    return _dequant(fmt, w[name + '.qweight'], w[name + '.scales'], w.get(name + '.qzeros'))


def _dequant(fmt, codes, scales, zeros):
    n = codes.shape[0]
    if fmt == 'q8':
        v = codes.double().view(n, -1, GROUP)
    else:
        v = torch.stack([codes & 15, codes >> 4], dim=-1).view(n, -1, GROUP).double() - zeros.double()[:, :, None]
    return (v * scales.double()[:, :, None]).view(n, -1)


def _norm(x, weight, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * weight.double()


def _rope(x, pos, cfg):
    """x [tokens, heads, head_dim] rotated at positions pos, half by half."""
    hd = x.shape[-1]
    inv = 1.0 / (cfg['rope_theta'] ** (torch.arange(0, hd, 2).float() / hd))
    ph = pos.double()[:, None] * inv.double().to(x.device)[None]
    c, s = ph.cos()[:, None], ph.sin()[:, None]
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


class _Sequence:
    """Tokens to run, their positions, which of them see which (a boolean [tokens, past + tokens] mask) and the K/V
    of earlier positions per layer (None without any)."""

    def __init__(self, tokens, pos=None, mask=None, window=None, past=None, n_past=0):
        n = len(tokens)
        self.tokens = torch.tensor(tokens, device=DEV)
        self.pos = torch.arange(n_past, n_past + n, device=DEV) if pos is None else torch.tensor(pos, device=DEV)
        if mask is None:
            i, j = self.pos[:, None], torch.arange(n_past + n, device=DEV)[None]
            mask = (j <= i) & (j > i - window) if window else j <= i
        self.mask, self.past, self.k, self.v = mask, past, None, None


def _model64(cfg, w, fmt, seqs):
    """Final hidden states (normalised) of every sequence; the last layer's keys and values stay in the sequences."""
    NH, NKV, HD, H = cfg['num_attention_heads'], cfg['num_key_value_heads'], head_dim(cfg), cfg['hidden_size']
    eps, G = cfg['rms_norm_eps'], NH // NKV
    emb = 'model.embed_tokens'
    rows = lambda t, i: None if t is None else t[i]
    for s in seqs:
        if fmt == 'f16':
            s.x = w[emb + '.weight'][s.tokens].double()
        else:
            s.x = _dequant(fmt, w[emb + '.qweight'][s.tokens], w[emb + '.scales'][s.tokens],
                           rows(w.get(emb + '.qzeros'), s.tokens))
    for l in range(cfg['num_hidden_layers']):
        p = f'model.layers.{l}.'
        att = [p + 'self_attn.' + n for n in ('q_proj', 'k_proj', 'v_proj')]
        wq, wk, wv = (_dense(w, n, fmt) for n in att)
        bq, bk, bv = (w[n + '.bias'].double() for n in att)
        wo = _dense(w, p + 'self_attn.o_proj', fmt)
        for s in seqs:
            n = len(s.tokens)
            h = _norm(s.x, w[p + 'input_layernorm.weight'], eps)
            q = _rope((h @ wq.T + bq).view(n, NH, HD), s.pos, cfg)
            k = _rope((h @ wk.T + bk).view(n, NKV, HD), s.pos, cfg)
            v = (h @ wv.T + bv).view(n, NKV, HD)
            s.k, s.v = k, v
            if s.past is not None:
                pk, pv = s.past(l)
                k, v = torch.cat([pk, k]), torch.cat([pv, v])
            out = torch.empty((n, NH, HD), dtype=torch.float64, device=DEV)
            for kh in range(NKV):
                qs = q[:, kh * G:(kh + 1) * G].permute(1, 0, 2).reshape(G * n, HD)
                sc = (qs @ k[:, kh].T / math.sqrt(HD)).view(G, n, -1).masked_fill(~s.mask[None], -math.inf)
                pr = sc.softmax(-1).view(G * n, -1)
                out[:, kh * G:(kh + 1) * G] = (pr @ v[:, kh]).view(G, n, HD).permute(1, 0, 2)
            s.x = s.x + out.view(n, NH * HD) @ wo.T
        wg, wu, wd = (_dense(w, p + 'mlp.' + n, fmt) for n in ('gate_proj', 'up_proj', 'down_proj'))
        for s in seqs:
            h = _norm(s.x, w[p + 'post_attention_layernorm.weight'], eps)
            s.x = s.x + (torch.nn.functional.silu(h @ wg.T) * (h @ wu.T)) @ wd.T
        del wq, wk, wv, wo, wg, wu, wd
    return [_norm(s.x, w['model.norm.weight'], eps) for s in seqs]


def _filled(case, cfg, b, n, n_slots, seed):
    """Layer l's K and V of positions [0, n) that `fill_cache(cache, n, seed)` gives sequence b of a pool of n_slots
    slots: hashed 24-bit uniforms in [-1, 1], rounded to fp16."""
    NKV, HD = cfg['num_key_value_heads'], head_dim(cfg)
    def srl(x, k):
        return (x >> k) & ((1 << (64 - k)) - 1)

    def signed(c):
        return c - (1 << 64) if c >= 1 << 63 else c

    def layer(l):
        kvh = torch.arange(NKV, device=DEV)[None, :, None]
        slot = torch.arange(n, device=DEV)[:, None, None]
        d = torch.arange(HD, device=DEV)[None, None, :]
        x = (((b * NKV + kvh) * n_slots + slot) * HD + d + (l << 40)) ^ seed
        x = x + signed(0x9E3779B97F4A7C15)
        x = (x ^ srl(x, 30)) * signed(0xBF58476D1CE4E5B9)
        x = (x ^ srl(x, 27)) * signed(0x94D049BB133111EB)
        x = x ^ srl(x, 31)
        u = [(y & 0xFFFFFF).float() * (1.0 / 16777216.0) for y in (x, srl(x, 24))]
        return tuple((2.0 * t - 1.0).half().double() for t in u)
    return layer


def _accept64(tree, p, q, u, T):
    """The acceptance walk on float64 distributions: trials in draft order, the residual after each rejection."""
    soft = lambda row: torch.softmax(row.double() / T, -1).cpu().numpy()
    cur, used, path = 0, 0, []
    pick = lambda d, t: int(np.searchsorted(np.cumsum(d), t * d.sum(), side='right'))
    while tree.n_trials[cur]:
        r, qq, nxt = soft(p[cur]), soft(q[cur]), -1
        t0 = tree.trial_start[cur]
        for child in tree.trials[t0:t0 + tree.n_trials[cur]]:
            x = tree.token[child]
            used += 1
            if u[used - 1] < r[x] / qq[x]:
                nxt = child
                break
            r = np.maximum(r - qq, 0.0)
            r = r / r.sum()
        if nxt < 0:
            return [len(path), *path, pick(r, u[used]), used + 1, 0]
        path.append(nxt)
        cur = nxt
    return [len(path), *path, pick(soft(p[cur]), u[used]), used + 1, 1]


def _sample64(row, T, top_k, top_p, u):
    """One filtered draw: z = l / T in fp32, ties of the k-th largest kept, the shortest prefix of the sorted order
    whose mass before each entry is at most top_p of the kept mass, then the inverse CDF in that order."""
    z = (row / np.float32(T)).astype(np.float32)
    order = np.argsort(-z, kind='stable')
    if 0 < top_k < z.size:
        order = order[z[order] >= z[order[top_k - 1]]]
    m = np.exp(z[order].astype(np.float64) - np.float64(z[order[0]]))
    c = np.cumsum(m)
    if top_p < 1.0:
        keep = c - m <= top_p * c[-1]
        order, c = order[keep], c[keep]
    return int(order[min(np.searchsorted(c, u * c[-1], side='right'), order.size - 1)])


def exact(case, seed):
    kind = case['kind']
    if kind == 'gemv':
        w, x = _gemv_inputs(case, seed)
        W = w[0].double() if case['fmt'] == 'f16' else _dequant(case['fmt'], *w)
        return x.double() @ W.T
    if kind == 'accept':
        tree, p, q, u = _walk_inputs(case, seed)
        return np.asarray(_accept64(tree, p, q, u, case['temperature']), dtype=np.int64)
    if kind == 'sample':
        lg, u = _sample_inputs(case, seed)
        lg = lg.cpu().numpy()
        return np.asarray([_sample64(lg[i], case['temperature'], case['top_k'], case['top_p'], u[i])
                           for i in range(case['rows'])], dtype=np.int64)
    cfg, w = _weights(case, seed)
    fmt, window = case['fmt'], case.get('window') or None
    texts = _texts(case, seed)
    if kind == 'prefill':
        seqs = [_Sequence(texts, window=window)]
    elif kind == 'verify':
        prompt, tree = texts
        P, n = len(prompt), tree.size
        mask = torch.zeros((P + n, P + n), dtype=torch.bool, device=DEV)
        mask[:P, :P] = torch.ones((P, P), dtype=torch.bool, device=DEV).tril()
        mask[P:, :P] = True
        for i in range(n):
            j = i
            while j >= 0:
                mask[P + i, P + j] = True
                j = tree.parent[j]
        seqs = [_Sequence(prompt + tree.token, list(range(P)) + [P + d for d in tree.depth], mask)]
    else:
        lens, prompts, toks = texts
        if case.get('fill'):
            slots = max(lens) + 64
            seqs = [_Sequence([t], past=_filled(case, cfg, b, n, slots, seed + 16 * b), n_past=n)
                    for b, (n, t) in enumerate(zip(lens, toks))]
        else:
            seqs = [_Sequence(p + [t], window=window) for p, t in zip(prompts, toks)]
    hid = _model64(cfg, w, fmt, seqs)
    head = _dense(w, 'model.embed_tokens' if cfg['tie_word_embeddings'] else 'lm_head', fmt)
    if kind == 'prefill':
        s = seqs[0]
        n = len(texts)
        first = max(0, n - (window + 64)) if window else 0        # the ring keeps window + 64 positions
        kv = []
        for t in (s.k, s.v):
            full = torch.zeros((1, n + 64, *t.shape[1:]), dtype=torch.float64, device=DEV)
            full[0, first:n] = t[first:]
            kv.append(full)
        return {'logits': (hid[0] if case['all_logits'] else hid[0][-1:]) @ head.T, 'k': kv[0], 'v': kv[1]}
    if kind == 'verify':
        return {'logits': hid[0][len(texts[0]):] @ head.T}
    logits = torch.stack([h[-1] for h in hid]) @ head.T
    out = {'logits': logits}
    if len(hid) >= MIN_IDS:
        out['ids'] = logits.argmax(-1).cpu().numpy().astype(np.int32)
        if kind == 'prompts':
            before = torch.stack([h[-2] for h in hid]) @ head.T
            out['first'] = before.argmax(-1).cpu().numpy().astype(np.int64)
    return out
