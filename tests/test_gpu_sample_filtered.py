"""GPU filtered sampling (sp_op_sample_filtered: temperature, top-k, top-p, inverse CDF) against the oracle's
sort-based restatement: bit-exact token ids for the same logits and uniforms, at the full Qwen2 vocabulary and with
heavy ties; generate(temperature > 0) draws every token through it.  Both C entries, calls of more draws than one launch
sequence holds, and calls of several threads and streams."""
import threading

import numpy as np
import pytest
import torch

from oracle.sample_ref import sample_filtered
from seedplane_amd import _lib
from seedplane_amd.presets import preset
from seedplane_amd.qwen_engine import Qwen2Engine
from seedplane_amd.speculative import uniforms
from seedplane_amd.synth import make_weights

pytestmark = pytest.mark.gpu

CASES = [(0.7, 0, 1.0), (1.3, 40, 1.0), (0.8, 0, 0.9), (0.8, 50, 0.5), (1.0, 1, 1.0), (0.6, 0, 1e-6),
         (1.1, 1999, 0.95), (0.9, 7, 0.3), (0.8, 151935, 0.99), (2.0, 100000, 1.0)]


@pytest.fixture(scope='module')
def eng(gpu_device):
    cfg, w = make_weights(preset('tiny'), 'f32', seed=0)
    return Qwen2Engine(config=cfg, tensors=w, max_tokens=16)


def _rows(V, seed):
    g = np.random.default_rng(seed)
    rows = (g.standard_normal((6, V)) * 3.0).astype(np.float32)
    rows[4] = np.round(rows[4] * 2) / 2                     # heavy ties
    rows[5] = 0.0
    rows[5, ::7] = 1.0                                      # ties at the maximum
    return rows


@pytest.mark.parametrize('V', [151936, 1000])
@pytest.mark.parametrize('case', range(len(CASES)))
def test_gpu_draws_equal_oracle(eng, V, case):
    T, k, p = CASES[case]
    print(f'sample_filtered V={V} T={T} k={k} p={p}', flush=True)
    rows = _rows(V, seed=case)
    n = rows.shape[0]
    u = uniforms(11, case, 3 * n)
    u[0], u[1] = 0.0, 1.0 - 2.0 ** -53                      # the two ends of the inverse CDF
    lg = torch.from_numpy(rows).cuda()
    got = eng.sample_gpu(lg, [i % n for i in range(3 * n)], u, T, k, p)
    want = [sample_filtered(rows[i % n], T, k, p, u[i]) for i in range(3 * n)]
    assert got == want


def test_gpu_sample_rejects_bad_arguments(eng):
    lg = torch.zeros((2, 100), dtype=torch.float32, device='cuda')
    with pytest.raises(ValueError):
        eng.sample_gpu(lg, [0], [0.5], 0.0)
    with pytest.raises(ValueError):
        eng.sample_gpu(lg, [0], [0.5], 1.0, 0, 0.0)
    # every row index is checked on the host before the launch: nothing out of bounds reaches the kernel
    with pytest.raises(ValueError):
        eng.sample_gpu(lg, [0], [0.5, 0.5], 1.0)                 # fewer rows than draws
    with pytest.raises(ValueError):
        eng.sample_gpu(lg, [2], [0.5], 1.0)                      # row past the end
    with pytest.raises(ValueError):
        eng.sample_gpu(lg, [-1], [0.5], 1.0)
    with pytest.raises(ValueError):
        eng.sample_gpu(torch.zeros((100, 2), device='cuda').t(), [0], [0.5], 1.0)   # strided rows
    with pytest.raises(ValueError):
        eng.sample_gpu(lg, None, [0.5, 0.5], 1.0, rows_dev=torch.zeros(1, dtype=torch.int32, device='cuda'))
    flat = np.zeros(100, dtype=np.float32)
    assert eng.sample_gpu(lg, [1, 0], [0.25, 0.75], 1.0) == [sample_filtered(flat, 1.0, 0, 1.0, u) for u in (0.25, 0.75)]


def test_generate_with_temperature_uses_gpu_draws(eng):
    prompt = [1, 2, 3, 4, 5]
    toks = list(eng.generate(prompt, max_new_tokens=6, temperature=0.8, top_k=20, top_p=0.9, seed=3))
    assert len(toks) == 6
    seq = prompt + toks
    lg, _ = eng.forward(seq[:-1], eng.new_cache(16), all_logits=True)
    rows = lg[len(prompt) - 1:].cpu().numpy()
    for i, t in enumerate(toks):
        assert t == sample_filtered(rows[i], 0.8, 20, 0.9, uniforms(3, i, 1)[0]), i


MIXED = [(0.8, 50, 0.9), (0.8, 0, 0.9), (1.1, 1999, 0.95), (0.7, 0, 1.0), (1.3, 40, 1.0)]


def _device_draws(eng, lg, rows, u, T, k, p):
    """sp_op_sample_filtered on the current stream, not waited for: the ids as a device tensor."""
    r = torch.tensor(rows, dtype=torch.int32, device='cuda')
    ud = torch.tensor(u, dtype=torch.float64, device='cuda')
    out = torch.empty(len(u), dtype=torch.int32, device='cuda')
    _lib.check(eng.lib.sp_op_sample_filtered(lg.data_ptr(), lg.shape[1], lg.stride(0), r.data_ptr(), ud.data_ptr(), len(u), T, k,
                                             p, out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    return out, (r, ud)


@pytest.mark.parametrize('n', [255, 256, 257, 600])
def test_more_draws_than_one_launch_holds(eng, n):
    """Both entries around the 256 draws of one launch sequence, filters changing from call to call."""
    V = 3000
    rows = _rows(V, seed=n)
    lg = torch.from_numpy(rows).cuda()
    at = [i % rows.shape[0] for i in range(n)]
    for j, (T, k, p) in enumerate(MIXED):
        u = uniforms(n, j, n)
        want = [sample_filtered(rows[i], T, k, p, x) for i, x in zip(at, u)]
        assert eng.sample_gpu(lg, at, u, T, k, p) == want, (T, k, p)
        out, _ = _device_draws(eng, lg, at, u, T, k, p)
        assert out.tolist() == want, (T, k, p)


def test_calls_of_threads_and_streams_take_turns(eng):
    """Host calls of two threads on streams of their own, and device calls queued on two streams without a wait between
    them: each gives what it gives alone (the scratch is one per device)."""
    V, n, calls = 40000, 16, 24
    g = torch.Generator(device='cuda').manual_seed(1)
    lg = torch.randn((2, n, V), generator=g, device='cuda') * 3.0
    at = list(range(n))
    args = [MIXED[j % len(MIXED)] for j in range(calls)]
    want = [[eng.sample_gpu(lg[s], at, uniforms(s, j, n), *args[j]) for j in range(calls)] for s in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[None] * calls, [None] * calls]

    def work(s):
        with torch.cuda.stream(streams[s]):
            for j in range(calls):
                got[s][j] = eng.sample_gpu(lg[s], at, uniforms(s, j, n), *args[j])

    threads = [threading.Thread(target=work, args=(s,)) for s in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == want
    queued, held = [[], []], []
    for j in range(calls):
        for s in range(2):
            with torch.cuda.stream(streams[s]):
                out, keep = _device_draws(eng, lg[s], at, uniforms(s, j, n), *args[j])
            queued[s].append(out)
            held.append(keep)
    torch.cuda.synchronize()
    assert [[o.tolist() for o in q] for q in queued] == want


def test_host_entry_refuses_a_capturing_stream(eng):
    lg = torch.randn((2, 500), device='cuda')
    before = eng.sample_gpu(lg, [0, 1], [0.3, 0.6], 1.0, 50, 0.9)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    u, out = np.array([0.3, 0.6]), np.empty(2, dtype=np.int32)
    rows = torch.tensor([0, 1], dtype=torch.int32, device='cuda')
    dst = torch.zeros(4, device='cuda')
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        dst.add_(1.0)
        rc = eng.lib.sp_op_sample_filtered_host(lg.data_ptr(), 500, 500, rows.data_ptr(), None, u.ctypes.data, 2, 1.0, 50, 0.9,
                                                out.ctypes.data, torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.SP_ESTATE
    graph.replay()
    torch.cuda.synchronize()
    assert dst.tolist() == [1.0] * 4 and eng.sample_gpu(lg, [0, 1], [0.3, 0.6], 1.0, 50, 0.9) == before
