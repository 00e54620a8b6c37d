"""The step's greedy ids from one launch (row words raised by 64 blocks, cleared by the last one): the first index of
the row's largest logit for vocabularies below, at and past the block and load-batch edges, call after call, for one
column and for a batch, in the caller's array and as the fed token.  And persistent steps of two engines on two streams:
each waits for the other's, so both give what they give alone."""
import pytest
import torch

from seedplane_amd import _lib
from seedplane_amd.presets import preset
from seedplane_amd.qwen_engine import Qwen2Engine
from seedplane_amd.synth import make_weights, random_prompt
from tests.conftest import small_cfg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('vocab', [3, 64, 65, 1000, 16385, 140000])
def test_ids_are_the_first_argmax_of_the_logits(gpu_device, vocab):
    print(f'ids of {vocab} logits', flush=True)
    cfg, w = make_weights(preset('tiny', vocab_size=vocab), 'q8', seed=vocab)
    emb = w['model.embed_tokens.qweight']                       # tied head: equal rows give equal logits
    if vocab >= 64:
        emb[vocab // 2:vocab // 2 + 20] = emb[7:27]
        w['model.embed_tokens.scales'][vocab // 2:vocab // 2 + 20] = w['model.embed_tokens.scales'][7:27]
    eng = Qwen2Engine(config=cfg, tensors=w, max_tokens=16)
    eng.reserve(5, 64)
    caches = [eng.new_cache(64) for _ in range(5)]
    rows = torch.empty((5, vocab), device=eng.device)
    toks = random_prompt(5, vocab, seed=1)
    for step in range(4):
        ids = eng.decode(toks, caches, logits_out=rows)
        assert [int(i) for i in ids] == rows.cpu().argmax(dim=1).tolist(), step
        one = eng.decode(toks[:1], caches[:1], logits_out=rows[:1])
        assert int(one[0]) == int(rows[0].cpu().argmax()), step
        toks = [(t * 7 + 3) % vocab for t in toks]
    flat = rows[0].cpu()
    assert int(torch.nonzero(flat == flat.max())[0]) == int(flat.argmax())   # torch takes the first of equal maxima


def test_two_engines_on_two_streams(gpu_device):
    cfg, w = make_weights(small_cfg(), 'q8', seed=4)

    def make(stream):
        with torch.cuda.stream(stream):
            e = Qwen2Engine(config=cfg, tensors=w, max_tokens=16)
            c = e.new_cache(128)
            e.forward([1, 2, 3, 4, 5], c)
        assert e.persistent_status()[0]
        return e, c

    s = [torch.cuda.Stream(), torch.cuda.Stream()]
    pairs = [make(x) for x in s]
    want = pairs[0][0].decode_greedy([9], [pairs[0][1]], 40)[0]
    pairs[0][1].length = 5
    got = [[], []]
    fed = [9, 9]
    for i in range(40):                            # queued without waiting: the launches of both streams interleave
        for k, (e, c) in enumerate(pairs):
            col = e._column(fed[k] if i == 0 else -1, c, c.length, c.length)
            e.run([col], _lib.SP_F_LOGITS | _lib.SP_F_ARGMAX | (_lib.SP_F_FEED if i else 0))
            got[k].append(torch.empty(1, dtype=torch.int32).pin_memory())
            _lib.check(e.lib.sp_engine_copy_ids(e.h, 1, got[k][-1].data_ptr()), e.h)
            c.length += 1
    for k, (e, _) in enumerate(pairs):
        _lib.check(e.lib.sp_engine_sync(e.h), e.h)
        assert [int(t) for t in got[k]] == want


@pytest.mark.parametrize('n', [9, 31, 64])
def test_ids_of_many_long_rows(gpu_device, n):
    """Batches whose rows share the launch's blocks (fewer per row than for one row), step after step."""
    print(f'ids of {n} rows', flush=True)
    vocab = 140000
    cfg, w = make_weights(preset('tiny', vocab_size=vocab), 'q8', seed=n)
    eng = Qwen2Engine(config=cfg, tensors=w, max_tokens=64)
    eng.reserve(n, 32)
    caches = [eng.new_cache(32) for _ in range(n)]
    rows = torch.empty((n, vocab), device=eng.device)
    toks = random_prompt(n, vocab, seed=n)
    for step in range(3):
        ids = eng.decode(toks, caches, logits_out=rows)
        assert [int(i) for i in ids] == rows.cpu().argmax(dim=1).tolist(), step
        toks = [(t * 5 + 1) % vocab for t in toks]
