"""Token ids and positions in every form that torch.as_tensor(ids, dtype=torch.long).flatten() takes (the reference's
conversion): plain lists, nested ones, scalar tensors on the CPU and on the GPU, arrays and tensors of any shape."""
import numpy as np
import pytest
import torch

from seedplane_amd.presets import preset
from seedplane_amd.qwen_engine import Qwen2Engine, _id_array
from seedplane_amd.synth import make_weights

FORMS = [[1, 2, 3], [[1, 2], [3, 4]], (5, 6), [], [7.0, 8.0], [True, 2], [np.int32(4), 5], [torch.tensor(3), torch.tensor(4)],
         [torch.tensor([1]), torch.tensor([2])], torch.tensor([[1, 2]]), torch.tensor(9), np.array([[3], [4]], dtype=np.uint8),
         range(4), 6]


@pytest.mark.parametrize('form', range(len(FORMS)))
def test_as_torch_converts_them(form):
    ids = FORMS[form]
    try:
        want = torch.as_tensor(ids, dtype=torch.long).flatten().tolist()
    except (TypeError, ValueError, RuntimeError) as e:
        with pytest.raises(type(e)):
            _id_array(ids)
        return
    got = _id_array(ids)
    assert got.dtype == np.int64 and got.tolist() == want


@pytest.mark.gpu
def test_scalar_tensors_on_the_gpu(gpu_device):
    cfg, w = make_weights(preset('tiny'), 'f32', seed=0)
    eng = Qwen2Engine(config=cfg, tensors=w, max_tokens=16)
    prompt = [1, 2, 3, 4, 5]
    lg, cache = eng.forward(prompt, eng.new_cache(64))
    nxt = lg[0].argmax()
    a, _ = eng.forward([nxt], cache)                       # the id stays a GPU tensor in a list
    cache.length = 5
    b, _ = eng.forward([int(nxt)], cache)
    c, _ = eng.forward([torch.tensor(t, device=eng.device) for t in prompt + [int(nxt)]], eng.new_cache(64),
                       positions=[torch.tensor(p, device=eng.device) for p in range(6)])
    d, _ = eng.forward(prompt + [int(nxt)], eng.new_cache(64))
    assert torch.equal(a, b) and torch.equal(c, d)
