"""The update of many tensors takes tensors of more than 2^30 parameters, between
others, and more tensors than one launch holds."""

import ctypes

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd import _lib  # noqa: E402
from coffeegpu_amd.surrogate import _TENSOR  # noqa: E402

DEV = "cuda:0"
LR, B1, B2, EPS, T = 1e-2, 0.9, 0.999, 1e-8, 3


def state(n, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    base = torch.randn((4, min(n, 5000)), device=DEV, generator=g)
    base[3] = base[3].abs()
    return [base[q].repeat(-(-n // base.shape[1]))[:n].contiguous() for q in range(4)]


@pytest.mark.parametrize("sizes", [(2000, (1 << 30) + 1000, 300), tuple(range(1000, 1097))])
def test_update_of_many_tensors(sizes):
    if torch.cuda.mem_get_info()[0] < 40 * max(sizes):
        pytest.skip("needs 43 GB of GPU memory")
    tensors = [state(n, k) for k, n in enumerate(sizes)]
    want = []
    for p, gr, m, v in tensors:
        # one call per tensor on its last values
        want.append([q[-200:].clone() for q in (p, gr, m, v)])
    L = _lib.load()
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for w in want:
        _lib.check(L.coffee_unet_adam(*(ctypes.c_void_p(q.data_ptr()) for q in w), 200, LR, B1, B2, EPS, T,
                                      None, None, 0, 0, s))
    packed = b"".join(_TENSOR.pack(*(q.data_ptr() for q in t), 0, 0, t[0].numel(), 0, 0) for t in tensors)
    _lib.check(L.coffee_unet_adam_many(packed, len(tensors), LR, B1, B2, EPS, T, s))
    for t, w in zip(tensors, want):
        for a, b in zip(t, w):
            assert torch.equal(a[-200:], b)
    del tensors
    torch.cuda.empty_cache()
