"""Output gradients at addresses that the fused backward pass has to copy from: any
size after any other, any shape of the array, any stream of the network's."""

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd.surrogate import UNet, pad16  # noqa: E402

DEV = "cuda:0"


def batch(net, n, h, w, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn((n, h, w, pad16(net.cin)), generator=g, device=DEV).to(torch.bfloat16)
    d = 0.01 * torch.randn((n, h, w, pad16(net.cout)), generator=g, device=DEV)
    return x.view(torch.int16).view(-1), d.to(torch.bfloat16)


def off_by_two(d):
    buf = torch.empty(d.numel() + 1, dtype=d.dtype, device=DEV)
    buf[1:] = d.reshape(-1)
    return buf[1:].view(d.shape)


def grads(net, x, d, n, h, w):
    net.forward(x, n, h, w)
    dx = net.backward(d)[: n * h * w * 16].clone()
    return [dx] + [P[k].clone() for P in net.params.values() for k in ("gw", "gb")]


@pytest.mark.parametrize("shaped", [False, True])
def test_misaligned_gradients_of_several_sizes(shaped):
    net = UNet(2, 16, 7, 6, seed=3)
    for n, h, w in ((4, 16, 32), (1, 8, 16), (2, 16, 32), (5, 16, 32)):
        x, d = batch(net, n, h, w, seed=n)
        want = grads(net, x, d.view(torch.int16).view(-1), n, h, w)
        m = off_by_two(d)
        got = grads(net, x, m if shaped else m.view(torch.int16).view(-1), n, h, w)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
