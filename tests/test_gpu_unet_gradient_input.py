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


def test_misaligned_gradient_is_read_on_the_networks_stream():
    side = torch.cuda.Stream()
    net = UNet(2, 16, 7, 6, seed=3, stream=side)
    n, h, w = 2, 16, 32
    x, d = batch(net, n, h, w, seed=5)
    flat = d.view(torch.int16).view(-1)
    torch.cuda.synchronize()
    want = grads_on(side, net, x, flat, n, h, w)
    late = off_by_two(torch.zeros_like(flat))
    a = torch.randn((4096, 4096), device=DEV)
    net.forward(x, n, h, w)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(8):  # some milliseconds before the gradient is there
            a = a @ a * 1e-3
        late.copy_(flat)
    net.backward(late)
    side.synchronize()
    for got, ref in zip([net.dx[: n * h * w * 16]] + parameters(net), want):
        assert torch.equal(got, ref)


def parameters(net):
    return [P[k] for P in net.params.values() for k in ("gw", "gb")]


def grads_on(stream, net, x, d, n, h, w):
    net.forward(x, n, h, w)
    dx = net.backward(d)
    stream.synchronize()
    return [dx[: n * h * w * 16].clone()] + [t.clone() for t in parameters(net)]


def test_parameter_gradients_without_memory_for_all_layers(monkeypatch):
    net = UNet(3, 32, 7, 6, seed=3)
    n, h, w = 2, 16, 48
    x, d = batch(net, n, h, w, seed=5)
    flat = d.view(torch.int16).view(-1)
    want = grads(net, x, flat, n, h, w)
    whole = net._bufs.pop(("part",)).numel()
    buf, asked = net._buf, []

    def short(key, numel, dtype):
        if key == ("part",):
            asked.append(numel)
            if numel > whole // 2:
                raise torch.OutOfMemoryError("no memory for the partial sums of all layers")
        return buf(key, numel, dtype)

    monkeypatch.setattr(net, "_buf", short)
    for t in parameters(net):
        t.fill_(float("nan"))
    got = grads(net, x, flat, n, h, w)
    assert asked[0] == whole and 0 < asked[1] <= whole // 2
    for a, b in zip(got, want):
        assert torch.equal(a, b)
