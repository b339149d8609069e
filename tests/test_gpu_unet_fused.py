"""The network's passes with pools, upsamplings, concatenations, masks and skip
sums inside the convolutions against the same passes with one kernel each: every
stored activation and activation gradient is rounded at the same places, so
outputs, input gradients and parameter gradients (the same sums in the same order)
are equal bit for bit, and so is the update of all tensors in one launch."""

import ctypes

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd import _lib  # noqa: E402
from coffeegpu_amd.surrogate import UNet, _p, pad16  # noqa: E402


def batch(net, n, h, w, seed):
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    x = torch.randn((n, h, w, pad16(net.cin)), generator=g, device="cuda:0").to(torch.bfloat16)
    t = torch.randn((n, h, w, net.cout), generator=g, device="cuda:0")
    return x.view(torch.int16).view(-1), t.view(-1)


def grads(net):
    return [t.clone() for P in net.params.values() for t in (P["gw"], P["gb"])]


# widths of the coarse levels on and off multiples of 16 (either order of products,
# all of 128 channels with tiles of 8 rows), one-pixel coarse levels, tile heights 4,
# 8 and 16, one level, three-channel-block levels; the last one needs 256 channels in
# pairs of rows and runs by parts
@pytest.mark.parametrize("levels,base,n,h,w,fused", [
    (4, 32, 2, 32, 128, True), (4, 32, 1, 24, 72, True), (4, 32, 3, 8, 8, True),
    (3, 16, 2, 20, 36, True), (2, 32, 9, 64, 256, True), (1, 16, 2, 5, 7, True),
    (3, 64, 1, 16, 64, True), (4, 64, 1, 8, 8, False)])
def test_fused_passes_equal_the_separate_kernels(levels, base, n, h, w, fused):
    net = UNet(levels, base, 7, 6, seed=levels + base)
    x, t = batch(net, n, h, w, seed=h + w)
    assert net._fused(x, n, h, w) == fused
    want = net._forward_by_parts(x, n, h, w).clone()
    wl, d = net.loss_and_grad(want, t, n, h, w)
    wdx = net.backward(d).clone()
    wg = grads(net)
    out = net.forward(x, n, h, w)
    loss, d = net.loss_and_grad(out, t, n, h, w)
    dx = net.backward(d)
    assert torch.equal(out, want) and loss == wl
    assert torch.equal(dx[: n * h * w * 16], wdx[: n * h * w * 16])
    for a, b in zip(grads(net), wg):
        assert torch.equal(a, b)


def test_unaligned_inputs_give_the_same_network():
    net = UNet(2, 16, 7, 6, seed=3)
    n, h, w = 1, 8, 16
    x, t = batch(net, n, h, w, seed=5)
    out = net.forward(x, n, h, w).clone()
    loss, d = net.loss_and_grad(out, t, n, h, w)
    dx = net.backward(d).clone()
    shifted = torch.empty(d.numel() + 1, dtype=torch.int16, device="cuda:0")
    shifted[1:] = d
    net.forward(x, n, h, w)
    assert torch.equal(net.backward(shifted[1:]), dx)
    shifted[1:] = x
    off = net.forward(shifted[1:], n, h, w)  # by parts
    assert float((off - out).abs().max()) <= 3e-2 * float(out.abs().max())


def test_one_launch_update_equals_one_call_per_tensor():
    net = UNet(3, 16, 7, 6, seed=4)
    g = torch.Generator(device="cuda:0").manual_seed(1)
    for P in net.params.values():
        for k in ("gw", "gb", "mw", "mb"):
            P[k].copy_(torch.randn(P[k].shape, generator=g, device="cuda:0"))
        for k in ("vw", "vb"):
            P[k].copy_(torch.rand(P[k].shape, generator=g, device="cuda:0"))
    want = {name: {k: P[k].clone() for k in ("w", "b", "mw", "mb", "vw", "vb")}
            for name, P in net.params.items()}
    L, s = _lib.load(), net._s()
    net.t = 4
    net.adam_step(lr=1e-2)
    for name, P in net.params.items():
        W = want[name]
        for k in ("w", "b"):
            _lib.check(L.coffee_unet_adam(_p(W[k]), _p(P["g" + k]), _p(W["m" + k]), _p(W["v" + k]),
                                          W[k].numel(), 1e-2, 0.9, 0.999, 1e-8, 5, None, None, 0, 0, s))
        for k, v in W.items():
            assert torch.equal(P[k], v), (name, k)
        wb = P["wb"].view(torch.bfloat16).view(9, P["cop"], P["cip"])
        assert torch.equal(wb, P["w"].to(torch.bfloat16))
        wbt = P["wbt"].view(torch.bfloat16).view(9, P["cip"], P["cop"])
        assert torch.equal(wbt, wb.transpose(1, 2).contiguous())


def test_inconsistent_forms_are_refused():
    L = _lib.load()
    one = ctypes.c_void_p(1 << 20)  # never dereferenced
    from coffeegpu_amd.surrogate import _CONV, _WGRAD

    def conv(n=1, h=8, w=16, ci=32, c1=32, co=32, cs=32, up=0, form=0, in2=0, out=1 << 20, pool=0):
        return L.coffee_unet_conv3x3_fused(_CONV.pack(
            1 << 20, in2, 1 << 20, 0, out, 0, 0, 0, 0, pool, n, h, w, ci, c1, co, cs, 0, 0, up, form), one)

    for bad in (dict(h=0), dict(ci=24), dict(c1=16), dict(out=0), dict(up=1, h=7), dict(form=3, w=15),
                dict(form=4), dict(form=1, cs=16), dict(out=(1 << 20) + 2), dict(ci=96, c1=96),
                dict(pool=1 << 20, ci=256, c1=256), dict(form=2, pool=1 << 20)):
        assert conv(**bad) < 0, bad
    layer = _WGRAD.pack(1 << 20, 0, 1 << 20, 1 << 20, 1 << 20, 1, 8, 16, 32, 32, 32, 0, 4)
    need = ctypes.c_long()
    assert L.coffee_unet_wgrad_many(layer, 1, None, 0, ctypes.byref(need), None) == 0
    assert need.value >= 9 * 32 * 32 + 32
    assert L.coffee_unet_wgrad_many(layer, 1, one, need.value - 1, None, None) < 0
