"""The kernels a convolution is computed by, chosen from its sizes: the same bits
from either, and the chosen one no slower than the other.  The other one is reached
with an output two bytes off the alignment that the tile kernel asks for."""

import ctypes
import time

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from coffeegpu_amd import _lib  # noqa: E402

DEV = "cuda:0"


def ptr(t):
    return ctypes.c_void_p(t.data_ptr() if t is not None else 0)


def rand(g, *shape):
    return torch.randn(shape, device=DEV, generator=g)


def microseconds(*calls):
    """Of one call of each among others of its own: the least of eight runs of 20, the
    calls in turn."""
    best = [1e30] * len(calls)
    for _ in range(8):
        for k, f in enumerate(calls):
            f()
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                f()
            torch.cuda.synchronize()
            best[k] = min(best[k], (time.perf_counter() - t) / 20 * 1e6)
    return best


# (images, rows, columns), channels in and out: many images of a few pixels, single rows and
# columns, ragged extents with 128 and 256 channels, where the tile took 1.9 to 200
# times as long; the last four are faster with it
@pytest.mark.parametrize("shape,ci,co", [
    ((65536, 1, 1), 64, 64), ((65536, 2, 2), 256, 16), ((8192, 4, 4), 32, 64), ((8, 16384, 1), 16, 16),
    ((8, 1, 16384), 256, 32), ((16, 78, 89), 256, 256), ((12, 48, 134), 128, 128), ((3, 54, 130), 256, 128),
    ((8, 16, 8), 256, 256), ((12, 11, 14), 128, 128), ((1, 256, 255), 16, 16), ((6, 73, 40), 64, 64)])
def test_conv_takes_the_faster_kernel(shape, ci, co):
    n, h, w = shape
    g = torch.Generator(device=DEV).manual_seed(7)
    x = rand(g, n * h * w * ci).bfloat16()
    wt = (rand(g, 9 * co * ci) * (9 * ci) ** -0.5).bfloat16()
    b = rand(g, co)
    y = torch.zeros(n * h * w * co, device=DEV, dtype=torch.bfloat16)
    z = torch.zeros(n * h * w * co + 1, device=DEV, dtype=torch.bfloat16)[1:]
    L, s = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def call(out):
        _lib.check(L.coffee_unet_conv3x3(ptr(x), ptr(wt), ptr(b), ptr(out), None, n, h, w, ci, co, 0, 1, s))

    picked, other = microseconds(lambda: call(y), lambda: call(z))
    assert torch.equal(y, z)
    # 1.4: the estimate that decides is up to a third off, and short calls vary
    assert picked <= 1.4 * other, (picked, other)


# (levels, base, images, rows, columns), and whether the forward and the backward
# pass pay in their fused form: none, the second one, both
@pytest.mark.parametrize("levels,base,n,h,w,pays", [
    (4, 32, 4096, 8, 8, (False, False)), (4, 32, 512, 8, 8, (False, True)), (3, 32, 4096, 4, 4, (False, False)),
    (3, 32, 2048, 4, 4, (False, True)), (4, 32, 3, 40, 72, (True, True))])
def test_network_on_small_images_takes_the_faster_passes(levels, base, n, h, w, pays):
    from coffeegpu_amd.surrogate import UNet, pad16

    net = UNet(levels, base, 7, 6, seed=1)
    g = torch.Generator(device=DEV).manual_seed(h)
    x = rand(g, n * h * w * pad16(7)).bfloat16().view(torch.int16)
    t = rand(g, n * h * w * 6)

    def grads(out):
        loss, d = net.loss_and_grad(out, t, n, h, w)
        dx = net.backward(d)[: n * h * w * 16].clone()
        return [dx] + [P[k].clone() for P in net.params.values() for k in ("gw", "gb")]

    assert net._fused(x, n, h, w)
    want = [net._forward_by_parts(x, n, h, w).clone()]
    want += grads(want[0])
    other = [net._forward_fused(x, n, h, w).clone()]
    other += grads(other[0])
    got = [net.forward(x, n, h, w).clone()]
    assert net._tape[2] == pays[1]
    got += grads(got[0])
    for a, b, c in zip(got, want, other):
        assert torch.equal(a, b) and torch.equal(a, c)
    assert net._pays(n, h, w) == pays
    picked, parts = microseconds(lambda: net.forward(x, n, h, w), lambda: net._forward_by_parts(x, n, h, w))
    # 1.5: the fused pass of 512 x 8 x 8 takes 1.8 times as long as the one by parts
    assert picked <= 1.5 * parts, (picked, parts)


# both orders of products: 32-channel chunks, and taps
@pytest.mark.parametrize("ci,co,w", [(64, 64, 128), (128, 128, 128), (32, 32, 128), (64, 64, 40), (16, 16, 24)])
@pytest.mark.parametrize("off", [1, 2, 3])
def test_bias_at_any_float(ci, co, w, off):
    n, h = 4, 37
    g = torch.Generator(device=DEV).manual_seed(9)
    x = rand(g, n * h * w * ci).bfloat16()
    wt = (rand(g, 9 * co * ci) * (9 * ci) ** -0.5).bfloat16()
    b = rand(g, co + 4)
    L, s = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    outs = []
    for bias in (b[off:off + co].clone(), b[off:off + co]):
        y = torch.zeros(n * h * w * co, device=DEV, dtype=torch.bfloat16)
        z = torch.zeros(n * h * w * co, device=DEV)
        _lib.check(L.coffee_unet_conv3x3(ptr(x), ptr(wt), ptr(bias), ptr(y), ptr(z), n, h, w, ci, co, 0, 1, s))
        outs.append((y, z))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


def test_conv_of_half_a_billion_pixels_keeps_its_order():
    """2^29 pixels and more of a shape summed by 32-channel chunks: the first and last
    images as a call on these alone computes them."""
    n, h, w, ci, co = 65537, 64, 128, 64, 64
    need = n * h * w * (ci + co) * 2
    if torch.cuda.mem_get_info()[0] < need + (8 << 30):
        pytest.skip("needs 137 GB of GPU memory")
    g = torch.Generator(device=DEV).manual_seed(11)
    some = rand(g, 16, h * w * ci).bfloat16()
    x = torch.empty(n, h * w * ci, device=DEV, dtype=torch.bfloat16)
    for k in range(0, n, 16):
        x[k:k + 16] = some[: min(16, n - k)]
    wt = (rand(g, 9 * co * ci) * (9 * ci) ** -0.5).bfloat16()
    b = rand(g, co)
    y = torch.empty(n, h * w * co, device=DEV, dtype=torch.bfloat16)
    z = torch.empty(16, h * w * co, device=DEV, dtype=torch.bfloat16)
    L, s = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for a, out, m in ((x, y, n), (some, z, 16)):
        _lib.check(L.coffee_unet_conv3x3(ptr(a), ptr(wt), ptr(b), ptr(out), None, m, h, w, ci, co, 0, 1, s))
    assert torch.equal(y[:16], z) and torch.equal(y[-1], z[(n - 1) % 16])
    mid = n // 32 * 16
    assert torch.equal(y[mid:mid + 16], z)
    del x, y
    torch.cuda.empty_cache()


# channels and pixels for which the one-layer call takes the kernel with a tap per
# workgroup (whole and partial blocks of 64 channels, ranges of one and many steps, a
# remainder of pixels), and two for which it does not; the many-layer call never does
@pytest.mark.parametrize("shape,ci,co,nsplit", [
    ((16, 91, 79), 64, 64, 224), ((10, 99, 44), 256, 64, 85), ((1, 256, 255), 96, 48, 127), ((3, 33, 33), 96, 48, 1),
    ((8, 67, 93), 96, 64, 97), ((65, 9, 9), 128, 128, 10), ((1, 256, 255), 16, 16, 127), ((2, 24, 148), 256, 256, 13)])
def test_one_layer_weight_gradient_equals_the_many_layer_call(shape, ci, co, nsplit):
    from coffeegpu_amd.surrogate import _WGRAD

    n, h, w = shape
    g = torch.Generator(device=DEV).manual_seed(13)
    x = rand(g, n * h * w * ci).bfloat16()
    dz = rand(g, n * h * w * co).bfloat16()
    L, s = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    part = torch.empty(nsplit * 9 * ci * co, device=DEV)
    gw, gb, mw, mb = (torch.full((m,), float("nan"), device=DEV) for m in (9 * ci * co, co) * 2)
    _lib.check(L.coffee_unet_conv3x3_wgrad(ptr(x), ptr(dz), ptr(part), nsplit, ptr(gw), ptr(gb), n, h, w, ci, co, s))
    layer = _WGRAD.pack(x.data_ptr(), 0, dz.data_ptr(), mw.data_ptr(), mb.data_ptr(), n, h, w, ci, ci, co, 0, nsplit)
    need = ctypes.c_long()
    _lib.check(L.coffee_unet_wgrad_many(layer, 1, None, 0, ctypes.byref(need), s))
    work = torch.empty(need.value, device=DEV)
    _lib.check(L.coffee_unet_wgrad_many(layer, 1, ptr(work), need.value, None, s))
    assert torch.equal(gw, mw) and torch.equal(gb, mb)


def test_weight_gradient_of_two_billion_pixels_keeps_its_order():
    """Past 2^31 pixels, where only some images within one range are not zero: the same
    sums, bit for bit, as over these images alone."""
    n, h, w, c, at = 262145, 64, 128, 16, 100000
    if torch.cuda.mem_get_info()[0] < n * h * w * c * 4 + (8 << 30):
        pytest.skip("needs 138 GB of GPU memory")
    per = -(-n * h * w // 256)
    first = at * h * w
    assert per % 32 == 0 and (first % per) % 32 == 0 and first % per + 4 * h * w <= per
    g = torch.Generator(device=DEV).manual_seed(15)
    x = torch.zeros(n, h * w * c, device=DEV, dtype=torch.bfloat16)
    dz = torch.zeros(n, h * w * c, device=DEV, dtype=torch.bfloat16)
    sx, sz = rand(g, 4, h * w * c).bfloat16(), rand(g, 4, h * w * c).bfloat16()
    x[at:at + 4], dz[at:at + 4] = sx, sz
    part = torch.empty(256 * 9 * c * c, device=DEV)
    L, s = _lib.load(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = []
    for a, b, m, nsplit in ((x, dz, n, 256), (sx, sz, 4, 1)):
        gw = torch.empty(9 * c * c, device=DEV)
        _lib.check(L.coffee_unet_conv3x3_wgrad(ptr(a), ptr(b), ptr(part), nsplit, ptr(gw), None, m, h, w, c, c, s))
        out.append(gw)
    assert torch.equal(*out)
    del x, dz
    torch.cuda.empty_cache()
