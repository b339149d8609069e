"""The tiled U-Net kernels at the edges of their tiles and channel blocks, against
the FP64 CPU oracle.  Inputs and weights are BF16 on both sides, so only the FP32
accumulation differs: at most K 2^-24 relative to the sum of magnitudes, about
sqrt(K) 2^-24 of the largest output for K <= 2304 products (convolution) or pixels
(weight gradient); bound 1e-5."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

import unet_oracle as UO  # noqa: E402
from coffeegpu_amd import _lib  # noqa: E402


def bf16_round(x):
    return torch.from_numpy(np.asarray(x, np.float32)).to(torch.bfloat16).double().numpy()


def dev_bf16(x):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(torch.bfloat16).to("cuda:0")


def s():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def p(t):
    return ctypes.c_void_p(t.data_ptr())


# channels staged at once (16, 32, 64, 128, 256) by taps, chunks of 32 with the tile
# heights 4, 8 and 16 and channel blocks of 16, 32 and 64; widths and heights one
# below, at and one above the tiles; 96 channels without the chunk order
@pytest.mark.parametrize("cin,cout,flip,n,h,w", [
    (16, 32, 0, 3, 1, 1), (16, 16, 1, 1, 9, 17), (32, 32, 0, 2, 8, 16), (32, 16, 1, 2, 7, 15),
    (64, 32, 0, 1, 9, 33), (64, 64, 1, 1, 4, 31), (128, 16, 0, 2, 5, 17), (128, 32, 1, 1, 3, 16),
    (256, 16, 0, 1, 4, 16), (256, 48, 1, 2, 5, 3), (256, 128, 0, 1, 3, 16),
    (128, 128, 1, 17, 9, 32), (32, 64, 0, 8, 17, 512), (32, 32, 0, 16, 65, 32), (96, 32, 0, 2, 9, 16)])
def test_conv3x3_tile_edges(cin, cout, flip, n, h, w):
    rng = np.random.default_rng(cin + 3 * cout + h)
    x = bf16_round(rng.standard_normal((n, h, w, cin)))
    W = bf16_round(rng.standard_normal((3, 3, cin, cout)) * 0.2)
    b = rng.standard_normal(cout).astype(np.float32).astype(np.float64)
    want = UO.conv3x3(x, W[::-1, ::-1] if flip else W, b)
    out32 = torch.empty(n * h * w * cout, dtype=torch.float32, device="cuda:0")
    bd = torch.from_numpy(b.astype(np.float32)).to("cuda:0")
    xd, wd = dev_bf16(x), dev_bf16(np.transpose(W.reshape(9, cin, cout), (0, 2, 1)))
    _lib.check(_lib.load().coffee_unet_conv3x3(p(xd), p(wd), p(bd), None, p(out32), n, h, w, cin,
                                               cout, flip, 0, s()))
    got = out32.cpu().numpy().reshape(n, h, w, cout)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()


# channel blocks of 16 and 32 on either side, partial tiles in both directions, one
# range, one tile per range, uneven ranges, no room for the bias partials
@pytest.mark.parametrize("n,h,w,cin,cout,nsplit", [
    (1, 1, 1, 16, 16, 1), (2, 8, 16, 32, 32, 2), (3, 9, 17, 16, 32, 5), (1, 7, 15, 32, 16, 3),
    (2, 17, 33, 96, 48, 7), (5, 8, 16, 48, 96, 4), (1, 25, 16, 256, 256, 4), (2, 9, 31, 32, 64, 100)])
def test_conv3x3_wgrad_tile_edges(n, h, w, cin, cout, nsplit):
    rng = np.random.default_rng(7 * cin + cout + h)
    x = bf16_round(rng.standard_normal((n, h, w, cin)))
    dz = bf16_round(rng.standard_normal((n, h, w, cout)))
    _, dW, db = UO.conv3x3_bwd(x, np.zeros((3, 3, cin, cout)), dz)
    part = torch.empty(nsplit * 9 * cout * cin, dtype=torch.float32, device="cuda:0")
    gw = torch.empty(9 * cout * cin, dtype=torch.float32, device="cuda:0")
    gb = torch.empty(cout, dtype=torch.float32, device="cuda:0")
    xd, dzd = dev_bf16(x), dev_bf16(dz)
    _lib.check(_lib.load().coffee_unet_conv3x3_wgrad(p(xd), p(dzd), p(part), nsplit, p(gw), p(gb),
                                                     n, h, w, cin, cout, s()))
    got = np.transpose(gw.cpu().numpy().reshape(9, cout, cin), (0, 2, 1)).reshape(3, 3, cin, cout)
    assert np.abs(got - dW).max() <= 1e-5 * np.abs(dW).max()
    assert np.abs(gb.cpu().numpy() - db).max() <= 1e-5 * np.abs(db).max()
