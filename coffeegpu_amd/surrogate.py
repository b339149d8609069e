"""Learned warm start for the batched log-spherical pulsar runs.

A 2D convolutional U-Net (BF16 weights and activations, FP32 accumulation)
maps the rotating-dipole start of a run (6 field channels, orthonormal
components times r^RPOW, and R_LC as a 7th broadcast channel) to its
near-steady magnetosphere.  Forward, backward and Adam are the project's own
gfx950 kernels (include/coffee_unet.h, coffeegpu_amd/csrc/unet.hip); torch
tensors only hold device memory.  The plain dipole start stays the fallback.

Network (levels L, base channels c0, c_l = c0 2^l): encoder level l = two
3x3 conv + ReLU after a 2x2 average pool (l > 0); decoder level l = nearest
2x upsample, 3x3 conv + ReLU, concatenation with the encoder output of level
l, two 3x3 conv + ReLU; head = 3x3 conv to 6 channels.  Channel counts are
padded to multiples of 16 on the device (padded weights stay zero).
"""

from __future__ import annotations

import ctypes
import struct
from typing import Dict, List, Optional, Tuple

import numpy as np

from . import _lib

RPOW = 2.0  # fields enter the network as orthonormal components times r^RPOW


def _torch():
    import torch

    return torch


def pad16(c: int) -> int:
    return (c + 15) // 16 * 16


def layer_specs(levels: int, base: int, cin: int, cout: int) -> List[Tuple[str, int, int, bool]]:
    """(name, cin, cout, relu) of every convolution, in forward order."""
    specs = []
    c_prev = cin
    for l in range(levels):
        c = base << l
        specs.append((f"enc{l}a", c_prev, c, True))
        specs.append((f"enc{l}b", c, c, True))
        c_prev = c
    for l in range(levels - 2, -1, -1):
        c = base << l
        specs.append((f"dec{l}up", c << 1, c, True))
        specs.append((f"dec{l}a", 2 * c, c, True))
        specs.append((f"dec{l}b", c, c, True))
    specs.append(("head", base, cout, False))
    return specs


def _p(t) -> ctypes.c_void_p:
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


# coffee_unet_conv, coffee_unet_wgrad and coffee_unet_tensor of include/coffee_unet.h
_CONV = struct.Struct("10P11i4x")
_WGRAD = struct.Struct("5P8i")
_TENSOR = struct.Struct("6Pl2i")
_OUT, _MASKED, _POOL_BACK, _UP_BACK = range(4)


def _a(t) -> int:
    return t.data_ptr() if t is not None else 0


class UNet:
    """U-Net on the device.  Parameters: FP32 masters W[tap][co][ci] (padded),
    biases, Adam moments, BF16 copies W and WT."""

    def __init__(self, levels: int = 4, base: int = 32, cin: int = 7, cout: int = 6,
                 seed: int = 0, device: str = "cuda:0", stream=None):
        self.levels, self.base, self.cin, self.cout = levels, base, cin, cout
        self.specs = layer_specs(levels, base, cin, cout)
        self.device = device
        self._lib = _lib.load()
        self._stream = stream
        self.params: Dict[str, dict] = {}
        rng = np.random.default_rng(seed)
        for name, ci, co, relu in self.specs:
            cip, cop = pad16(ci), pad16(co)
            w = np.zeros((9, cop, cip), dtype=np.float32)
            std = np.sqrt(2.0 / (9 * ci))
            w[:, :co, :ci] = (rng.standard_normal((9, co, ci)) * std).astype(np.float32)
            b = np.zeros(cop, dtype=np.float32)
            self.params[name] = self._alloc_param(w, b, ci, co, relu)
        self.t = 0
        self._bufs: Dict[tuple, object] = {}
        self._fusable: Dict[tuple, bool] = {}  # by (n, h, w), as _pay
        self._pay: Dict[tuple, Tuple[bool, bool]] = {}
        # free pinned arrays for the partial sums of the loss (written by the device,
        # summed by the host): one for each thread that is in loss_and_grad
        self._works: List[object] = []

    # ---- parameters ------------------------------------------------------
    def _alloc_param(self, w: np.ndarray, b: np.ndarray, ci: int, co: int, relu: bool) -> dict:
        torch = _torch()
        dev = self.device
        cop, cip = w.shape[1], w.shape[2]
        P = {"ci": ci, "co": co, "cip": cip, "cop": cop, "relu": relu,
             "w": torch.from_numpy(np.ascontiguousarray(w)).to(dev),
             "b": torch.from_numpy(np.ascontiguousarray(b)).to(dev)}
        for k in ("mw", "vw", "gw"):
            P[k] = torch.zeros_like(P["w"])
        for k in ("mb", "vb", "gb"):
            P[k] = torch.zeros_like(P["b"])
        P["wb"] = torch.empty(w.size, dtype=torch.int16, device=dev)
        P["wbt"] = torch.empty(w.size, dtype=torch.int16, device=dev)
        self._refresh_bf16(P)
        return P

    def _refresh_bf16(self, P):
        _lib.check(self._lib.coffee_unet_weights_bf16(_p(P["w"]), _p(P["wb"]), _p(P["wbt"]),
                                                      P["cop"], P["cip"], self._s()))

    def set_params(self, params_np: Dict[str, Tuple[np.ndarray, np.ndarray]]):
        """Load weights given as W[ky, kx, ci, co], b[co] (the oracle's layout)."""
        torch = _torch()
        for name, ci, co, _ in self.specs:
            W, b = params_np[name]
            P = self.params[name]
            w = np.zeros((9, P["cop"], P["cip"]), dtype=np.float32)
            w[:, :co, :ci] = np.transpose(W.reshape(9, ci, co), (0, 2, 1))
            bb = np.zeros(P["cop"], dtype=np.float32)
            bb[:co] = b
            P["w"].copy_(torch.from_numpy(w))
            P["b"].copy_(torch.from_numpy(bb))
            self._refresh_bf16(P)

    def get_grads(self) -> Dict[str, Tuple[np.ndarray, np.ndarray]]:
        """Gradients in the oracle's layout (W[ky, kx, ci, co], b[co])."""
        out = {}
        for name, ci, co, _ in self.specs:
            P = self.params[name]
            g = P["gw"].cpu().numpy()[:, :co, :ci]
            out[name] = (np.transpose(g, (0, 2, 1)).reshape(3, 3, ci, co).astype(np.float64),
                         P["gb"].cpu().numpy()[:co].astype(np.float64))
        return out

    def num_params(self) -> int:
        return sum(9 * ci * co + co for _, ci, co, _ in self.specs)

    def state_dict(self) -> Dict[str, np.ndarray]:
        out = {}
        for name, P in self.params.items():
            out[name + ".w"] = P["w"].cpu().numpy()
            out[name + ".b"] = P["b"].cpu().numpy()
        return out

    # ---- buffers ---------------------------------------------------------
    def _s(self):
        torch = _torch()
        s = self._stream if self._stream is not None else torch.cuda.current_stream()
        return ctypes.c_void_p(s.cuda_stream)

    def _buf(self, key, numel, dtype):
        torch = _torch()
        t = self._bufs.get(key)
        if t is None or t.numel() < numel or t.dtype != dtype:
            t = torch.empty(numel, dtype=dtype, device=self.device)
            self._bufs[key] = t
        return t

    # ---- kernels -----------------------------------------------------------
    def _conv(self, x, P, n, h, w, out, out32=None, relu=None):
        _lib.check(self._lib.coffee_unet_conv3x3(
            _p(x), _p(P["wb"]), _p(P["b"]), _p(out), _p(out32), n, h, w, P["cip"], P["cop"], 0,
            int(P["relu"] if relu is None else relu), self._s()))

    def _convs(self, n: int, h: int, w: int):
        """(forward, backward) sizes n, h, w, cin, cout, pairs of every convolution."""
        for name, _, _, _ in self.specs:
            P = self.params[name]
            l = 0 if name == "head" else int(name[3:].rstrip("abup"))
            pool = name.startswith("enc") and name.endswith("b") and l < self.levels - 1
            yield ((n, h >> l, w >> l, P["cip"], P["cop"], int(pool)),
                   (n, h >> l, w >> l, P["cop"], P["cip"], int(name.endswith("up"))))

    def _fused(self, x, n: int, h: int, w: int) -> bool:
        """Whether every convolution of the two passes can take its neighbours
        (pools, upsamplings, concatenations, masks) into its loads and stores."""
        if h % (1 << self.levels - 1) or w % (1 << self.levels - 1) or x.data_ptr() % 16:
            return False
        ok = self._fusable.get((n, h, w))
        if ok is None:
            fits = self._lib.coffee_unet_conv3x3_fusable
            ok = all(fits(*c) == 1 for pair in self._convs(n, h, w) for c in pair) and all(
                P["cip"] == 2 * P["cop"] for name, P in self.params.items()
                if name.startswith("dec") and name.endswith("a"))
            self._fusable[n, h, w] = ok
        return ok

    def _pays(self, n: int, h: int, w: int) -> Tuple[bool, bool]:
        """Whether the fused form of the (forward, backward) pass is the faster one.
        It saves launches and passes over the activations, measured as about 5.5
        us of a forward and 45 of a backward pass per convolution and 0.6 ns per pixel
        for 32 base channels; but all its convolutions run on tiles, which many
        images of a few pixels leave nearly empty (4 levels of 32 channels, forward:
        512 x 8 x 8 785 us fused and 437 by parts, 4096 x 8 x 8 5.8 and 0.8 ms)."""
        pays = self._pay.get((n, h, w))
        if pays is None:
            passes = 0.6e-3 * n * h * w * self.base / 32
            excess = [sum(self._lib.coffee_unet_conv3x3_excess(*c) for c in p)
                      for p in zip(*self._convs(n, h, w))]
            convs = len(self.specs)
            pays = (excess[0] <= 5.5 * convs + passes, excess[1] <= 45 * convs + passes)
            self._pay[n, h, w] = pays
        return pays

    def forward(self, x, n: int, h: int, w: int):
        """x: BF16 (int16 storage) NHWC tensor with pad16(cin) channels.
        Returns the FP32 NHWC output (pad16(cout) channels, first cout valid)."""
        fused, back = self._pays(n, h, w) if self._fused(x, n, h, w) else (False, False)
        if fused:
            return self._forward_fused(x, n, h, w)
        out = self._forward_by_parts(x, n, h, w)
        if back:
            self._tape = (self._joined_tape(self._tape[0]), n, True)
        return out

    def _joined_tape(self, tape):
        """The tape of the fused forward pass from that of the pass by parts."""
        out, ys = [], {}
        for k, (name, x, y, h, w) in enumerate(tape):
            x2, c1, up = None, self.params[name]["cip"], 0
            if name.endswith("up"):
                x, up = tape[k - 1][2], 1
            elif name.startswith("dec") and name.endswith("a"):
                x, x2, c1 = tape[k - 1][2], ys["enc" + name[3:-1] + "b"], c1 // 2
            ys[name] = y
            out.append((name, x, x2, c1, up, y, h, w))
        return out

    def _conv_fused(self, s, x, x2, c1, up, P, n, h, w, out=None, out32=None, pool=None, *,
                    form=_OUT, out2=None, csplit=0, mask=None, skip=None):
        """forward (form _OUT) or, with the other forms, the backward data pass"""
        back = form != _OUT or c1 is None
        ci, co = (P["cop"], P["cip"]) if back else (P["cip"], P["cop"])
        c = _CONV.pack(_a(x), _a(x2), _a(P["wbt" if back else "wb"]), 0 if back else _a(P["b"]),
                       _a(out), _a(out2), _a(out32), _a(mask), _a(skip), _a(pool), n, h, w, ci,
                       c1 or ci, co, csplit or co, int(back), int(P["relu"] and not back), up, form)
        _lib.check(self._lib.coffee_unet_conv3x3_fused(c, s))

    def _forward_fused(self, x, n, h, w):
        """One launch per convolution.  The pool of an encoder level is stored by
        the convolution before it; upsampled and concatenated inputs are read in
        place.  The tape holds (name, x, x2, cin1, up, y, h, w) per convolution."""
        torch = _torch()
        s = self._s()
        tape = []
        it = iter(self.specs)
        skips = []

        def conv(x, hh, ww, x2=None, c1=None, up=0, pool=None):
            name = next(it)[0]
            P = self.params[name]
            y = self._buf(("y", name), n * hh * ww * P["cop"], torch.int16)
            c1 = c1 or P["cip"]
            self._conv_fused(s, x, x2, c1, up, P, n, hh, ww, y, pool=pool)
            tape.append((name, x, x2, c1, up, y, hh, ww))
            return y, P["cop"]

        cur, hh, ww = x, h, w
        for l in range(self.levels):
            if l > 0:
                cur, hh, ww = pool, hh // 2, ww // 2
            cur, cc = conv(cur, hh, ww)
            pool = None
            if l < self.levels - 1:
                pool = self._buf(("pool", l + 1), n * (hh // 2) * (ww // 2) * cc, torch.int16)
            cur, cc = conv(cur, hh, ww, pool=pool)
            skips.append(cur)
        for l in range(self.levels - 2, -1, -1):
            hh, ww = hh * 2, ww * 2
            cur, cc = conv(cur, hh, ww, up=1)
            cur, cc = conv(cur, hh, ww, x2=skips[l], c1=cc)
            cur, cc = conv(cur, hh, ww)
        name = next(it)[0]
        P = self.params[name]
        out32 = self._buf(("out32",), n * hh * ww * P["cop"], torch.float32)
        self._conv_fused(s, cur, None, P["cip"], 0, P, n, hh, ww, out32=out32)
        tape.append((name, cur, None, P["cip"], 0, None, hh, ww))
        self._tape = (tape, n, True)
        return out32[: n * hh * ww * P["cop"]]

    @staticmethod
    def _nsplit(npix: int) -> int:
        """Pixel ranges of a weight gradient (part of its FP32 sum)."""
        return max(1, min(256, npix // 512))

    def _backward_fused(self, dout):
        """One launch per convolution for the activation gradients, which leave
        each of them as the dz of the convolution before, then all parameter
        gradients."""
        torch = _torch()
        s = self._s()
        tape, n, _ = self._tape
        npix = lambda k: n * tape[k][6] * tape[k][7]  # noqa: E731
        if dout.data_ptr() % 16:
            # a copy on the network's stream, which need not be torch's current one
            c, moved = pad16(self.cout), dout
            dout = self._buf(("dout16",), npix(0) * c, torch.int16)
            _lib.check(self._lib.coffee_unet_combine(_p(dout), c, 0, _p(moved), c, 0, None, 0, 0, None,
                                                     0, 0, c, npix(0), s))
        dzs = {len(tape) - 1: dout}
        dskip = {}

        def dz_of(k):
            dzs[k] = self._buf(("dz", tape[k][0]), npix(k) * self.params[tape[k][0]]["cop"], torch.int16)
            return dzs[k]

        for k in range(len(tape) - 1, -1, -1):
            name, _, _, c1, up, _, hh, ww = tape[k]
            P = self.params[name]
            kw = {}
            if k == 0:
                out = self._buf(("dx", name), npix(k) * P["cip"], torch.int16)
                self._conv_fused(s, dzs[k], None, None, 0, P, n, hh, ww, out)
                self.dx = out
                break
            mask, out = tape[k - 1][5], dz_of(k - 1)
            if up:
                form = _UP_BACK
            elif name.startswith("enc") and name.endswith("a"):
                form = _POOL_BACK
                kw["skip"] = dskip[int(name[3:-1]) - 1]
            else:
                form = _MASKED
                if c1 < P["cip"]:
                    l = int(name[3:-1])
                    kw["csplit"] = c1
                    kw["out2"] = dskip[l] = self._buf(("dskip", l), npix(k) * (P["cip"] - c1), torch.int16)
            self._conv_fused(s, dzs[k], None, None, 0, P, n, hh, ww, out, form=form, mask=mask, **kw)
        self._parameter_gradients([
            _WGRAD.pack(_a(x), _a(x2), _a(dzs[k]), _a(self.params[name]["gw"]),
                        _a(self.params[name]["gb"]), n, hh, ww, self.params[name]["cip"], c1,
                        self.params[name]["cop"], up, self._nsplit(n * hh * ww))
            for k, (name, x, x2, c1, up, _, hh, ww) in enumerate(tape)])
        return self.dx

    def _parameter_gradients(self, layers):
        """All layers together: their partial sums take the most memory of a training
        step's workspaces (base 32, 4 levels: 101 MB on 8 x 64 x 128, 613 MB on 16 x 128 x 256).
        Where that cannot be had, one layer after the other (9 and 75 MB), in 2 launches
        each instead of 3 to 4 for all; the same bits."""
        torch, s = _torch(), self._s()
        many = self._lib.coffee_unet_wgrad_many

        def need(l):
            floats = ctypes.c_long()
            _lib.check(many(b"".join(l), len(l), None, 0, ctypes.byref(floats), s))
            return floats.value

        groups = [layers]
        try:
            part = self._buf(("part",), need(layers), torch.float32)
        except torch.OutOfMemoryError:
            groups = [[l] for l in layers]
            part = self._buf(("part",), max(map(need, groups)), torch.float32)
        for g in groups:
            _lib.check(many(b"".join(g), len(g), _p(part), part.numel(), None, s))

    def _forward_by_parts(self, x, n, h, w):
        torch = _torch()
        L = self.levels
        tape = []
        it = iter(self.specs)
        skips = []
        cur, cc, hh, ww = x, pad16(self.cin), h, w
        for l in range(L):
            if l > 0:
                pooled = self._buf(("pool", l), n * (hh // 2) * (ww // 2) * cc, torch.int16)
                _lib.check(self._lib.coffee_unet_pool2(_p(cur), _p(pooled), n, hh, ww, cc, self._s()))
                cur, hh, ww = pooled, hh // 2, ww // 2
            for part in ("a", "b"):
                name = next(it)[0]
                P = self.params[name]
                y = self._buf(("y", name), n * hh * ww * P["cop"], torch.int16)
                self._conv(cur, P, n, hh, ww, y)
                tape.append((name, cur, y, hh, ww))
                cur, cc = y, P["cop"]
            skips.append((cur, cc, hh, ww))
        for l in range(L - 2, -1, -1):
            up = self._buf(("up", l), n * (hh * 2) * (ww * 2) * cc, torch.int16)
            hh, ww = hh * 2, ww * 2
            _lib.check(self._lib.coffee_unet_up2(_p(cur), _p(up), n, hh, ww, cc, self._s()))
            name = next(it)[0]
            P = self.params[name]
            y = self._buf(("y", name), n * hh * ww * P["cop"], torch.int16)
            self._conv(up, P, n, hh, ww, y)
            tape.append((name, up, y, hh, ww))
            sk, skc, _, _ = skips[l]
            c = P["cop"]
            cat = self._buf(("cat", l), n * hh * ww * 2 * c, torch.int16)
            npix = n * hh * ww
            _lib.check(self._lib.coffee_unet_combine(_p(cat), 2 * c, 0, _p(y), c, 0, None, 0, 0,
                                                     None, 0, 0, c, npix, self._s()))
            _lib.check(self._lib.coffee_unet_combine(_p(cat), 2 * c, c, _p(sk), skc, 0, None, 0,
                                                     0, None, 0, 0, c, npix, self._s()))
            cur, cc = cat, 2 * c
            for part in ("a", "b"):
                name = next(it)[0]
                P = self.params[name]
                y = self._buf(("y", name), n * hh * ww * P["cop"], torch.int16)
                self._conv(cur, P, n, hh, ww, y)
                tape.append((name, cur, y, hh, ww))
                cur, cc = y, P["cop"]
        name = next(it)[0]
        P = self.params[name]
        out32 = self._buf(("out32",), n * hh * ww * P["cop"], torch.float32)
        self._conv(cur, P, n, hh, ww, None, out32=out32, relu=False)
        tape.append((name, cur, None, hh, ww))
        self._tape = (tape, n, False)
        return out32[: n * hh * ww * P["cop"]]

    def backward(self, dout):
        """dout: BF16 gradient of the loss w.r.t. the FP32 output (same layout).
        Fills every parameter's gradient (gw, gb)."""
        if self._tape[2]:
            return self._backward_fused(dout)
        torch = _torch()
        tape, n, _ = self._tape
        pos = [len(tape) - 1]

        def conv_back(dz):
            name, xin, y, hh, ww = tape[pos[0]]
            pos[0] -= 1
            P = self.params[name]
            npix = n * hh * ww
            nsplit = self._nsplit(npix)
            part = self._buf(("part",), nsplit * 9 * P["cop"] * P["cip"], torch.float32)
            _lib.check(self._lib.coffee_unet_conv3x3_wgrad(
                _p(xin), _p(dz), _p(part), nsplit, _p(P["gw"]), _p(P["gb"]), n, hh, ww, P["cip"],
                P["cop"], self._s()))
            dx = self._buf(("dx", name), npix * P["cip"], torch.int16)
            _lib.check(self._lib.coffee_unet_conv3x3(
                _p(dz), _p(P["wbt"]), None, _p(dx), None, n, hh, ww, P["cop"], P["cip"], 1, 0,
                self._s()))
            return dx, P["cip"], hh, ww

        def masked(key, a, ast, aoff, c, y, npix, b=None, bst=0, boff=0):
            out = self._buf(("dz", key), npix * c, torch.int16)
            _lib.check(self._lib.coffee_unet_combine(_p(out), c, 0, _p(a), ast, aoff, _p(b), bst,
                                                     boff, _p(y), c, 0, c, npix, self._s()))
            return out

        L = self.levels
        d, dc, hh, ww = conv_back(dout)  # head (no activation)
        dcat = [None] * L
        for l in range(0, L - 1):
            for part in ("b", "a"):
                name, _, y, hh, ww = tape[pos[0]]
                c = self.params[name]["cop"]
                dz = masked(name, d, dc, 0, c, y, n * hh * ww)
                d, dc, hh, ww = conv_back(dz)
            # d: gradient of concat(y_up, skip_l), 2c channels
            dcat[l] = (d, dc)
            name, _, y, hh, ww = tape[pos[0]]
            c = self.params[name]["cop"]
            dz = masked(name, d, dc, 0, c, y, n * hh * ww)
            d, dc, hh, ww = conv_back(dz)
            up = self._buf(("dup", l), n * (hh // 2) * (ww // 2) * dc, torch.int16)
            _lib.check(self._lib.coffee_unet_up2_bwd(_p(d), _p(up), n, hh, ww, dc, self._s()))
            d, hh, ww = up, hh // 2, ww // 2
        for l in range(L - 1, -1, -1):
            name, _, y, hh, ww = tape[pos[0]]
            c = self.params[name]["cop"]
            if dcat[l] is not None:
                dcl, dcc = dcat[l]
                dz = masked(name, d, dc, 0, c, y, n * hh * ww, b=dcl, bst=dcc, boff=dcc // 2)
            else:
                dz = masked(name, d, dc, 0, c, y, n * hh * ww)
            d, dc, hh, ww = conv_back(dz)
            name, _, y, hh, ww = tape[pos[0]]
            c = self.params[name]["cop"]
            dz = masked(name, d, dc, 0, c, y, n * hh * ww)
            d, dc, hh, ww = conv_back(dz)
            if l > 0:
                pd = self._buf(("dpool", l), n * (hh * 2) * (ww * 2) * dc, torch.int16)
                _lib.check(self._lib.coffee_unet_pool2_bwd(_p(d), _p(pd), n, hh * 2, ww * 2, dc,
                                                           self._s()))
                d, hh, ww = pd, hh * 2, ww * 2
        self.dx = d
        return d

    def loss_and_grad(self, out32, target, n: int, h: int, w: int) -> Tuple[float, object]:
        torch = _torch()
        cop = pad16(self.cout)
        dout = self._buf(("dout",), n * h * w * cop, torch.int16)
        loss = ctypes.c_double()
        try:
            work = self._works.pop()
        except IndexError:
            work = torch.empty(1024, dtype=torch.float64, pin_memory=True)
        try:
            _lib.check(self._lib.coffee_unet_mse_pinned(_p(out32), cop, _p(target), self.cout,
                                                        n * h * w, _p(dout), _p(work),
                                                        ctypes.byref(loss), self._s()))
        finally:
            self._works.append(work)
        return loss.value, dout

    def adam_step(self, lr: float = 1e-3, beta1: float = 0.9, beta2: float = 0.999,
                  eps: float = 1e-8):
        self.t += 1
        tensors = b"".join(
            _TENSOR.pack(_a(P["w"]), _a(P["gw"]), _a(P["mw"]), _a(P["vw"]), _a(P["wb"]),
                         _a(P["wbt"]), P["w"].numel(), P["cop"], P["cip"])
            + _TENSOR.pack(_a(P["b"]), _a(P["gb"]), _a(P["mb"]), _a(P["vb"]), 0, 0,
                           P["b"].numel(), 0, 0)
            for P in self.params.values())
        _lib.check(self._lib.coffee_unet_adam_many(tensors, 2 * len(self.params), lr, beta1, beta2,
                                                   eps, self.t, self._s()))
