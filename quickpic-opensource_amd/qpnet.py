"""The learned corrector seed: a 4-level U-Net (3x3 convolutions, 16-32-64-128
channels, average pooling, nearest upsampling, skip concatenations, a 1x1
FP32 output layer) whose forward and backward passes are the library's own
BF16-MFMA kernels (include/qpnet.h).  PyTorch only provides device memory and
the stream.

Input channels (8): B_perp of the two previous slices (real space, 4), and of
the current slice the plasma charge, the predictor current J_x, J_y and psi.
Output (2): the correction of B_perp over its linear extrapolation
2 B(xi-1) - B(xi-2).  The network only seeds the corrector; the plain
iteration to the residual tolerance decides the answer.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import torch

import qpslice as qps

CH = (16, 32, 64, 128)
NIN, NOUT = 8, 2

_NET = None


def _lib():
    global _NET
    if _NET is None:
        L = qps.lib()
        vp, i, sz, f, u16p, fp, dp = (C.c_void_p, C.c_int, C.c_size_t, C.c_float, C.c_void_p,
                                      C.c_void_p, C.c_void_p)
        sig = {
            "qp_net_conv3x3": [vp, u16p, u16p, i, i, i, i, u16p, fp, u16p, i, i, i, i],
            "qp_net_conv3x3_wgrad": [vp, u16p, i, i, u16p, u16p, i, i, i, i, i, fp, fp, fp],
            "qp_net_flip_weights": [vp, u16p, i, i, u16p],
            "qp_net_pool2": [vp, u16p, i, u16p, i, i, i, i],
            "qp_net_pool2_bwd": [vp, u16p, i, u16p, i, i, i, i, i],
            "qp_net_up2": [vp, u16p, i, u16p, i, i, i, i],
            "qp_net_up2_bwd": [vp, u16p, i, u16p, i, i, i, i],
            "qp_net_pack_input": [vp, fp, i, sz, i, fp, i, i, u16p, i],
            "qp_net_head": [vp, u16p, i, i, fp, fp, i, sz, fp],
            "qp_net_head_bwd": [vp, u16p, i, i, fp, i, sz, fp, u16p, i, fp, fp],
            "qp_net_mse": [vp, fp, fp, sz, fp, dp, i],
            "qp_net_adam": [vp, fp, fp, fp, fp, sz, f, f, f, f, i, u16p],
            "qp_net_unet_forward": [vp, vp, fp, sz, i],
            "qp_net_unet_backward": [vp, vp, fp],
            "qp_net_adam_params": [vp, vp, i, f, f, f, f, i],
            "qp_net_to_bf16": [vp, fp, sz, u16p],
            "qp_net_block_mean": [vp, i, C.POINTER(C.c_void_p), C.POINTER(C.c_int), i, i, i, i,
                                  fp],
            "qp_net_seed_apply": [vp, fp, i, i, i, f, fp, fp, i, sz, vp, i, i, sz, i, i],
            "qp_net_seed_combine": [vp, vp, vp, vp, sz, i, i],
            "qp_net_graph_begin": [vp],
            "qp_net_graph_end": [vp, C.POINTER(C.c_void_p)],
            "qp_net_graph_launch": [vp, vp],
            "qp_net_graph_destroy": [vp],
        }
        for name, args in sig.items():
            fn = getattr(L, name)
            fn.argtypes = args
            fn.restype = C.c_int
        _NET = L
    return _NET


class _Conv(C.Structure):
    _fields_ = [(k, C.c_void_p) for k in ("w", "b", "wt", "gw", "gb")] + \
        [("cin", C.c_int), ("cout", C.c_int)]


class _Unet(C.Structure):
    """qp_net_unet; a and g: x0, ea[3], cat[3], pool[3], ba, bb, da[3], db[3]."""
    _fields_ = [("conv", _Conv * 14), ("a", C.c_void_p * 18), ("g", C.c_void_p * 18)] + \
        [(k, C.c_void_p) for k in ("in_scale", "hw", "hb", "ghwb", "out", "gout", "mse_part",
                                   "part")] + \
        [("npart", C.c_size_t), ("c", C.c_int * 4)] + \
        [(k, C.c_int) for k in ("nin", "nout", "H", "W", "nmse", "nhead", "nchunk")]


# the network's maps in the order of qp_net_maps
MAPS = ("x0", "e1a", "e2a", "e3a", "cat1", "cat2", "cat3", "p1", "p2", "p3", "ba", "bb",
        "d1a", "d2a", "d3a", "d1b", "d2b", "d3b")


class _Param(C.Structure):
    _fields_ = [(k, C.c_void_p) for k in ("w", "g", "m", "v", "wb")] + [("n", C.c_size_t)]


def _call(fn, *args):
    rc = fn(*args)
    if rc != 0:
        raise qps.QPError(rc, qps.lib().qp_last_error().decode())


def ptr(t, offset=0):
    """Device address of a tensor, plus an element offset."""
    return C.c_void_p(t.data_ptr() + offset * t.element_size()) if t is not None else None


def stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def block_mean(planes, f, H, W, out):
    """planes: list of (device address, row pitch, is_fp64); out: FP32
    tensor [len(planes)][H][W] of f x f block means."""
    n = len(planes)
    ps = (C.c_void_p * n)(*[p for p, _, _ in planes])
    lds = (C.c_int * n)(*[ld for _, ld, _ in planes])
    dbl = sum(1 << c for c, (_, _, d) in enumerate(planes) if d)
    _call(_lib().qp_net_block_mean, stream(), n, ps, lds, dbl, f, H, W, ptr(out))


def seed_apply(corr, H, W, f, s, hist, dst, dst_double, ld_d, pl_d, ny1, nx1):
    """dst <- 2 hist[0] - hist[1] + s up(corr) (see qpnet.h), or s up(corr)
    when hist is None; hist: FP32 tensor [2][2][ny1][nx1]; dst: device address
    of the 2-component plane."""
    a, b = (ptr(hist[0]), ptr(hist[1])) if hist is not None else (None, None)
    _call(_lib().qp_net_seed_apply, stream(), ptr(corr), H, W, f, s, a, b, nx1, ny1 * nx1,
          C.c_void_p(dst), 1 if dst_double else 0, ld_d, pl_d, ny1, nx1)


def seed_combine(epw, hist, corr, n, extrap, dbl):
    """k space: e = epw; epw = 2 e - hist (+ corr) if extrap; hist = e
    (device addresses; corr may be None)."""
    _call(_lib().qp_net_seed_combine, stream(), C.c_void_p(epw), C.c_void_p(hist),
          C.c_void_p(corr) if corr else None, n, 1 if extrap else 0, 1 if dbl else 0)


def bf16_bits(a: torch.Tensor) -> torch.Tensor:
    """float32 -> BF16 bit patterns (int16 tensor), round to nearest even."""
    return a.to(torch.bfloat16).view(torch.int16)


def bits_to_f32(b: torch.Tensor) -> torch.Tensor:
    return b.view(torch.bfloat16).to(torch.float32)


# ---------------------------------------------------------------------------
# layer-level entry points (also used by the tests)
# ---------------------------------------------------------------------------
def conv3x3(x, H, W, cs_in, cin, w16, bias, out, cs_out, cout, relu=True, accum=False,
            mask=None, x_off=0, out_off=0):
    _call(_lib().qp_net_conv3x3, stream(), ptr(x, x_off), ptr(mask, x_off) if mask is not None
          else None, H, W, cs_in, cin, ptr(w16), ptr(bias), ptr(out, out_off), cs_out, cout,
          1 if relu else 0, 1 if accum else 0)


def conv3x3_wgrad(x, cs_in, cin, dy, yout, cs_out, cout, H, W, part, dw, db, x_off=0,
                  y_off=0, nchunk=32):
    _call(_lib().qp_net_conv3x3_wgrad, stream(), ptr(x, x_off), cs_in, cin, ptr(dy, y_off),
          ptr(yout, y_off), cs_out, cout, H, W, nchunk, ptr(part), ptr(dw), ptr(db))


def flip_weights(w16, cout, cin, wt):
    _call(_lib().qp_net_flip_weights, stream(), ptr(w16), cout, cin, ptr(wt))


class Conv:
    """3x3 convolution with ReLU: FP32 master weights [9][cout][cin], their
    BF16 copy, FP32 bias, gradients and Adam moments."""

    def __init__(self, cin, cout, gen, dev):
        self.cin, self.cout = cin, cout
        fan_in = 9 * cin
        w = torch.randn((9, cout, cin), generator=gen) * np.sqrt(2.0 / fan_in)
        self.w = w.to(dev)
        self.b = torch.zeros(cout, device=dev)
        self.w16 = bf16_bits(self.w)
        self.wt16 = torch.empty_like(self.w16)
        self.gw = torch.zeros_like(self.w)
        self.gb = torch.zeros_like(self.b)
        self.m = [torch.zeros_like(self.w), torch.zeros_like(self.b)]
        self.v = [torch.zeros_like(self.w), torch.zeros_like(self.b)]

    def params(self):
        return [(self.w, self.gw, self.m[0], self.v[0], self.w16), (self.b, self.gb, self.m[1],
                                                                     self.v[1], None)]


class UNet:
    """The 4-level U-Net.  Buffers are allocated per input size (H, W
    divisible by 8)."""

    def __init__(self, seed=0, device="cuda"):
        gen = torch.Generator().manual_seed(seed)
        self.dev = torch.device(device)
        c1, c2, c3, c4 = CH
        self.enc = [Conv(16, c1, gen, self.dev), Conv(c1, c1, gen, self.dev),
                    Conv(c1, c2, gen, self.dev), Conv(c2, c2, gen, self.dev),
                    Conv(c2, c3, gen, self.dev), Conv(c3, c3, gen, self.dev),
                    Conv(c3, c4, gen, self.dev), Conv(c4, c4, gen, self.dev)]
        self.dec = [Conv(c4 + c3, c3, gen, self.dev), Conv(c3, c3, gen, self.dev),
                    Conv(c3 + c2, c2, gen, self.dev), Conv(c2, c2, gen, self.dev),
                    Conv(c2 + c1, c1, gen, self.dev), Conv(c1, c1, gen, self.dev)]
        hw = torch.randn((NOUT, c1), generator=gen) * np.sqrt(1.0 / c1) * 0.1
        self.hw = hw.to(self.dev)
        self.hb = torch.zeros(NOUT, device=self.dev)
        self.ghwb = torch.zeros(NOUT * (c1 + 1), device=self.dev)
        self.hm = [torch.zeros_like(self.hw), torch.zeros_like(self.hb)]
        self.hv = [torch.zeros_like(self.hw), torch.zeros_like(self.hb)]
        self.in_scale = torch.ones(NIN, device=self.dev)
        self.out_scale = 1.0
        self.step = 0
        self._shape = None
        self._graph = None     # (key, executable graph) of the captured forward

    # -- buffers ------------------------------------------------------------
    def _alloc(self, H, W):
        if self._shape == (H, W):
            return
        assert H % 8 == 0 and W % 8 == 0
        c1, c2, c3, c4 = CH
        z = lambda h, w, c: torch.zeros((h * w * c,), dtype=torch.int16, device=self.dev)  # noqa
        s = {}
        s["x0"] = z(H, W, 16)
        s["e1a"] = z(H, W, c1)
        s["cat1"] = z(H, W, c2 + c1)
        s["p1"] = z(H // 2, W // 2, c1)
        s["e2a"] = z(H // 2, W // 2, c2)
        s["cat2"] = z(H // 2, W // 2, c3 + c2)
        s["p2"] = z(H // 4, W // 4, c2)
        s["e3a"] = z(H // 4, W // 4, c3)
        s["cat3"] = z(H // 4, W // 4, c4 + c3)
        s["p3"] = z(H // 8, W // 8, c3)
        s["ba"] = z(H // 8, W // 8, c4)
        s["bb"] = z(H // 8, W // 8, c4)
        s["d3a"] = z(H // 4, W // 4, c3)
        s["d3b"] = z(H // 4, W // 4, c3)
        s["d2a"] = z(H // 2, W // 2, c2)
        s["d2b"] = z(H // 2, W // 2, c2)
        s["d1a"] = z(H, W, c1)
        s["d1b"] = z(H, W, c1)
        self.a = s
        self.g = {k: torch.zeros_like(v) for k, v in s.items()}
        self.out = torch.zeros((NOUT, H * W), device=self.dev)
        self.gout = torch.zeros_like(self.out)
        # partial sums of the gradients: the layers of the two finer levels, and
        # of the coarser ones where they have as many pixels
        cut = [sum(10 * v.cin * v.cout for v in cv) for cv in self._levels()]
        npart = 32 * sum(n for i, n in enumerate(cut) if i < 2 or H * W >> 2 * i > 2048)
        self.part = torch.zeros(max(npart, 64 * NOUT * (c1 + 1)), device=self.dev)
        self.mse_part = torch.zeros(256, dtype=torch.float64, device=self.dev)
        self._shape = (H, W)

    def _levels(self):
        """The convolutions on the grid coarsened 1, 2, 4 and 8 times."""
        e, d = self.enc, self.dec
        return [e[0:2] + d[4:6], e[2:4] + d[2:4], e[4:6] + d[0:2], e[6:8]]

    def _table(self):
        """The network's buffers for qp_net_unet_forward and _backward."""
        p = torch.Tensor.data_ptr
        t = _Unet((_Conv * 14)(*[(p(v.w16), p(v.b), p(v.wt16), p(v.gw), p(v.gb), v.cin, v.cout)
                                 for v in self.enc + self.dec]),
                  (C.c_void_p * 18)(*[p(self.a[k]) for k in MAPS]),
                  (C.c_void_p * 18)(*[p(self.g[k]) for k in MAPS]),
                  *[p(x) for x in (self.in_scale, self.hw, self.hb, self.ghwb, self.out, self.gout,
                                   self.mse_part, self.part)],
                  self.part.numel(), CH, NIN, NOUT, *self._shape, self.mse_part.numel(), 64, 32)
        return t

    # -- forward --------------------------------------------------------------
    def forward(self, planes, plane, ld, H, W):
        """planes: FP32 device tensor holding NIN planes (plane elements apart,
        row pitch ld); returns the FP32 output [NOUT][H*W] (in output units)."""
        self._alloc(H, W)
        _call(_lib().qp_net_unet_forward, stream(), C.byref(self._table()), ptr(planes), plane, ld)
        return self.out

    def forward_graph(self, planes, plane, ld, H, W):
        """forward() replayed from a HIP graph captured on the first call
        with these buffers and sizes (the weights are read at replay, so
        training between replays is seen); returns the output buffer.  The
        legacy null stream cannot be captured: from it, the graph runs on a
        side stream ordered after and before the caller's work."""
        cur = torch.cuda.current_stream()
        if cur.cuda_stream == 0:
            if getattr(self, "_side", None) is None:
                self._side = torch.cuda.Stream()
            self._side.wait_stream(cur)
            with torch.cuda.stream(self._side):
                out = self.forward_graph(planes, plane, ld, H, W)
            cur.wait_stream(self._side)
            return out
        key = (planes.data_ptr(), plane, ld, H, W, cur.cuda_stream)
        if self._graph is None or self._graph[0] != key:
            self.drop_graph()
            self.forward(planes, plane, ld, H, W)   # buffers allocated outside the capture
            st = stream()
            _call(_lib().qp_net_graph_begin, st)
            try:
                self.forward(planes, plane, ld, H, W)
            finally:
                ge = C.c_void_p()
                _call(_lib().qp_net_graph_end, st, C.byref(ge))
            self._graph = (key, ge)
            return self.out
        _call(_lib().qp_net_graph_launch, self._graph[1], stream())
        return self.out

    def drop_graph(self):
        if self._graph is not None:
            _call(_lib().qp_net_graph_destroy, self._graph[1])
            self._graph = None

    # -- backward -------------------------------------------------------------
    def backward(self, target):
        """MSE against target [NOUT][H*W] (output units); fills every
        gradient; returns the loss."""
        n = self.out.numel()
        _call(_lib().qp_net_unet_backward, stream(), C.byref(self._table()), ptr(target))
        return float(self.mse_part.sum().item()) / n

    def adam(self, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8):
        self.step += 1
        ps = [_Param(w.data_ptr(), gw.data_ptr(), m.data_ptr(), v.data_ptr(),
                     w16.data_ptr() if w16 is not None else None, w.numel())
              for cv in self.enc + self.dec for w, gw, m, v, w16 in cv.params()]
        # the head's gradients: per output a row of its weights' and its bias's
        c1 = CH[0]
        for o in range(NOUT):
            for n, at, off, t in ((c1, o * c1, 0, (self.hw, self.hm[0], self.hv[0])),
                                  (1, o, c1, (self.hb, self.hm[1], self.hv[1]))):
                w, m, v = (x.data_ptr() + 4 * at for x in t)
                ps.append(_Param(w, self.ghwb.data_ptr() + 4 * (o * (c1 + 1) + off), m, v, None, n))
        _call(_lib().qp_net_adam_params, stream(), (_Param * len(ps))(*ps), len(ps), lr, b1, b2,
              eps, self.step)

    # -- persistence ------------------------------------------------------------
    def state(self):
        d = {f"enc{i}_w": c.w.cpu() for i, c in enumerate(self.enc)}
        d.update({f"enc{i}_b": c.b.cpu() for i, c in enumerate(self.enc)})
        d.update({f"dec{i}_w": c.w.cpu() for i, c in enumerate(self.dec)})
        d.update({f"dec{i}_b": c.b.cpu() for i, c in enumerate(self.dec)})
        d.update({"head_w": self.hw.cpu(), "head_b": self.hb.cpu(),
                  "in_scale": self.in_scale.cpu(),
                  "out_scale": torch.tensor([self.out_scale])})
        return d

    def load(self, d):
        for i, c in enumerate(self.enc):
            c.w.copy_(d[f"enc{i}_w"])
            c.b.copy_(d[f"enc{i}_b"])
            c.w16.copy_(bf16_bits(c.w))
        for i, c in enumerate(self.dec):
            c.w.copy_(d[f"dec{i}_w"])
            c.b.copy_(d[f"dec{i}_b"])
            c.w16.copy_(bf16_bits(c.w))
        self.hw.copy_(d["head_w"])
        self.hb.copy_(d["head_b"])
        self.in_scale.copy_(d["in_scale"])
        self.out_scale = float(d["out_scale"][0])
