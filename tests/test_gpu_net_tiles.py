"""The 3x3 convolution and its gradients at the sizes where their tiles end:
pixel groups of 16 (one, two or four in a row of a block), channels from one
tile to more than fit in LDS, and chunks of at most 16, 32, 64 and more pixels
(whole in a block or through partial sums).  Against 64-bit sums of the same
BF16 operands, each with the rounding bound of its sum."""
import numpy as np
import pytest
import torch

qps = pytest.importorskip("qpslice")
qpnet = pytest.importorskip("qpnet")

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _bf(a):
    return qpnet.bits_to_f32(a).double().cpu().numpy()


def _rand(shape, g):
    return qpnet.bf16_bits(torch.randn(shape, generator=g).cuda())


def _taps(x):
    """x (H, W, C) -> (9, H, W, C), tap t the pixel t % 3 - 1 right, t / 3 - 1 down."""
    H, W, _ = x.shape
    p = np.pad(x, ((1, 1), (1, 1), (0, 0)))
    return np.stack([p[t // 3:t // 3 + H, t % 3:t % 3 + W] for t in range(9)])


@pytest.mark.parametrize("H,W", [(1, 1), (5, 16), (7, 17), (3, 33), (9, 48), (4, 65), (2, 150)])
@pytest.mark.parametrize("cin,cout", [(16, 16), (48, 32), (192, 16), (208, 16)])
@pytest.mark.parametrize("masked", [False, True])
def test_convolution_tiles(H, W, cin, cout, masked):
    print(f"[gpu-test] conv {H}x{W} {cin}->{cout} mask {masked}", flush=True)
    g = torch.Generator().manual_seed(H * 1000 + W + cin)
    cs = cin + 16
    x, m, w = _rand((H, W, cs), g), _rand((H, W, cs), g), _rand((9, cout, cin), g)
    b = torch.randn(cout, generator=g).cuda()
    out = torch.zeros((H, W, cout), dtype=torch.int16, device="cuda")
    qpnet.conv3x3(x, H, W, cs, cin, w, b, out, cout, cout, relu=False, mask=m if masked else None)
    xd = _bf(x)[:, :, :cin]
    if masked:
        xd = xd * (_bf(m)[:, :, :cin] > 0)
    t, wd, bd = _taps(xd), _bf(w), b.double().cpu().numpy()
    want = np.einsum("thwc,toc->hwo", t, wd) + bd
    size = np.einsum("thwc,toc->hwo", np.abs(t), np.abs(wd)) + np.abs(bd)
    # the sum in FP32, then half a unit of BF16
    err = np.abs(_bf(out) - want)
    assert (err <= (9 * cin + 2) * EPS * size + 2.0 ** -8 * np.abs(want)).all()


@pytest.mark.parametrize("H,W,nchunk", [(16, 16, 32), (24, 40, 32), (32, 33, 32), (50, 40, 32),
                                        (7, 9, 5), (72, 40, 32), (3, 1000, 7), (1, 5, 40)])
@pytest.mark.parametrize("cin,cout", [(16, 32), (48, 16)])
def test_weight_gradient_chunks(H, W, nchunk, cin, cout):
    print(f"[gpu-test] wgrad {H}x{W} {cin}->{cout} chunks {nchunk}", flush=True)
    g = torch.Generator().manual_seed(H * 1000 + W + cin + nchunk)
    cs, co = cin + 16, cout + 16
    x, dy, y = _rand((H, W, cs), g), _rand((H, W, co), g), _rand((H, W, co), g)
    part = torch.full((nchunk * 9 * cout * cin,), float("nan"), device="cuda")
    dw = torch.full((9, cout, cin), float("nan"), device="cuda")
    db = torch.full((cout,), float("nan"), device="cuda")
    qpnet.conv3x3_wgrad(x, cs, cin, dy, y, co, cout, H, W, part, dw, db, nchunk=nchunk)
    t = _taps(_bf(x)[:, :, :cin])
    d = (_bf(dy) * (_bf(y) > 0))[:, :, :cout]
    want = np.einsum("hwo,thwc->toc", d, t)
    size = np.einsum("hwo,thwc->toc", np.abs(d), np.abs(t))
    n = H * W * EPS
    assert (np.abs(dw.double().cpu().numpy() - want) <= n * size).all()
    assert (np.abs(db.double().cpu().numpy() - d.sum((0, 1))) <= n * np.abs(d).sum((0, 1))).all()
