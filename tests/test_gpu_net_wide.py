"""The 3x3 convolution with all output channels in a wave, which planes of many
pixel groups take for channel counts that no other kernel is compiled for, and for
operands not aligned to 16 bytes: ragged rows, masked and not, ReLU and addition
into the output, against 64-bit sums of the same BF16 operands with the rounding
bound of each sum."""
import pytest
import torch

qps = pytest.importorskip("qpslice")
qpnet = pytest.importorskip("qpnet")

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _rand(shape, g):
    return qpnet.bf16_bits(torch.randn(shape, generator=g).cuda())


def _conv(x, w):
    """x (H, W, cin), w (9, cout, cin), both doubles on the CPU."""
    cout, cin = w.shape[1:]
    k = w.reshape(3, 3, cout, cin).permute(2, 3, 0, 1)
    return torch.nn.functional.conv2d(x.permute(2, 0, 1)[None], k, padding=1)[0].permute(1, 2, 0)


@pytest.mark.parametrize("H,W,cin,cout,pad,off", [
    (97, 258, 80, 96, 4, 0), (50, 500, 256, 32, 4, 0), (113, 500, 32, 32, 4, 4),
    (193, 256, 16, 32, 8, 0), (100, 250, 16, 96, 8, 0), (260, 250, 48, 112, 8, 0),
    (241, 275, 32, 192, 8, 0)])
@pytest.mark.parametrize("masked", [False, True])
def test_wide_convolution(H, W, cin, cout, pad, off, masked):
    print(f"[gpu-test] wide conv {H}x{W} {cin}->{cout} off {off} mask {masked}", flush=True)
    g = torch.Generator().manual_seed(H + W + cin)
    cs = cin + pad
    x, m, w = _rand((H, W, cs), g), _rand((H, W, cs), g), _rand((9, cout, cin), g)
    b = torch.randn(cout, generator=g).cuda()
    was = _rand((H, W, cout), g)
    out = was.clone()
    # a pixel's last channel but off is the next pixel's: the rows hold cs channels
    pad = torch.zeros(off, dtype=torch.int16, device="cuda")
    xf, mf = (torch.cat([t.reshape(-1), pad]) for t in (x, m))
    qpnet.conv3x3(xf, H, W, cs, cin, w, b, out, cout, cout, relu=not masked, accum=masked,
                  mask=mf if masked else None, x_off=off)
    f64 = lambda t: qpnet.bits_to_f32(t).double().cpu()  # noqa: E731
    xd, md = (f64(t)[off:off + H * W * cs].reshape(H, W, cs)[:, :, :cin] for t in (xf, mf))
    if masked:
        xd = xd * (md > 0)
    wd, bd = f64(w), b.double().cpu()
    want, size = _conv(xd, wd) + bd, _conv(xd.abs(), wd.abs()) + bd.abs()
    if masked:
        want, size = want + f64(was), size + f64(was).abs()
    else:
        want = want.clamp(min=0.0)
    # the sum of 9 cin + 2 terms in FP32, then half a unit of BF16
    bar = (9 * cin + 3) * EPS * size + 2.0 ** -8 * (want.abs() + (9 * cin + 3) * EPS * size)
    assert bool(((f64(out) - want).abs() <= bar).all())
