"""Weight and bias gradients of chunks larger than a block takes whole: a chunk to
four waves (few chunks) and to one (many tiles), runs that end within a step of
four, against 64-bit sums of the same BF16 operands with the rounding bound of the
FP32 sums."""
import pytest
import torch

qps = pytest.importorskip("qpslice")
qpnet = pytest.importorskip("qpnet")

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _rand(shape, g):
    return qpnet.bf16_bits(torch.randn(shape, generator=g).cuda())


def _f64(t):
    return qpnet.bits_to_f32(t).double().cpu()


def _wgrad(H, W, cin, cout, nchunk, bias):
    g = torch.Generator().manual_seed(H * 1000 + W + cin + nchunk)
    cs, co = cin + 16, cout + 16
    x, dy, y = _rand((H, W, cs), g), _rand((H, W, co), g), _rand((H, W, co), g)
    part = torch.full((nchunk * 9 * cout * cin,), float("nan"), device="cuda")
    dw = torch.full((9, cout, cin), float("nan"), device="cuda")
    db = torch.full((cout,), float("nan"), device="cuda") if bias else None
    qpnet.conv3x3_wgrad(x, cs, cin, dy, y, co, cout, H, W, part, dw, db, nchunk=nchunk)
    return (_f64(x)[:, :, :cin], (_f64(dy) * (_f64(y) > 0))[:, :, :cout],
            dw.double().cpu(), db.double().cpu() if bias else None)


def _check(H, W, cin, cout, nchunk, bias):
    print(f"[gpu-test] wgrad {H}x{W} {cin}->{cout} chunks {nchunk} bias {bias}", flush=True)
    x, d, dw, db = _wgrad(H, W, cin, cout, nchunk, bias)
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    dm = d.reshape(H * W, cout).T.contiguous()
    n = H * W * EPS
    for t in range(9):
        xt = p[t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(H * W, cin)
        assert bool(((dw[t] - dm @ xt).abs() <= n * (dm.abs() @ xt.abs())).all()), t
    if bias:
        assert bool(((db - dm.sum(1)).abs() <= n * dm.abs().sum(1)).all())


@pytest.mark.parametrize("H,W,nchunk", [(5, 13, 1), (9, 29, 1), (16, 16, 1), (31, 33, 2),
                                        (40, 77, 7), (64, 65, 32), (130, 200, 100)])
@pytest.mark.parametrize("cin,cout", [(16, 16), (48, 32)])
@pytest.mark.parametrize("bias", [False, True])
def test_few_chunks(H, W, nchunk, cin, cout, bias):
    _check(H, W, cin, cout, nchunk, bias)


@pytest.mark.parametrize("bias", [False, True])
def test_many_tiles(bias):
    _check(47, 51, 192, 192, 29, bias)


@pytest.mark.parametrize("H,W,nchunk", [(130, 100, 144), (130, 100, 145), (131, 100, 200),
                                        (100, 651, 600)])
def test_bias_of_more_chunks_than_taps_and_channels(H, W, nchunk):
    """Its partial sums do not fit where those of the weights leave room."""
    _check(H, W, 16, 32, nchunk, True)
