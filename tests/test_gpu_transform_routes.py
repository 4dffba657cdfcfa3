"""The transforms of whole fields through transposed planes (the x pass stores or
reads the columns of the y pass) against the form with a transpose of its own,
which the other tests hold to the oracle: every length on either side, one to
three components, sine and cosine kinds, forward, and back with the guard row.
Both run the same 2n-point transforms, whose rounding is at most about
2 log2(2n) units of the largest value: 64 2^-24 of the peak covers two passes."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("indx,indy", [(4, 4), (4, 10), (5, 6), (6, 5), (7, 4), (8, 8), (9, 8),
                                       (9, 9), (10, 7), (10, 10), (11, 6), (6, 11), (11, 11)])
def test_transform_routes_agree(indx, indy):
    print(f"[gpu-test] transform routes {indx} {indy}", flush=True)
    ctx = qps.Ctx(indx, indy, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=qps.FP32)
    rng = np.random.default_rng(indx + 16 * indy)
    for dim, kind in ((1, 1), (2, 1), (3, 1), (3, 2), (3, 3)):
        x = rng.standard_normal((dim, ctx.ny + 1, ctx.nx + 1))
        res = []
        for tune in (-1, 3):   # the default, and the transpose with other LDS padding
            ctx.tune(qps.TUNE_FFT, tune)
            f = qps.Field2d(ctx, dim)
            f.upload(x, space=0)
            f.fftrk(kind)
            k = f.download(1)
            f.fftkr(kind)
            res.append((k, f.download(0)))
        for a, b in zip(*res):
            peak = np.abs(b).max()
            assert peak > 0.0
            assert np.abs(a - b).max() <= 64 * 2.0 ** -24 * peak, (dim, kind)
    ctx.close()
