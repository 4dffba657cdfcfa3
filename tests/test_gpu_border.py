"""Border sums formed by the x transforms (nx <= 512) against the deposit's own
border kernel (the separate transforms), which the other tests hold to the
oracle: the deposited planes themselves, with one and two species, tiles in
four, two and one band, in grids whose last x-transform block holds only the
folded row and in grids where it does not exist; the planes' values are what
later slices, diagnostics and the learned seed read.  FP64: 1e-10 of each plane's
peak (rounding alone); FP32: 1e-4 (the slices' FP32 noise is 1e-6 to 1e-5)."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu

PLANES = ("F_CU", "F_DCU", "F_AMU", "F_QE", "F_QB")


def _run(indx, indy, ions, precision, separate):
    ctx = qps.Ctx(indx, indy, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=precision)
    if separate:   # any value but the default takes the separate kernels
        ctx.tune(qps.TUNE_FFT, 0 if precision == qps.FP64 else 1)
    sp = [qps.Species(ctx, ppc=(2, 2))]
    if ions:
        sp.append(qps.Species(ctx, ppc=(1, 1), q=1.0, m=1836.0))
    bm = qps.Beam(ctx, center=(0.4, -0.3, 0.4), sigma=(1.2, 1.0, 0.2), np_=(16, 16, 32), peak=2.0)
    sim = qps.Sim(ctx, sp, [bm])
    sim.begin_step()
    for j in range(1, 5):
        sim.slice(j, iter_max=2)
    out = {k: sim.field(getattr(qps, k)).download(0) for k in PLANES}
    out["part"] = [s.download() for s in sp]
    ctx.close()
    return out


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("ions", [False, True])
@pytest.mark.parametrize("indx,indy", [(4, 4), (6, 5), (5, 8), (7, 8), (8, 7), (8, 8), (8, 9)])
def test_border_sums_in_the_transform(indx, indy, ions, precision):
    print(f"[gpu-test] border {indx} {indy} {ions} {precision}", flush=True)
    p = getattr(qps, precision)
    got, want = _run(indx, indy, ions, p, False), _run(indx, indy, ions, p, True)
    bar = 1e-10 if precision == "FP64" else 1e-4
    for k in PLANES:
        peak = np.abs(want[k]).max()
        assert peak > 0.0, k
        assert np.abs(got[k] - want[k]).max() <= bar * peak, k
    for a, b in zip(got["part"], want["part"]):
        assert a.shape == b.shape
