"""The slice loop's fused field solves (y transforms and modes in one kernel)
against the separate transforms and k-space kernels, which the other tests hold
to the oracle, on every transform length and on non-square grids, k planes and
their last rows included; and a slice that starts from a B_perp with values on
the row kx = nx.  FP64: 1e-10 of each field's peak (rounding alone); FP32: 1e-4
(the slices' FP32 noise is 1e-6 to 1e-5 of the peak)."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu

REAL = ("F_PSI", "F_PSIT", "F_FXY", "F_BXYZ")
KSPACE = ("F_CU", "F_DCU", "F_AMU", "F_EPW", "F_EPWB", "F_QE")


def _run(indx, indy, precision, separate, tol):
    ctx = qps.Ctx(indx, indy, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=precision)
    if separate:   # any value but the default takes the separate kernels
        ctx.tune(qps.TUNE_FFT, 0 if precision == qps.FP64 else 1)
    sp = qps.Species(ctx, ppc=(2, 1))
    bm = qps.Beam(ctx, center=(0.4, -0.3, 0.4), sigma=(1.2, 1.0, 0.2), np_=(16, 16, 32), peak=2.0)
    sim = qps.Sim(ctx, [sp], [bm])
    ctx.tune(qps.TUNE_SEED, 1)
    sim.begin_step()
    passes = []
    for j in range(1, 6):
        if j == 4:
            rng = np.random.default_rng(3)
            e = sim.field(qps.F_EPW).download(1)
            e[:, -1, :] = 1e-3 * rng.standard_normal(e[:, -1, :].shape)
            sim.field(qps.F_EPW).upload(e, space=1)
        passes.append(sim.slice(j, iter_max=3, tol=tol)[0])
    out = {k: sim.field(getattr(qps, k)).download(0) for k in REAL}
    out.update({k + " k": sim.field(getattr(qps, k)).download(1) for k in KSPACE})
    out["psit k"] = sim.field(qps.F_PSIT).download(1)
    out["bxyz k"] = sim.field(qps.F_BXYZ).download(1)
    ctx.close()
    return out, passes


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("indx,indy,tol", [(4, 4, 0.0), (4, 6, 1e-3), (6, 5, 0.0), (5, 7, 1e-3),
                                           (8, 7, 0.0), (7, 8, 0.0), (9, 10, 1e-3), (10, 9, 0.0)])
def test_fused_field_solve_equals_separate_kernels(indx, indy, tol, precision):
    print(f"[gpu-test] spectral {indx} {indy} {tol} {precision}", flush=True)
    p = getattr(qps, precision)
    got, n = _run(indx, indy, p, False, tol)
    want, m = _run(indx, indy, p, True, tol)
    assert n == m
    bar = 1e-10 if precision == "FP64" else 1e-4
    for k in want:
        peak = np.abs(want[k]).max()
        assert peak > 0.0, k
        assert np.abs(got[k] - want[k]).max() <= bar * peak, k
