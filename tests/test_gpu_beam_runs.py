"""The beam's charge deposit with eight particles a thread (long runs of one cell,
as the push has sorted them) and with one (short runs, or an order that is not
known): integer sums, so the same charge bit for bit, as the same particles in
random order give, whatever the cells' runs and the particle count."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ind,indz,sigma,np_", [
    (5, 4, 0.3, (64, 64, 64)),      # runs of hundreds: eight a thread
    (5, 4, 0.02, (16, 16, 17)),     # a small beam in few cells: eight a thread
    (7, 6, 1.5, (64, 64, 65)),      # about one particle a cell: one a thread
    (5, 4, 2.0, (3, 3, 7))])        # less than a wavefront
def test_charge_by_either_kernel(ind, indz, sigma, np_):
    print(f"[gpu-test] beam runs {ind} {indz} {sigma} {np_}", flush=True)
    ctx = qps.Ctx(ind, ind, indz, precision=qps.FP64)
    bm = qps.Beam(ctx, center=(0.0, 0.0, 5.0), sigma=(sigma, sigma, sigma), np_=np_, peak=2.0)
    e, b = qps.Field3d(ctx, 3), qps.Field3d(ctx, 3)
    bm.push(e, b, ctx.dex, ctx.dxi)
    part = bm.download()
    bm.qdp()
    want = bm.charge()
    assert np.abs(want).max() > 0.0
    bm.upload(part[np.random.default_rng(2).permutation(len(part))])
    bm.qdp()
    assert np.array_equal(bm.charge(), want)
    bm.push(e, b, ctx.dex, ctx.dxi)   # sorted again: no field, so only z has moved
    bm.qdp()
    assert bm.charge().sum() == pytest.approx(want.sum(), rel=1e-9)
    ctx.close()
