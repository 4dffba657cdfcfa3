"""The banded current deposit against its form of one block per tile, node by node.

All charges have one sign here and all particles move towards +x and +y, so the
terms of cu(1), cu(2) and of amu have one sign each and a node's sum is the sum of
its terms' absolute values.  A node has at most N terms, the particles of its four
cells; in any order their sum is rounded to (N - 1) eps of itself, which makes
2 N eps for the two forms, and a term of some thirty operations without
cancellation adds 32 eps."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu


def _deposit(indx, indy, ppc, precision, variant):
    ctx = qps.Ctx(indx, indy, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=precision)
    if variant is not None:
        ctx.tune(qps.TUNE_AMJDP, variant)
    sp = qps.Species(ctx, ppc=ppc)
    rng = np.random.default_rng(indx + 10 * indy)
    p = sp.download()
    p[:, 0] += rng.uniform(-0.4, 0.4, len(p)) / ppc[0]
    p[:, 1] += rng.uniform(-0.4, 0.4, len(p)) / ppc[1]
    p[:, 2:4] = rng.uniform(0.5, 1.5, (len(p), 2))
    sp.upload(p)
    f = {n: qps.Field2d(ctx, d) for n, d in (("psi", 1), ("e", 2), ("b", 3), ("psit", 1),
                                            ("cu", 3), ("amu", 3), ("dcu", 2))}
    for n in f:
        f[n].as_(0.0)
    sp.extpsi(f["psi"], ctx.dex)
    sp.amjdp(f["e"], f["b"], f["psit"], f["cu"], f["amu"], f["dcu"], ctx.dex)
    out = f["cu"].download(0)[:2], f["amu"].download(0)
    n = 4 * int(sp.cell_counts().max())
    ctx.close()
    return out, n


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("indx,indy,ppc", [(4, 4, (1, 1)), (6, 6, (5, 5)), (8, 7, (3, 2)),
                                           (7, 8, (8, 4)), (8, 8, (2, 1))])
def test_band_sums(indx, indy, ppc, precision):
    print(f"[gpu-test] band sums {indx} {indy} {ppc} {precision}", flush=True)
    p = getattr(qps, precision)
    (got, n), (want, _) = (_deposit(indx, indy, ppc, p, v) for v in (None, 11))
    eps = 2.0 ** -53 if precision == "FP64" else 2.0 ** -24
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0.0
        for c in range(len(b)):
            assert b[c].min() >= 0.0 or b[c].max() <= 0.0, c   # one sign
        assert np.all(np.abs(a - b) <= (2 * n + 32) * eps * np.abs(b))
