"""The current deposit on grids of few tiles (several blocks to a tile, each a
band of its rows) against its form of one block per tile, which the other tests
hold to the oracle: four, two and one band, sparse and dense cells, after a push
that moved particles.  A node's sum has at most N = 4 x 2 ppc terms (a push
gathers no more than twice the cells' particles here); in either order it is
rounded to N eps times its terms' sum, itself at most N times the plane's peak
where the terms cancel."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu


def _run(indx, indy, ppc, precision, variant):
    ctx = qps.Ctx(indx, indy, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=precision)
    if variant is not None:
        ctx.tune(qps.TUNE_AMJDP, variant)
    sp = qps.Species(ctx, ppc=ppc)
    f = {n: qps.Field2d(ctx, d) for n, d in (("psi", 1), ("e", 2), ("b", 3), ("psit", 1),
                                            ("cu", 3), ("amu", 3), ("dcu", 2))}
    rng = np.random.default_rng(indx * 10 + indy)
    for n, d in (("psi", 1), ("e", 2), ("b", 3), ("psit", 1)):
        f[n].upload(0.05 * rng.standard_normal((d, ctx.ny + 1, ctx.nx + 1)), space=0)
    out = []
    for _ in range(2):
        for n in ("cu", "amu", "dcu"):
            f[n].as_(0.25)
        sp.extpsi(f["psi"], ctx.dex)
        sp.amjdp(f["e"], f["b"], f["psit"], f["cu"], f["amu"], f["dcu"], ctx.dex)
        out += [f[n].download(0) for n in ("cu", "amu", "dcu")]
        sp.push(f["e"], f["b"], f["psit"], ctx.dex)
    out.append(sp.download())
    ctx.close()
    return out


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("indx,indy,ppc", [(4, 4, (1, 1)), (5, 6, (2, 2)), (7, 7, (5, 5)),
                                           (8, 7, (2, 2)), (7, 8, (8, 4)), (8, 8, (2, 1))])
def test_banded_current_deposit(indx, indy, ppc, precision):
    print(f"[gpu-test] bands {indx} {indy} {ppc} {precision}", flush=True)
    p = getattr(qps, precision)
    got, want = (_run(indx, indy, ppc, p, v) for v in (None, 11))
    n = 8 * ppc[0] * ppc[1]
    eps = 2.0 ** -52 if precision == "FP64" else 2.0 ** -23
    for a, b in zip(got[:-1], want[:-1]):
        peak = np.abs(b).max()
        assert peak > 0.0
        assert np.abs(a - b).max() <= n * n * eps * peak
    assert np.array_equal(got[-1], want[-1])   # the deposit moves no particle


def _pushed(indx, indy, ppc, precision, in_place):
    ctx = qps.Ctx(indx, indy, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=precision)
    if in_place:
        ctx.tune(qps.TUNE_PUSH, 1)
    sp = qps.Species(ctx, ppc=ppc)
    f = {n: qps.Field2d(ctx, d) for n, d in (("e", 2), ("b", 3), ("psit", 1))}
    rng = np.random.default_rng(indx + 7 * indy)
    for n, d in (("e", 2), ("b", 3), ("psit", 1)):
        f[n].upload(0.2 * rng.standard_normal((d, ctx.ny + 1, ctx.nx + 1)), space=0)
    out = []
    for _ in range(3):
        sp.push(f["e"], f["b"], f["psit"], ctx.dex)
        out += [sp.download(), sp.cell_counts()]
    ctx.close()
    return out


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("indx,indy,ppc", [(4, 4, (5, 5)), (6, 5, (2, 2)), (7, 7, (3, 2)),
                                           (8, 8, (2, 1)), (7, 7, (1, 1)), (9, 8, (2, 2))])
def test_push_blocks_keep_the_order(indx, indy, ppc, precision):
    """Blocks of 256 and of 1024 threads put every particle where the push in
    place and the scatter behind it put it, bit for bit."""
    print(f"[gpu-test] push blocks {indx} {indy} {ppc} {precision}", flush=True)
    p = getattr(qps, precision)
    for a, b in zip(_pushed(indx, indy, ppc, p, False), _pushed(indx, indy, ppc, p, True)):
        assert np.array_equal(a, b)
