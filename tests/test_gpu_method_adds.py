"""qdp and amjdp add the deposit to the caller's fields in the deposit's own
stores: bit for bit the deposit into zeroed fields and the additions behind it
(an addition of two numbers is rounded once, whichever kernel does it), on the
nodes of every kind; and fields that are the deposit's inputs too keep the
additions behind the deposit."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("indx,indy", [(4, 4), (7, 6), (8, 8), (9, 5)])
def test_additions_in_the_deposit(indx, indy, precision):
    print(f"[gpu-test] method adds {indx} {indy} {precision}", flush=True)
    p = getattr(qps, precision)
    ctx = qps.Ctx(indx, indy, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=p)
    dt = np.float64 if precision == "FP64" else np.float32
    rng = np.random.default_rng(indx + indy)
    sp = qps.Species(ctx, ppc=(2, 2))
    f = {n: qps.Field2d(ctx, d) for n, d in (("q", 1), ("e", 2), ("b", 3), ("psit", 1),
                                             ("cu", 3), ("amu", 3), ("dcu", 2))}
    base = {n: rng.standard_normal((f[n].dim, ctx.ny + 1, ctx.nx + 1)).astype(dt)
            for n in ("q", "cu", "amu", "dcu")}
    for n in ("e", "b", "psit"):
        f[n].upload(0.05 * rng.standard_normal((f[n].dim, ctx.ny + 1, ctx.nx + 1)), space=0)
    part = sp.download()

    def deposit(names):
        sp.upload(part)
        if names == ("q",):
            sp.qdp(f["q"])
        else:
            sp.amjdp(f["e"], f["b"], f["psit"], f["cu"], f["amu"], f["dcu"], ctx.dex)
        return {n: f[n].download(0).astype(dt) for n in names}

    for names in (("q",), ("cu", "amu", "dcu")):
        for n in names:
            f[n].as_(0.0)
        alone = deposit(names)
        for n in names:
            f[n].upload(base[n], space=0)
        got = deposit(names)
        for n in names:
            want = alone[n] + base[n]
            if n == "q":   # the background comes last: qn + (deposit + q)
                tol = 4 * np.finfo(dt).eps * (np.abs(alone[n]) + np.abs(base[n]) + 2)
                assert (np.abs(got[n] - want) <= tol).all()
            else:
                assert np.array_equal(got[n], want.astype(dt)), n
    # b as an input and as the current's target
    b0 = f["b"].download(0).astype(dt)
    f["cu"].as_(0.0), f["amu"].as_(0.0), f["dcu"].as_(0.0)
    alone = deposit(("cu", "amu", "dcu"))
    f["amu"].as_(0.0), f["dcu"].as_(0.0)
    sp.upload(part)
    sp.amjdp(f["e"], f["b"], f["psit"], f["b"], f["amu"], f["dcu"], ctx.dex)
    assert np.array_equal(f["b"].download(0).astype(dt), (alone["cu"] + b0).astype(dt))
    assert np.array_equal(f["amu"].download(0).astype(dt), alone["amu"])
    ctx.close()

