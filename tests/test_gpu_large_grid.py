"""The plasma push on a grid of more than 8192 tiles, whose cell offsets are summed
in two levels, against the push in place and the scan and scatter behind it: every
particle at the same place, every cell with the same count, bit for bit, after
pushes that move particles between cells."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu


def _pushed(precision, in_place):
    ctx = qps.Ctx(11, 11, 4, box=(-10.0, 10.0, -10.0, 10.0, 0.0, 1.0), precision=precision)
    assert (ctx.nx // 16) * (ctx.ny // 16) > 8192
    if in_place:
        ctx.tune(qps.TUNE_PUSH, 1)
    sp = qps.Species(ctx, ppc=(1, 1))
    f = {n: qps.Field2d(ctx, d) for n, d in (("e", 2), ("b", 3), ("psit", 1))}
    rng = np.random.default_rng(11)
    for n, d in (("e", 2), ("b", 3), ("psit", 1)):
        f[n].upload(0.2 * rng.standard_normal((d, ctx.ny + 1, ctx.nx + 1)), space=0)
    out = []
    for _ in range(2):
        sp.push(f["e"], f["b"], f["psit"], ctx.dex)
        out += [sp.download(), sp.cell_counts()]
    ctx.close()
    return out


@pytest.mark.parametrize("precision", ["FP32", "FP64"])
def test_push_with_two_level_offsets(precision):
    print(f"[gpu-test] push on 2048^2 {precision}", flush=True)
    p = getattr(qps, precision)
    got, want = _pushed(p, False), _pushed(p, True)
    start = np.bincount(want[1].ravel().astype(np.int64), minlength=2)
    assert start[1] < want[1].size   # particles have changed cells
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
