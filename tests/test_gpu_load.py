"""The plasma loader's kernels (dist2d_000/010/012, fdist2d_class.f03:212-950)
on the smallest and non-square grids, with odd particle counts per cell, and
again after a push has moved the particles: every particle equals the
oracle's, positions bit for bit (FP32: rounded relative to the tile), charges
to 1e-14 (FP32: one rounding, 6e-8), in cell order."""
import numpy as np
import pytest

from oracle import qpo

qps = pytest.importorskip("qpslice")

pytestmark = pytest.mark.gpu

PROFILES = {0: {}, 10: dict(center=(0.7, -1.1), inner_radius=(2.1, 1.3), outer_radius=(6.3, 4.9)),
            12: dict(center=(0.3, 0.2), radial=((0.5, 2.0, 3.5, 8.0), (0.2, 1.0, 0.4, 0.1)))}


@pytest.mark.parametrize("precision", ["FP64", "FP32"])
@pytest.mark.parametrize("indx,indy,ppc,profile", [(4, 4, (1, 1), 0), (4, 6, (3, 2), 0),
                                                   (6, 4, (1, 5), 10), (5, 5, (5, 3), 12)])
def test_loaded_particles_equal_the_oracle(precision, indx, indy, ppc, profile):
    print(f"[gpu-test] load {indx} {indy} {ppc} {profile} {precision}", flush=True)
    grid = qpo.Grid(indx, indy, 4)
    want = qpo.Species(grid, qpo.SpeciesSpec(ppc=ppc, profile=profile, density=0.7,
                                             **PROFILES[profile]), grid.dz).part
    if precision == "FP32":
        o = np.floor(want[:, :2] / 16.0) * 16.0
        want = want.copy()
        want[:, :2] = (want[:, :2] - o).astype(np.float32) + o
    want = want[np.lexsort(want[:, :2].T[::-1])]
    ctx = qps.Ctx(indx, indy, 4, precision=getattr(qps, precision))
    try:
        sp = qps.Species(ctx, ppc=ppc, density=0.7)
        if profile:
            sp.set_profile(profile, **PROFILES[profile])
        e, b, z = qps.Field2d(ctx, 2), qps.Field2d(ctx, 3), qps.Field2d(ctx, 1)
        e.as_(0.01)
        for load in range(2):
            got = sp.download()
            c = qpo.cell_of(grid.nx, grid.ny, np.ascontiguousarray(got))
            cx, cy = c % grid.nx, c // grid.nx
            key = ((cy // 16) * (grid.nx // 16) + cx // 16) * 256 + (cy % 16) * 16 + cx % 16
            assert np.all(np.diff(key) >= 0)
            assert np.array_equal(sp.cell_counts(), np.bincount(c, minlength=grid.nx * grid.ny))
            got = got[np.lexsort(got[:, :2].T[::-1])]
            assert got.shape == want.shape
            assert np.array_equal(got[:, :7], want[:, :7])
            bar = 1e-14 if precision == "FP64" else 6e-8
            assert np.abs(got[:, 7] / want[:, 7] - 1.0).max() <= bar
            sp.push(e, b, z, ctx.dex)   # an odd number of pushes leaves the other buffers current
            assert not np.array_equal(sp.download()[:, :2], want[:, :2])
            sp.renew(0.0)
    finally:
        ctx.close()
