"""The batched scan's captured slices are cut into a start with the first
passes, one part per further pass and an end: whatever number of passes a
slice takes and wherever the cut lies, the passes and fields are bitwise those
of eager slices run one after the other."""
import numpy as np
import pytest

qps = pytest.importorskip("qpslice")
qpscan = pytest.importorskip("qpscan")

pytestmark = pytest.mark.gpu


# fewer passes than the start holds, exactly as many, one more, and many; a
# tolerance that is met early, midway, and never
@pytest.mark.parametrize("iter_max", [1, 4, 5, 20])
@pytest.mark.parametrize("tol", [1e-1, 1e-5, 1e-14, 0.0])
def test_scan_parts_equal_eager(iter_max, tol):
    print(f"[gpu-test] scan parts iter_max={iter_max} tol={tol}", flush=True)
    insts = qpscan.draw(3, grids=[6, 7], ppcs=[2, 3], indz=5, beam_np=(16, 16, 64), seed=7,
                        iter_=iter_max, tol=tol, seed_mode=1)
    try:
        n = 8
        qpscan.run_sequential(insts, n)
        passes = [list(x.passes) for x in insts]
        want = [x.fields() + [x.sp.download()] for x in insts]
        qpscan.run_graph(insts, n, chunk=3)
        for i, x in enumerate(insts):
            assert list(x.passes) == passes[i], i
            for a, b in zip(want[i], x.fields() + [x.sp.download()]):
                assert np.array_equal(a, b), i
    finally:
        for x in insts:
            x.close()
