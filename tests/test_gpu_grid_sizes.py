"""The grid build and the reductions over particles at the sizes where their
split has edges: one workgroup and several, workgroups that take several items
per lane, cells whose workgroup sorts its run in LDS and in memory, grids of
less and more cells than a workgroup takes.  Exact against the oracle and
NumPy."""
import numpy as np
import pytest

from hidem_amd import _abi as A

pytestmark = pytest.mark.gpu


def cloud(n, size):
    r = np.random.default_rng(n)
    p = A.Particles.zeros(n)
    for f in ("xCord", "yCord", "zCord"):
        p.arrays[f][:] = r.random(n) * size
    p.arrays["radius"][:] = 0.05
    for f in ("xDiff", "yDiff", "zDiff"):
        p.arrays[f][:] = r.normal(scale=1e-3, size=n)
    return p


@pytest.mark.parametrize("n,size,spacing", [(2, 1.0, 0.3), (63, 1.0, 0.3), (257, 4.0, 0.62), (256, 4.0, 0.7),
                                            (1025, 10.0, 1.0), (2048, 3.0, 1.6), (2049, 3.0, 1.6), (6000, 6.0, 2.1),
                                            (20000, 12.0, 0.9)])
def test_grid(n, size, spacing, orc):
    print("  n", n, "spacing", spacing, flush=True)
    p = cloud(n, size)
    with A.Context(A.HDM_PREC_FP64) as c:
        c.upload(p, None)
        for _ in range(2):   # a build after another starts from its own values
            c.grid_build(spacing)
            info = c.grid_info()
            col, order = c.grid_download()
            c.neighbours_build(spacing / 3)
            counts, starts, lst = c.neighbours_download()
    _, g = orc.grid_build(p, spacing)
    assert (info.X, info.Y, info.Z) == g["dims"]
    assert (info.xMin, info.yMin, info.zMin) == g["mins"]
    assert info.occupiedCells == g["nOcc"]
    assert info.maxPerCell == np.bincount(g["colours"]).max()
    assert np.array_equal(col, g["colours"])
    assert np.array_equal(order, g["order"])
    oc, os_, ol = orc.neigh_build(p, spacing, spacing / 3)
    assert np.array_equal(counts, oc) and np.array_equal(starts, os_) and np.array_equal(lst, ol)


@pytest.mark.parametrize("n", [2, 64, 65, 257, 524288, 600001])
def test_reductions(n):
    print("  n", n, flush=True)
    p = cloud(n, 100.0)
    with A.Context(A.HDM_PREC_FP64) as c:
        c.upload(p, None)
        h = c.skin_heuristic(10)
        c.skin_snapshot()
        zero = c.skin_exact()
        c.grid_build(7.0)
        info = c.grid_info()
    m = [max(0.0, p.arrays[f].max()) for f in ("xDiff", "yDiff", "zDiff")]
    assert h == 10 * np.sqrt(m[0] * m[0] + m[1] * m[1] + m[2] * m[2])
    assert zero == 0.0
    for f, lo, hi in (("xCord", info.xMin, info.xMax), ("yCord", info.yMin, info.yMax), ("zCord", info.zMin, info.zMax)):
        assert (lo, hi) == (p.arrays[f].min(), p.arrays[f].max())
