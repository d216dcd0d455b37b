"""The link list build at the sizes where its split has edges: links whose
first endpoints come in runs of every length and in no order at all, a wave
that holds the end of the list, lists up to and above the width that is sorted
in LDS, particles without links.  Lists, slots' strain and flags equal a NumPy
build."""
import numpy as np
import pytest

from hidem_amd import _abi as A

pytestmark = pytest.mark.gpu


def links(n, per, order, seed):
    """per random partners of each particle, each pair once."""
    r = np.random.default_rng(seed)
    a = np.repeat(np.arange(n), per)
    b = r.integers(0, n, a.size)
    lo, hi = np.minimum(a, b), np.maximum(a, b)
    pair = np.unique(np.stack([lo, hi], 1)[lo != hi], axis=0)
    swap = r.random(len(pair)) < 0.5
    a, b = np.where(swap, pair[:, 1], pair[:, 0]), np.where(swap, pair[:, 0], pair[:, 1])
    if order == "sorted":
        k = np.lexsort((b, a))
        a, b = a[k], b[k]
    elif order == "random":
        k = r.permutation(len(a))
        a, b = a[k], b[k]
    m = len(a)
    return A.Links(m, a.astype(np.int32), b.astype(np.int32), (r.random(m) < 0.8).astype(np.uint8),
                   np.full(m, 1.0), np.full(m, 1.0), [r.normal(size=2 * m).astype(np.float32).astype(np.float64) for _ in range(6)])


@pytest.mark.parametrize("prec", [A.HDM_PREC_FP64, A.HDM_PREC_MIXED])
@pytest.mark.parametrize("n,per,order", [(2, 1, "sorted"), (64, 3, "sorted"), (65, 3, "random"), (300, 1, "sorted"),
                                         (300, 20, "sorted"), (1000, 6, "random"), (130, 60, "sorted"),
                                         (129, 29, "random"), (5000, 6, "pairs")])
def test_lists(prec, n, per, order):
    l = links(n, per, order, n)
    p = A.Particles.zeros(n + 3)   # the last three have no links
    r = np.random.default_rng(n)
    for f in ("xCord", "yCord", "zCord"):
        p.arrays[f][:] = r.random(n + 3) * 10
    p.arrays["radius"][:] = 0.1
    with A.Context(prec) as c:
        c.upload(p, l)
        for _ in range(2):   # the second build starts from the tiled strain
            c.links_build()
            counts, starts, ids, other, end = c.linklists_download()
            back = c.download_links()
    want = [[] for _ in range(n + 3)]
    for k, (a, b) in enumerate(zip(l.a.tolist(), l.b.tolist())):
        want[a].append((k, b, 0))
        want[b].append((k, a, 1))
    print("  n", n, "links", l.n, "most", max(map(len, want)), flush=True)
    assert counts.tolist() == [len(w) for w in want]
    flat = [x for w in want for x in w]
    assert ids.tolist() == [x[0] for x in flat]
    assert other.tolist() == [x[1] for x in flat]
    assert end.tolist() == [x[2] for x in flat]
    assert np.array_equal(back.state, l.state)
    for k in range(6):
        assert np.array_equal(back.ct[k], l.ct[k]), k
