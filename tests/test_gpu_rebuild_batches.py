"""Runs whose rebuild decisions are taken in batches (exact test) or from
maxima kept for every tenth step only (heuristic): rebuild steps and results
equal those of the same decisions taken one step at a time, whatever the
threshold and however the run is split."""
import copy

import numpy as np
import pytest

from hidem_amd import _abi as A
from hidem_amd import params

pytestmark = pytest.mark.gpu

FIELDS = ("xCord", "yCord", "zCord", "xTheta", "yTheta", "zTheta", "xDiff", "yDiff", "zDiff", "uDiff", "vDiff", "wDiff",
          "xForce", "yForce", "zForce", "uForce", "vForce", "wForce")


def inputs():
    cfg = params.load_config("iceblock_16k")
    cfg["lattice"]["fccSpacing"] = 0.985 * 2 ** 0.5  # overlapping neighbours, so particles move
    cfg["lattice"]["linkGenScale"] = 1.05 * 0.985
    return params.build_inputs(cfg, [6, 5, 4])


def same(a, b):
    (p, l), (q, m) = a, b
    for f in FIELDS:
        assert np.array_equal(p[f].view(np.uint64), q[f].view(np.uint64)), f
    assert np.array_equal(l.state, m.state)
    for k in range(6):
        assert np.array_equal(l.ct[k].view(np.uint64), m.ct[k].view(np.uint64)), k


def params_at(s, policy, threshold):
    rp = copy.deepcopy(s.run)
    rp.policy = policy
    if threshold is not None:
        rp.interactDist = rp.force.attractDistance + threshold
    return rp


@pytest.mark.parametrize("prec", [A.HDM_PREC_FP64, A.HDM_PREC_MIXED])
@pytest.mark.parametrize("pieces", [[(1, None)], [(16, None), (17, 1e-4)], [(40, 2e-3), (3, -1.0), (2, 2e-3)],
                                    [(20, 1e-5), (1, 0.0), (30, 3e-4), (0, 1e-4), (5, 1e-3)]])
def test_exact(prec, pieces):
    s, p, l = inputs()
    with A.Context(prec) as c, A.Context(prec) as d:
        for x in (c, d):
            x.upload(p, l)
            x.links_build()
        ts, built = 0, False
        for steps, threshold in pieces:
            rp = params_at(s, A.HDM_REBUILD_EXACT, threshold)
            log = np.asarray(c.run(rp, steps, log_rebuilds=True)[1])
            thr = rp.interactDist - rp.force.attractDistance
            want = []
            for _ in range(steps):
                regen = not built or 2.0 * d.skin_exact() >= thr
                if regen:
                    d.grid_build(rp.searchDistance)
                    d.neighbours_build(rp.interactDist)
                    d.skin_snapshot()
                    built = True
                want.append(regen)
                d.force(rp.force)
                d.integrate(rp.integ)
                if ts * rp.dt > rp.breakTime:
                    d.brk(rp.brk)
                ts += 1
            print("  steps", steps, "threshold", threshold, "rebuilds", sum(want), flush=True)
            assert log.astype(bool).tolist() == want
        same((c.download_particles(), c.download_links()), (d.download_particles(), d.download_links()))


@pytest.mark.parametrize("pieces", [[39], [9, 1, 1, 28], [10, 20, 9], [3, 8, 28]])
def test_heuristic_split(pieces):
    s, p, l = inputs()
    rp = params_at(s, A.HDM_REBUILD_HEURISTIC, 0.01)
    with A.Context(A.HDM_PREC_FP64) as c, A.Context(A.HDM_PREC_FP64) as d:
        for x in (c, d):
            x.upload(p, l)
            x.links_build()
        got = [r for k in pieces for r in np.asarray(c.run(rp, k, log_rebuilds=True)[1]).tolist()]
        want, acc = [], 0.0
        for ts in range(39):
            regen = ts == 0
            if ts % 10 == 0:
                acc += d.skin_heuristic(10)
                regen = regen or acc >= rp.interactDist / 2.0
            if regen:
                d.grid_build(rp.searchDistance)
                d.neighbours_build(rp.interactDist)
                acc = 0.0
            want.append(int(regen))
            d.force(rp.force)
            d.integrate(rp.integ)
            if ts * rp.dt > rp.breakTime:
                d.brk(rp.brk)
        print("  pieces", pieces, "rebuilds", sum(want), flush=True)
        assert got == want
        same((c.download_particles(), c.download_links()), (d.download_particles(), d.download_links()))
