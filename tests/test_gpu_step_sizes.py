"""The fused step at the sizes where its work split has edges: wave tiles of
64 particles, workgroups of 256, the largest state of the tile form (32,768
particles on 256 compute units) and one particle more, with contacts active
and links breaking in the steps (so particles sum their force a second time),
and particles of more than 64 links.  FP64 form against the CPU oracle bit for
bit; FP32 form against its own per-call kernels bit for bit."""
import numpy as np
import pytest

from hidem_amd import _abi as A
from hidem_amd import params

pytestmark = pytest.mark.gpu

FIELDS = ("xCord", "yCord", "zCord", "xTheta", "yTheta", "zTheta", "xDiff", "yDiff", "zDiff", "uDiff", "vDiff", "wDiff",
          "xForce", "yForce", "zForce", "uForce", "vForce", "wForce")


def bits_equal(a, b):
    return np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))


def first_particles(p, l, n):
    """The first n particles of (p, l) and the links among them."""
    q = A.Particles.zeros(n)
    for f in A.PARTICLE_FIELDS:
        q.arrays[f][:] = p[f][:n]
    q.type[:] = p.type[:n]
    keep = (l.a < n) & (l.b < n)
    m = int(keep.sum())
    return q, A.Links(m, l.a[keep].copy(), l.b[keep].copy(), l.state[keep].copy(), l.initialLen[keep].copy(),
                      l.maxLoad[keep].copy(), [np.zeros(2 * m) for _ in range(6)])


def check_both_forms(s, p, l, steps, orc, min_broken):
    sim = orc.OracleSim(p, l, s)
    sim.run(steps)
    with A.Context(A.HDM_PREC_FP64) as c:
        c.upload(p, l)
        c.links_build()
        c.run(s.run, steps)
        gp, gl = c.download_particles(), c.download_links()
    broken = int((sim.l.state == 0).sum())
    print("  n", p.n, "links", l.n, "broken", broken, flush=True)
    assert broken >= min_broken
    assert np.array_equal(gl.state, sim.l.state)
    for f in FIELDS:
        assert bits_equal(gp[f], sim.p[f]), f
    for k in range(6):
        assert bits_equal(gl.ct[k], sim.l.ct[k]), k
    # FP32 form: one run, and the same steps call by call on the run's list
    with A.Context(A.HDM_PREC_MIXED) as c, A.Context(A.HDM_PREC_MIXED) as d:
        for x in (c, d):
            x.upload(p, l)
            x.links_build()
        c.run(s.run, steps)
        d.grid_build(s.run.searchDistance)
        d.neighbours_build(s.run.interactDist)
        for ts in range(steps):
            d.force(s.run.force)
            d.integrate(s.run.integ)
            if ts * s.run.dt > s.run.breakTime:
                d.brk(s.run.brk)
        cp, cl, dp, dl = c.download_particles(), c.download_links(), d.download_particles(), d.download_links()
    for f in FIELDS:
        assert bits_equal(cp[f], dp[f]), f
    assert np.array_equal(cl.state, dl.state)
    for k in range(6):
        assert bits_equal(cl.ct[k], dl.ct[k]), k


@pytest.mark.parametrize("n", [2, 63, 64, 65, 257, 32768, 32769])
def test_sizes(n, orc):
    cfg = params.load_config("iceblock_16k")
    cfg["lattice"]["fccSpacing"] = 0.985 * 2 ** 0.5  # overlapping neighbours
    cfg["lattice"]["linkGenScale"] = 1.05 * 0.985
    s, p, l = params.build_inputs(cfg, [25, 20, 17] if n > 10000 else [6, 5, 4])
    p, l = first_particles(p, l, n)
    check_both_forms(s, p, l, 6, orc, min_broken=1 if n > 65 else 0)


def test_more_than_64_links_breaking(orc):
    cfg = params.load_config("iceblock_16k")
    cfg["lattice"]["linkGenScale"] = 2.7  # links over several neighbour shells
    s, p, l = params.build_inputs(cfg, [6, 5, 5])
    assert np.bincount(np.concatenate([l.a, l.b])).max() > 64
    l.maxLoad[:] *= 1e-5
    check_both_forms(s, p, l, 6, orc, min_broken=100)
