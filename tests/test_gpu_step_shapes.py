"""The launch shape of the fused step: what a caller chooses is what runs and
what hdm_exec_info names, for states of the tile form too, and without a choice
the tile form is named as such and can be gone back to.  Every shape computes
the same bits: the lane form at a size just above the tile form's limit that
fills neither the last workgroup nor the last wave of any shape, and the shape
of the largest states, with contacts active and links breaking in the steps.
FP64 form against the CPU oracle, FP32 form against its per-call kernels."""
import numpy as np
import pytest

from hidem_amd import _abi as A
from hidem_amd import params
from test_gpu_step_sizes import FIELDS, bits_equal, first_particles

pytestmark = pytest.mark.gpu

SHAPES = ["wg256-xcd", "wg128-xcd", "wg512-xcd", "wg256-linear", "wg128-xcd-occ", "wg256-xcd-occ", "wg64-xcd"]
STEPS = 5


def inputs(cells, n):
    cfg = params.load_config("iceblock_16k")
    cfg["lattice"]["fccSpacing"] = 0.985 * 2 ** 0.5  # overlapping neighbours
    cfg["lattice"]["linkGenScale"] = 1.05 * 0.985
    s, p, l = params.build_inputs(cfg, cells)
    return (s,) + first_particles(p, l, n)


def same(got, want):
    (p, l), (q, m) = got, want
    for f in FIELDS:
        assert bits_equal(p[f], q[f]), f
    assert np.array_equal(l.state, m.state)
    for k in range(6):
        assert bits_equal(l.ct[k], m.ct[k]), k


def run(prec, s, p, l, steps=STEPS, variant=-1):
    with A.Context(prec) as c:
        c.upload(p, l)
        c.links_build()
        c.set_exec(variant=variant)
        c.run(s.run, steps)
        return (c.download_particles(), c.download_links()), c.exec_info()


def call_by_call(s, p, l, steps=STEPS):
    """The same steps on the FP32 form's per-call kernels."""
    with A.Context(A.HDM_PREC_MIXED) as d:
        d.upload(p, l)
        d.links_build()
        d.grid_build(s.run.searchDistance)
        d.neighbours_build(s.run.interactDist)
        for ts in range(steps):
            d.force(s.run.force)
            d.integrate(s.run.integ)
            if ts * s.run.dt > s.run.breakTime:
                d.brk(s.run.brk)
        return d.download_particles(), d.download_links()


def oracle_run(orc, s, p, l, min_broken):
    sim = orc.OracleSim(p, l, s)
    sim.run(STEPS)
    broken = int((sim.l.state == 0).sum())
    print("  n", p.n, "links", l.n, "broken", broken, flush=True)
    assert broken >= min_broken
    return sim.p, sim.l


@pytest.fixture(scope="module")
def above_tiles(orc):
    s, p, l = inputs([25, 20, 17], 33001)
    return s, p, l, {A.HDM_PREC_FP64: oracle_run(orc, s, p, l, 10), A.HDM_PREC_MIXED: call_by_call(s, p, l)}


def test_choice_is_what_runs():
    s, p, l = inputs([6, 5, 4], 470)
    for prec in (A.HDM_PREC_FP64, A.HDM_PREC_MIXED):
        want, info = run(prec, s, p, l)
        assert (info["variant"], info["name"]) == (-1, "tile64")
        for v, name in enumerate(SHAPES):
            got, info = run(prec, s, p, l, variant=v)
            assert (info["variant"], info["name"]) == (v, name)
            same(got, want)


def test_tile_form_is_kept_and_gone_back_to():
    s, p, l = inputs([6, 5, 4], 470)
    rp = A.HdmRunParams.from_buffer_copy(s.run)
    rp.policy = A.HDM_REBUILD_LEARNED
    with A.Context(A.HDM_PREC_FP64) as c:
        c.upload(p, l)
        c.links_build()
        c.set_exec(graphs=True, variant=c.exec_info()["variant"])   # handed back: no choice
        c.run(rp, 30)
        assert c.exec_info()["name"] == "tile64"
        c.set_exec(graphs=True, variant=2)
        c.run(rp, 30)
        assert c.exec_info()["name"] == "wg512-xcd"
        c.set_exec(autotune=True, graphs=True)                     # nothing to tune
        c.run(rp, 30)
        info = c.exec_info()
        assert info["tuned"] and info["name"] == "tile64" and not any(info["tune_ms"])
        got = c.download_particles(), c.download_links()
    rp.policy = A.HDM_REBUILD_EXACT
    with A.Context(A.HDM_PREC_FP64) as c:
        c.upload(p, l)
        c.links_build()
        c.run(rp, 90)
        same(got, (c.download_particles(), c.download_links()))


@pytest.mark.parametrize("prec", [A.HDM_PREC_FP64, A.HDM_PREC_MIXED])
@pytest.mark.parametrize("variant", range(len(SHAPES)))
def test_lane_form_shapes(prec, variant, above_tiles):
    s, p, l, want = above_tiles
    print("  shape", SHAPES[variant], "prec", prec, flush=True)
    got, info = run(prec, s, p, l, variant=variant)
    assert info["name"] == SHAPES[variant]
    same(got, want[prec])


def test_shape_of_large_states(orc):
    s, p, l = inputs([45, 40, 37], 263001)
    got, info = run(A.HDM_PREC_FP64, s, p, l)
    assert info["name"] == "wg256-linear"
    same(got, oracle_run(orc, s, p, l, 100))
    same(run(A.HDM_PREC_MIXED, s, p, l)[0], call_by_call(s, p, l))


@pytest.mark.parametrize("prec", [A.HDM_PREC_FP64, A.HDM_PREC_MIXED])
def test_autotuned_lane_form(prec):
    """Every shape in turn, then graph replays of the chosen one, through
    rebuilds, against the same steps under the exact test (a block whose list
    lasts a few dozen steps, with links breaking)."""
    s, p, l = params.build_inputs(params.load_config("iceblock_16k"), [25, 20, 17])
    p, l = first_particles(p, l, 33001)
    l.maxLoad[:] *= 0.25
    out = []
    for policy in (A.HDM_REBUILD_EXACT, A.HDM_REBUILD_LEARNED):
        rp = A.HdmRunParams.from_buffer_copy(s.run)
        rp.policy = policy
        rp.interactDist = rp.force.attractDistance + 0.004
        with A.Context(prec) as c:
            c.upload(p, l)
            c.links_build()
            c.sched_configure(min_batch=16, max_batch=48)
            c.set_exec(autotune=True, graphs=True)
            log = [c.run(rp, k, log_rebuilds=True)[1] for k in (150, 151)]
            out.append((np.concatenate(log), (c.download_particles(), c.download_links()), c.exec_info()))
    (log_e, want, _), (log_l, got, info) = out
    print("  rebuilds", int(log_e.sum()), info, flush=True)
    assert log_e.sum() >= 2
    assert np.array_equal(log_e, log_l)
    same(got, want)
    assert info["tuned"] and all(t > 0 for t in info["tune_ms"]) and info["graph_replays"] > 0
    assert info["name"] in SHAPES
