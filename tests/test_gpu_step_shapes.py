"""The launch shape of the fused step: what a caller chooses is what runs and
what hdm_exec_info names, for states of the tile form too, and without a choice
the tile form is named as such and can be gone back to."""
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
