"""What runs with the rebuild test on the device report and remember.  Kernel
times count the steps and link breaks that were carried out, not launches that
a stale list turned into nothing.  A run of no steps leaves nothing behind."""
import numpy as np
import pytest

from hidem_amd import _abi as A
from hidem_amd import params

pytestmark = pytest.mark.gpu


def weak_block():
    """A block whose neighbour list lasts a few dozen steps, with links breaking."""
    s, p, l = params.build_inputs(params.load_config("iceblock_16k"), [12, 10, 9])
    l.maxLoad[:] *= 0.25
    s.run.interactDist = s.run.force.attractDistance + 0.004
    return s, p, l


@pytest.mark.parametrize("policy", [A.HDM_REBUILD_EXACT, A.HDM_REBUILD_LEARNED])
def test_kernel_times_count_what_ran(policy):
    s, p, l = weak_block()
    rp = A.HdmRunParams.from_buffer_copy(s.run)
    rp.policy = policy
    runs = [1, 150, 100, 149]
    with A.Context(A.HDM_PREC_FP64) as c:
        c.upload(p, l)
        c.links_build()
        c.sched_configure(min_batch=64, max_batch=64)
        c.set_timing(True)
        rebuilds = [int(np.sum(c.run(rp, k, log_rebuilds=True)[1])) for k in runs]
        times = c.kernel_times()
        stats = c.sched_stats()
    print("  rebuilds", rebuilds, {k: v[1] for k, v in times.items()}, stats, flush=True)
    assert sum(rebuilds) >= 3   # the first list, and trips inside batches
    # breakTime lies before the first step's time: one break per run, behind its last step
    broke_after = sum((sum(runs[:i + 1]) - 1) * rp.dt > rp.breakTime for i in range(len(runs)))
    assert times["break"][1] == broke_after
    if policy == A.HDM_REBUILD_EXACT:
        assert times["step"][1] == sum(runs)
    else:
        assert stats["steps_executed"] == sum(runs) < stats["steps_launched"] == times["step"][1]


@pytest.mark.parametrize("policy", [A.HDM_REBUILD_EXACT, A.HDM_REBUILD_LEARNED])
def test_run_of_no_steps(policy):
    """Between a grid build and the list build of the caller: the list is then
    fresh, so the next run builds none."""
    s, p, l = weak_block()
    rp = A.HdmRunParams.from_buffer_copy(s.run)
    rp.policy = policy
    with A.Context(A.HDM_PREC_FP64) as c:
        c.upload(p, l)
        c.links_build()
        assert np.asarray(c.run(rp, 2, log_rebuilds=True)[1]).tolist() == [1, 0]
        c.grid_build(rp.searchDistance)
        st = c.run(rp, 0)
        assert (st.steps, st.rebuilds, st.timestep) == (0, 0, 2)
        c.neighbours_build(rp.interactDist)
        assert np.asarray(c.run(rp, 3, log_rebuilds=True)[1]).tolist() == [0, 0, 0]
