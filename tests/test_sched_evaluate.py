"""What the scheduler's evaluation reports of the host's checks is what its runs
make of them (no GPU needed: the context is a stand-in that counts)."""
import types

import numpy as np
import pytest

from hidem_amd import _abi as A
from hidem_amd import sched_train


class Counting:
    """Counts runs and steps per policy; a run reads the guard at least once."""

    made = []

    def __init__(self, prec):
        self.runs = []

    def __enter__(self):
        Counting.made.append(self)
        return self

    def __exit__(self, *a):
        return False

    def run(self, rp, k):
        self.policy = rp.policy
        self.runs.append(k)
        return types.SimpleNamespace(rebuilds=0, seconds=0.0)

    def sched_stats(self):
        return {"host_checks": len(self.runs), "steps_launched": sum(self.runs), "steps_executed": sum(self.runs)}

    def download_particles(self):
        return A.Particles.zeros(1)

    def count_broken(self):
        return 0

    def __getattr__(self, name):
        return lambda *a, **k: None


@pytest.mark.parametrize("ts,steps", [(0, 30), (7, 25), (10, 41)])
def test_host_checks(monkeypatch, ts, steps):
    monkeypatch.setattr(A, "Context", Counting)
    Counting.made = []
    setup = types.SimpleNamespace(run=A.HdmRunParams())
    ev = sched_train.evaluate(setup, (None, None), ts, steps, object(), chunk=10)
    assert [sum(c.runs) for c in Counting.made] == [steps] * len(ev)
    for (name, r), c in zip(ev.items(), Counting.made):
        if c.policy == A.HDM_REBUILD_HEURISTIC:   # decides before every step whose number is a multiple of ten
            assert r["host_checks"] == len([t for t in range(ts, ts + steps) if t % 10 == 0])
        elif "host_checks" in r:
            assert r["host_checks"] == len(c.runs), name
    assert ev["exact"]["host_checks"] == steps
