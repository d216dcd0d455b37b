"""A state fetched into device memory field by field: after the first call the
others cost what they cost from a state whose arrays are current, as the
records are read once for all of them (4 million particles: a field is copied
in about 15 us, the records take several times that to read)."""
import ctypes as C
import time

import numpy as np
import pytest

from hidem_amd import _abi as A
from hidem_amd import params
from test_gpu_device_arrays import DeviceMemory

pytestmark = pytest.mark.gpu

FIELDS = ("xCord", "yCord", "zCord", "xDiff", "yDiff", "zDiff", "uDiff", "vDiff", "wDiff")


@pytest.mark.parametrize("prec", [A.HDM_PREC_FP64, A.HDM_PREC_MIXED])
def test_records_are_read_once(prec):
    s = params.derive(params.load_config("iceblock_16k"))
    p = A.gen_fcc(100, 100, 100, 1.04 * 2 ** 0.5, 0.5, 0.01, 1, order=A.HDM_ORDER_MORTON)
    out = np.zeros(p.n)
    mem = DeviceMemory()
    dst = C.cast(mem.upload(out, C.c_double), C.POINTER(C.c_double))

    def fetch(c):
        """Median time of a call over the fields, each once."""
        t = []
        for f in FIELDS:
            q = A.HdmParticlesHost()
            q.n = p.n
            setattr(q, f, dst)
            t0 = time.perf_counter()
            c._c(A.lib().hdm_particles_download(c._h, C.byref(q)), "hdm_particles_download")
            t.append(time.perf_counter() - t0)
        return float(np.median(t))

    with A.Context(prec) as c:
        c.upload(p, A.Links.zeros(0))
        c.links_build()
        c.run(s.run, 2)
        first, current = [], []
        for _ in range(5):
            c.run(s.run, 1)
            first.append(fetch(c))      # the arrays lag the records at the first call
            c.skin_heuristic(1)         # brings them up to date, whoever asked before
            current.append(fetch(c))
        print(f"  n {p.n}: after a step {1e6 * min(first):.1f} us a field, arrays current {1e6 * min(current):.1f} us",
              flush=True)
    mem.free()
    assert min(first) <= 1.5 * min(current)
