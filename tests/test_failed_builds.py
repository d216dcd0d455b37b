"""Calls after a build that failed half-way (no GPU needed): the library runs on
a stand-in for the HIP runtime, in a process of its own, whose kernels do
nothing and whose n-th wait for the stream reports an error.  Lists and grids that
such a build has left in pieces are refused, not walked."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from hidem_amd import _abi as A

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RUNTIME = r"""
#include <hip/hip_runtime_api.h>
#include <cstdlib>
#include <cstring>
extern "C" {
int failingWait = -1;   // waits until one fails
int clearingWait = -1;  // waits until one finds the words read back at zero
void *words = nullptr;  // where results are read back
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::calloc(n, 1); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    const hipError_t e = hipMalloc(p, n);
    words = *p;
    return e;
}
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    if (clearingWait > 0 && --clearingWait == 0) std::memset(words, 0, 64);
    return failingWait > 0 && --failingWait == 0 ? hipErrorUnknown : hipSuccess;
}
}
"""

PROGRAM = r"""
import ctypes as C, sys
sys.path.insert(0, {root!r})
rt = C.CDLL({lib!r}, mode=C.RTLD_GLOBAL)
import numpy as np
from hidem_amd import _abi as A
L = A.lib()
waits = C.c_int.in_dll(rt, "failingWait")
clearing = C.c_int.in_dll(rt, "clearingWait")
p = A.Particles.zeros(3)
p.arrays["xCord"][:] = [0.0, 1.0, 2.0]
p.arrays["radius"][:] = 0.5
l = A.Links.zeros(1)
l.b[:] = 1
c = A.Context(A.HDM_PREC_FP64)
c.upload(p, l)
{body}
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    d = tmp_path_factory.mktemp("runtime")
    src, lib = str(d / "runtime.cpp"), str(d / "runtime.so")
    with open(src, "w") as f:
        f.write(RUNTIME)
    subprocess.run(["g++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-w", "-shared", "-fPIC", "-o", lib, src],
                   check=True)
    return lib


def run(runtime, body):
    r = subprocess.run([sys.executable, "-c", PROGRAM.format(root=ROOT, lib=runtime, body=body)], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return [int(v) for v in r.stdout.split()]


def test_links_build(runtime):
    """A second link build that fails when the counts are read."""
    ok, failed, after, again = run(runtime, """
n = np.zeros(3, np.int32)
lists = lambda: L.hdm_linklists_download(c._h, A._ptr(n, C.c_int32), None, None, None, None, 0)
c.links_build()
ok = lists()
waits.value = 1
failed = L.hdm_links_build(c._h)
after = lists()
c.links_build()
print(ok, failed, after, lists())
""")
    assert (ok, failed, after, again) == (A.HDM_OK, -2, -6, A.HDM_OK)


def test_grid_build(runtime):
    """A second grid build that fails behind the sort: bounds of 0 in every
    component, then statistics of 0, the latter's wait failing."""
    first, list1, failed, list2, again, list3 = run(runtime, """
words = C.c_void_p.in_dll(rt, "words")
def grid(fails=False):
    C.memmove(words.value, (C.c_uint64 * 6)(*([1 << 63] * 6)), 48)   # ordered keys of 0.0
    clearing.value = 2
    waits.value = 2 if fails else -1
    return L.hdm_grid_build(c._h, 1.0)
neighbours = lambda: L.hdm_neighbours_build(c._h, 0.1)
c.links_build()
print(grid(), neighbours(), grid(True), neighbours(), grid(), neighbours())
""")
    assert (first, list1, again, list3) == (A.HDM_OK,) * 4
    assert (failed, list2) == (-2, -6)


def test_grid_out_of_range(runtime):
    """A grid of too many cells after one that was built, which stays."""
    first, failed, cells, after = run(runtime, """
words = C.c_void_p.in_dll(rt, "words")
clearing.value = 2
C.memmove(words.value, (C.c_uint64 * 6)(*([1 << 63] * 6)), 48)
first = L.hdm_grid_build(c._h, 1.0)
far = int(np.array([1e8]).view(np.uint64)[0])
C.memmove(words.value, (C.c_uint64 * 6)(*([1 << 63] * 3 + [far | 1 << 63] * 3)), 48)
failed = L.hdm_grid_build(c._h, 1.0)
g = c.grid_info()
C.memset(words.value, 0, 64)
print(first, failed, g.X * g.Y * g.Z, L.hdm_neighbours_build(c._h, 0.1))
""")
    assert (first, failed, cells, after) == (A.HDM_OK, -5, 1, A.HDM_OK)
