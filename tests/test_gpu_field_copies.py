"""Uploads and downloads of arrays in device memory, all fields of a call in
one launch: sizes around the launch's units (16 bytes, 16 KB), arrays aligned
to 8 bytes only (bytes for the type), arrays that overlap, part of the fields,
and host and device arrays mixed, with the state in the context's arrays and in
its records.  Every array equals the one a host download gives, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from hidem_amd import _abi as A
from hidem_amd import params
from test_gpu_device_arrays import DeviceMemory

pytestmark = pytest.mark.gpu

STEPS = 3


def at(mem, nbytes, shift):
    """A device array of nbytes, shift bytes behind a 256-byte boundary, in an allocation that just holds it."""
    base = mem.upload(np.zeros(nbytes + shift, np.uint8), C.c_uint8)
    return C.cast(base, C.c_void_p).value + shift


def put(mem, a, shift):
    a = np.ascontiguousarray(a)
    base = mem.upload(np.concatenate([np.zeros(shift, np.uint8), a.view(np.uint8).reshape(-1)]), C.c_uint8)
    return C.cast(base, C.c_void_p).value + shift


def get(mem, address, n, dtype):
    out = np.empty(n, dtype)
    mem.check(mem.hip.hipMemcpy(out.ctypes.data_as(C.c_void_p), C.c_void_p(address), C.c_size_t(out.nbytes), mem.D2H),
              "hipMemcpy")
    return out


def state(n):
    cfg = params.load_config("iceblock_16k")
    s, p, l = params.build_inputs(cfg, [12, 10, 9] if n > 480 else [6, 5, 4])
    q = A.Particles.zeros(n)
    for f in A.PARTICLE_FIELDS:
        q.arrays[f][:] = p[f][:n]
    q.type[:] = p.type[:n]
    keep = (l.a < n) & (l.b < n)
    m = int(keep.sum())
    r = np.random.default_rng(n)
    for f in ("xForce", "yForce", "zForce", "uForce", "vForce", "wForce"):
        q.arrays[f][:] = r.normal(scale=1e3, size=n)
    k = A.Links(m, l.a[keep].copy(), l.b[keep].copy(), l.state[keep].copy(), l.initialLen[keep].copy(),
                l.maxLoad[keep].copy(), [r.normal(size=2 * m) * 1e-3 for _ in range(6)])
    return s, q, k


def dp(address):
    return C.cast(C.c_void_p(address), C.POINTER(C.c_double))


@pytest.mark.parametrize("prec", [A.HDM_PREC_FP64, A.HDM_PREC_MIXED])
@pytest.mark.parametrize("n,shift,typeshift", [(2, 0, 0), (3, 8, 1), (64, 8, 3), (257, 0, 8), (2047, 16, 0),
                                               (2049, 8, 5), (4000, 0, 1)])
def test_device_fields(prec, n, shift, typeshift):
    print("  n", n, "shift", shift, flush=True)
    s, p, l = state(n)
    mem = DeviceMemory()
    ps, ls = A.HdmParticlesHost(), A.HdmLinksHost()
    ps.n, ls.n = n, l.n
    for f in A.PARTICLE_FIELDS:
        if f != "uForce":   # an optional array that is left out reads as zeros
            setattr(ps, f, dp(put(mem, p.arrays[f], shift)))
    p.arrays["uForce"][:] = 0
    ps.type = C.cast(C.c_void_p(put(mem, p.type, typeshift)), C.POINTER(C.c_uint8))
    ls.localPartIndA = C.cast(C.c_void_p(put(mem, l.a, typeshift & 4)), C.POINTER(C.c_int32))
    ls.localPartIndB = C.cast(C.c_void_p(put(mem, l.b, 0)), C.POINTER(C.c_int32))
    ls.state = C.cast(C.c_void_p(put(mem, l.state, typeshift)), C.POINTER(C.c_uint8))
    ls.initialLen, ls.maxLoad = dp(put(mem, l.initialLen, shift)), dp(put(mem, l.maxLoad, 0))
    for k in range(6):
        ls.CT[k] = dp(put(mem, l.ct[k], shift))
    with A.Context(prec) as h, A.Context(prec) as d:
        h.upload(p, l)
        d._c(A.lib().hdm_particles_upload(d._h, C.byref(ps)), "upload particles")
        d._c(A.lib().hdm_links_upload(d._h, C.byref(ls)), "upload links")
        d.n, d.L = n, l.n
        for moved in (False, True):
            if moved:
                for x in (h, d):
                    x.links_build()
                    x.run(s.run, STEPS)
            want, wl = h.download_particles(), h.download_links()
            # every field, device arrays
            out = {f: at(mem, 8 * n, shift) for f in A.PARTICLE_FIELDS}
            kind = at(mem, n, typeshift)
            qs = A.HdmParticlesHost()
            qs.n = n
            for f in A.PARTICLE_FIELDS:
                setattr(qs, f, dp(out[f]))
            qs.type = C.cast(C.c_void_p(kind), C.POINTER(C.c_uint8))
            d._c(A.lib().hdm_particles_download(d._h, C.byref(qs)), "download particles")
            for f in A.PARTICLE_FIELDS:
                assert np.array_equal(get(mem, out[f], n, np.uint64), want[f].view(np.uint64)), (moved, f)
            assert np.array_equal(get(mem, kind, n, np.uint8), want.type), moved
            # some fields, one of them in host memory
            host = np.empty(n)
            part = at(mem, 8 * n, shift)
            qs = A.HdmParticlesHost()
            qs.n = n
            qs.yDiff, qs.xCord = host.ctypes.data_as(C.POINTER(C.c_double)), dp(part)
            d._c(A.lib().hdm_particles_download(d._h, C.byref(qs)), "download particles")
            assert np.array_equal(host.view(np.uint64), want["yDiff"].view(np.uint64)), moved
            assert np.array_equal(get(mem, part, n, np.uint64), want["xCord"].view(np.uint64)), moved
            # two fields into one array: the later one stays
            qs = A.HdmParticlesHost()
            qs.n = n
            qs.xCord, qs.zTheta, qs.wForce = dp(part), dp(out["xCord"]), dp(part)
            d._c(A.lib().hdm_particles_download(d._h, C.byref(qs)), "download particles")
            assert np.array_equal(get(mem, part, n, np.uint64), want["wForce"].view(np.uint64)), moved
            assert np.array_equal(get(mem, out["xCord"], n, np.uint64), want["zTheta"].view(np.uint64)), moved
            # links
            m = l.n
            ct = [at(mem, 16 * m, shift) for _ in range(6)]
            alive, lena = at(mem, m, typeshift), at(mem, 4 * m, typeshift & 4)
            ks = A.HdmLinksHost()
            ks.n = m
            ks.state = C.cast(C.c_void_p(alive), C.POINTER(C.c_uint8))
            ks.localPartIndB = C.cast(C.c_void_p(lena), C.POINTER(C.c_int32))
            for k in range(6):
                if k != 4:
                    ks.CT[k] = dp(ct[k])
            d._c(A.lib().hdm_links_download(d._h, C.byref(ks)), "download links")
            assert np.array_equal(get(mem, alive, m, np.uint8), wl.state), moved
            assert np.array_equal(get(mem, lena, m, np.int32), l.b), moved
            for k in range(6):
                if k != 4:
                    assert np.array_equal(get(mem, ct[k], 2 * m, np.uint64), wl.ct[k].view(np.uint64)), (moved, k)
    mem.free()
