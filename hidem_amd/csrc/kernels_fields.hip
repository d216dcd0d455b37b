// Whole-array transfers between the context's arrays and arrays of the
// caller in device memory: every field of an upload or a download in one
// launch.  A copy per field costs 6 us on the device and, where each is waited
// for, 16 us of host time, which for states of some thousand particles is more
// than the steps between two downloads (50 steps and a download of 20 arrays:
// 593 -> 394 us at 960 particles, 1181 -> 981 us at 16k).
#include <cstring>

#include "hdm_context.h"
#include "kernel_common.h"

namespace hdm {

namespace {

constexpr int TPB = 256;
constexpr int64_t CHUNK = 16384;               // bytes of the wider side per workgroup
constexpr int64_t CHUNK_VALUES = CHUNK / 8;    // values, where the type changes

// One workgroup's chunk of a plain copy in units of V, all loads in flight
// before the first store; the bytes past the last whole unit go one by one.
template <class V>
__device__ __forceinline__ void copy_chunk(const FieldCopy &f, int64_t base) {
    constexpr int K = (int)(CHUNK / (TPB * (int64_t)sizeof(V)));
    constexpr int B = K < 8 ? K : 8;
    const char *src = static_cast<const char *>(f.src);
    char *dst = static_cast<char *>(f.dst);
    for (int k0 = 0; k0 < K; k0 += B) {
        V v[B];
#pragma unroll
        for (int k = 0; k < B; k++) {
            const int64_t o = base + ((k0 + k) * TPB + (int)threadIdx.x) * (int64_t)sizeof(V);
            if (o + (int64_t)sizeof(V) <= f.count) v[k] = *reinterpret_cast<const V *>(src + o);
        }
#pragma unroll
        for (int k = 0; k < B; k++) {
            const int64_t o = base + ((k0 + k) * TPB + (int)threadIdx.x) * (int64_t)sizeof(V);
            if (o + (int64_t)sizeof(V) <= f.count) *reinterpret_cast<V *>(dst + o) = v[k];
        }
    }
    const int64_t rest = f.count - f.count % (int64_t)sizeof(V);
    if (rest >= base && rest < base + CHUNK && rest + (int)threadIdx.x < f.count)
        dst[rest + threadIdx.x] = src[rest + threadIdx.x];
}

template <class S, class D>
__device__ __forceinline__ void convert_chunk(const FieldCopy &f, int64_t base) {
    const S *src = static_cast<const S *>(f.src);
    D *dst = static_cast<D *>(f.dst);
    S v[CHUNK_VALUES / TPB];
#pragma unroll
    for (int k = 0; k < CHUNK_VALUES / TPB; k++) {
        const int64_t i = base + k * TPB + threadIdx.x;
        if (i < f.count) v[k] = src[i];
    }
#pragma unroll
    for (int k = 0; k < CHUNK_VALUES / TPB; k++) {
        const int64_t i = base + k * TPB + threadIdx.x;
        if (i < f.count) dst[i] = (D)v[k];
    }
}

// Bound by memory: 16 KB per workgroup in 16-byte units where both sides are
// aligned to them (else 8-byte units, else bytes), blockIdx.y the field.
__global__ void __launch_bounds__(TPB) k_copy_fields(FieldCopies a) {
    const FieldCopy f = a.f[blockIdx.y];
    const int64_t chunk = blockIdx.x;
    if (f.kind == FieldCopy::WIDEN || f.kind == FieldCopy::NARROW) {
        if (chunk * CHUNK_VALUES >= f.count) return;
        if (f.kind == FieldCopy::WIDEN) convert_chunk<float, double>(f, chunk * CHUNK_VALUES);
        else convert_chunk<double, float>(f, chunk * CHUNK_VALUES);
        return;
    }
    if (chunk * CHUNK >= f.count) return;
    if (f.kind == FieldCopy::ZERO) {   // the context's own arrays: whole allocations, 256-byte aligned
        char *dst = static_cast<char *>(f.dst);
        for (int k = 0; k < (int)(CHUNK / (TPB * 16)); k++) {
            const int64_t o = chunk * CHUNK + (k * TPB + (int)threadIdx.x) * 16;
            if (o + 16 <= f.count) *reinterpret_cast<uint4 *>(dst + o) = make_uint4(0, 0, 0, 0);
            else for (int64_t t = o; t < f.count; t++) dst[t] = 0;
        }
        return;
    }
    const uint64_t at = reinterpret_cast<uint64_t>(f.src) | reinterpret_cast<uint64_t>(f.dst);
    if ((at & 15) == 0) copy_chunk<uint4>(f, chunk * CHUNK);
    else if ((at & 7) == 0) copy_chunk<uint2>(f, chunk * CHUNK);
    else copy_chunk<uint8_t>(f, chunk * CHUNK);
}

// Words of a small result into host memory that the device can write.  reset:
// then set these to zero (words of the result).
__global__ void __launch_bounds__(TPB) k_read_back(const uint32_t *src, int n, uint32_t *host, uint32_t *reset,
                                                   int nReset, const uint32_t *second) {
    for (int i = threadIdx.x; i < n; i += TPB) host[i] = src[i];
    if (second && threadIdx.x < 2) host[n + threadIdx.x] = second[threadIdx.x];
    __syncthreads();
    for (int i = threadIdx.x; i < nReset; i += TPB) reset[i] = 0;
}

}  // namespace

hipError_t read_back(Context &c, void *dst, const void *src, size_t bytes, uint32_t *reset, int nReset) {
    return read_back_with(c, dst, src, bytes, reset, nReset, nullptr, nullptr);
}

hipError_t read_back_with(Context &c, void *dst, const void *src, size_t bytes, uint32_t *reset, int nReset,
                          const uint64_t *second, uint64_t *value) {
    if (!c.mail || bytes + (second ? 8 : 0) > MAIL_BYTES || bytes % 4 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_read_back, dim3(1), dim3(TPB), 0, c.stream, static_cast<const uint32_t *>(src),
                       (int)(bytes / 4), static_cast<uint32_t *>(c.mail), reset, nReset,
                       reinterpret_cast<const uint32_t *>(second));
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(c.stream);
    if (e == hipSuccess) std::memcpy(dst, c.mail, bytes);
    if (e == hipSuccess && second) std::memcpy(value, static_cast<const char *>(c.mail) + bytes, sizeof(*value));
    return e;
}

hipError_t launch_copy_fields(hipStream_t stream, const FieldCopies &a) {
    int64_t chunks = 0;
    for (int k = 0; k < a.n; k++) {
        const FieldCopy &f = a.f[k];
        const bool converts = f.kind == FieldCopy::WIDEN || f.kind == FieldCopy::NARROW;
        const int64_t c = (f.count + (converts ? CHUNK_VALUES : CHUNK) - 1) / (converts ? CHUNK_VALUES : CHUNK);
        chunks = c > chunks ? c : chunks;
    }
    if (chunks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy_fields, dim3((unsigned)chunks, (unsigned)a.n), dim3(TPB), 0, stream, a);
    return hipGetLastError();
}

}  // namespace hdm
