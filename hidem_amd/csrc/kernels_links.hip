// Per-particle link lists and the side (CT) layout for gfx950.
//
//   link_count   LinkAccelSide::getMaxLinksPerParticle (LinkAccelSide.h:69-90)
//   link_fill    LinkAccelSide::generateLinks (:92-143): each link side placed
//                in a slot of its endpoint (the rank it was counted with), then
//                every particle's slots are sorted ascending (the reference
//                bubble-sorts, :123-137); generatePerParticleIndexes (:43-67)
//                resolves the other endpoint and which end this particle is.
//   ct_import /  LinkAccelSide::sortSideData + LinkDataHandler::
//   ct_export    reorderSideDataPadded (LinkDataHandler.h:176-191): the CT
//                side arrays are permuted so that particle p's k-th link side
//                lives in wave-tile slot k of p (the reference's AOS_CT order
//                makes each particle's sides contiguous; the wave tile makes
//                slot k of 64 consecutive particles contiguous instead, which
//                is what a 64-lane wavefront reads in one access).  sidePos
//                plays the role of sideIndEndA/B (LinkData::reindexSideData,
//                LinkData.h:183-208).
#include <cstring>

#include "hdm_context.h"
#include "kernel_common.h"

namespace hdm {

namespace {

constexpr int TPB = 256;

__device__ inline int64_t slot_index(int64_t p, int32_t k, int32_t width) {
    return (p >> 6) * (int64_t)64 * width + (int64_t)k * 64 + (p & 63);
}

// Links per particle, and in rank[2l], rank[2l + 1] the place of link l's two
// sides among their particles' in the order the additions came (k_link_sort
// settles it).  Bound by the atomics: a run of lanes with one first endpoint,
// as lists sorted by it have, shares an addition.  Every lane of the wave
// stays for the exchange.
__global__ void __launch_bounds__(TPB) k_link_count(const int32_t *__restrict__ A, const int32_t *__restrict__ B,
                                                     int64_t L, int64_t n, uint32_t *__restrict__ count,
                                                     int32_t *__restrict__ rank, uint64_t *errFlag) {
    const int64_t l = xcd_block_index(gridDim.x) * TPB + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int32_t a = l < L ? A[l] : 0, b = l < L ? B[l] : 0;
    const bool ok = l < L && a >= 0 && a < n && b >= 0 && b < n && a != b;
    if (l < L && !ok) atomicOr((unsigned long long *)errFlag, 1ull);
    const int32_t key = ok ? a : -1 - lane;   // a lane that is left out is a run of its own
    const int32_t before = __shfl_up(key, 1, 64);
    const uint64_t heads = __ballot(lane == 0 || before != key);
    const int leader = 63 - __clzll(heads & (~0ull >> (63 - lane)));
    const uint64_t after = lane == 63 ? 0 : heads >> (lane + 1);
    const int run = after ? __ffsll((unsigned long long)after) : 64 - lane;   // of a leader
    uint32_t ka = 0;
    if (ok && lane == leader) ka = atomicAdd(&count[a], (uint32_t)run);
    const uint32_t kb = ok ? atomicAdd(&count[b], 1u) : 0;
    ka = __shfl(ka, leader, 64) + (uint32_t)(lane - leader);
    if (ok) *reinterpret_cast<int2 *>(rank + 2 * l) = make_int2((int32_t)ka, (int32_t)kb);
}

// Side 2l (of endpoint A) and 2l + 1 (of B) of each link and the particle it
// leads to, with the broken flag, into their particles' slots.
__global__ void __launch_bounds__(TPB) k_link_fill(const int32_t *__restrict__ A, const int32_t *__restrict__ B,
                                                    const uint8_t *__restrict__ state, int64_t L, int32_t width,
                                                    const int32_t *__restrict__ rank, int32_t *__restrict__ slotLink,
                                                    int32_t *__restrict__ slotOther) {
    const int64_t l = xcd_block_index(gridDim.x) * TPB + threadIdx.x;
    if (l >= L) return;
    const int32_t a = A[l], b = B[l];
    const int32_t broken = state[l] == 0 ? SLOT_BROKEN : 0;
    const int2 k = *reinterpret_cast<const int2 *>(rank + 2 * l);
    const int64_t sa = slot_index(a, k.x, width), sb = slot_index(b, k.y, width);
    slotLink[sa] = (int32_t)(2 * l);
    slotOther[sa] = b | broken;
    slotLink[sb] = (int32_t)(2 * l + 1);
    slotOther[sb] = a | broken;
}

// A particle's slots: element k of the wave tile's column (LDS: the wave's copy).
struct Column {
    int32_t *side, *other;
    __device__ __forceinline__ int32_t &s(int k) const { return side[(int64_t)k * 64]; }
    __device__ __forceinline__ int32_t &o(int k) const { return other[(int64_t)k * 64]; }
};

// One wave per wave tile.  Sorts each particle's sides ascending, replaces
// them by link ids, notes each side's slot, and flags a particle whose sides
// name one partner twice, or itself.  Both slot words carry the link's broken
// flag in their sign bit, so the force gather needs no per-link state lookup.
// Bound by the latency of the exchanges: tiles of up to LINK_LDS_WIDTH slots
// are sorted in LDS, wider ones in place.  With the sort in memory, a second
// pass of atomics for the slots and the partner check in a launch of its own
// the lists of 290k particles with 1.7M links took 306 us, now 91.
constexpr int LINK_LDS_WIDTH = 64;

template <bool LDS>
__global__ void __launch_bounds__(64) k_link_sort(int64_t n, int32_t width, const uint32_t *__restrict__ count,
                                                   int32_t *slotLink, int32_t *slotOther,
                                                   int32_t *__restrict__ sidePos, uint64_t *dupFlag) {
    extern __shared__ int32_t tile[];   // LDS: [2][width][64]
    const int lane = threadIdx.x;
    const int64_t p = xcd_block_index(gridDim.x) * 64 + lane;
    if (p >= n) return;
    const int cnt = (int)count[p];
    const int64_t base = slot_index(p, 0, width);
    const Column mem{slotLink + base, slotOther + base};
    const Column c = LDS ? Column{tile + lane, tile + width * 64 + lane} : mem;
    if constexpr (LDS)
        for (int k = 0; k < cnt; k++) {
            c.s(k) = mem.s(k);
            c.o(k) = mem.o(k);
        }
    for (int i = 1; i < cnt; i++) {
        const int32_t v = c.s(i), w = c.o(i);
        int j = i - 1;
        while (j >= 0 && c.s(j) > v) {
            c.s(j + 1) = c.s(j);
            c.o(j + 1) = c.o(j);
            j--;
        }
        c.s(j + 1) = v;
        c.o(j + 1) = w;
    }
    bool dup = false;
    for (int k = 0; k < cnt; k++) {
        const int32_t side = c.s(k), other = c.o(k), q = other & SLOT_LINK_MASK;
        dup |= q == (int32_t)p;
        for (int j = 0; j < k && !dup; j++) dup = (c.o(j) & SLOT_LINK_MASK) == q;
        sidePos[side] = (int32_t)(base + (int64_t)k * 64);
        mem.s(k) = (side >> 1) | (other & SLOT_BROKEN);
        if constexpr (LDS) mem.o(k) = other;
    }
    if (dup) atomicOr((unsigned long long *)dupFlag, 1ull);
}

// The strain of one side at its place in the tile (ct_offset), in the vector
// accesses of ct_load and ct_store; ordinary ones, as other sides share the
// lines.
template <class CT>
__device__ __forceinline__ void ct_get(const CT *ct, int64_t d, CT v[6]) {
    if constexpr (sizeof(CT) == 4) {
        const ct_f4 a = *reinterpret_cast<const ct_f4 *>(ct + ct_offset<CT>(d, 0));
        const ct_f2 b = *reinterpret_cast<const ct_f2 *>(ct + ct_offset<CT>(d, 4));
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y;
    } else {
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const ct_d2 a = *reinterpret_cast<const ct_d2 *>(ct + ct_offset<CT>(d, 2 * j));
            v[2 * j] = a.x;
            v[2 * j + 1] = a.y;
        }
    }
}

template <class CT>
__device__ __forceinline__ void ct_put(CT *ct, int64_t d, const CT v[6]) {
    if constexpr (sizeof(CT) == 4) {
        *reinterpret_cast<ct_f4 *>(ct + ct_offset<CT>(d, 0)) = ct_f4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<ct_f2 *>(ct + ct_offset<CT>(d, 4)) = ct_f2{v[4], v[5]};
    } else {
#pragma unroll
        for (int j = 0; j < 3; j++) *reinterpret_cast<ct_d2 *>(ct + ct_offset<CT>(d, 2 * j)) = ct_d2{v[2 * j], v[2 * j + 1]};
    }
}

template <class CT>
__global__ void __launch_bounds__(TPB) k_ct_import(const int32_t *__restrict__ sidePos, int64_t nSides,
                                                    const double *__restrict__ s0, const double *__restrict__ s1,
                                                    const double *__restrict__ s2, const double *__restrict__ s3,
                                                    const double *__restrict__ s4, const double *__restrict__ s5,
                                                    CT *__restrict__ ct) {
    const int64_t i = xcd_block_index(gridDim.x) * TPB + threadIdx.x;
    if (i >= nSides) return;
    const CT v[6] = {(CT)s0[i], (CT)s1[i], (CT)s2[i], (CT)s3[i], (CT)s4[i], (CT)s5[i]};
    ct_put(ct, (int64_t)sidePos[i], v);
}

template <class CT>
__global__ void __launch_bounds__(TPB) k_ct_export(const int32_t *__restrict__ sidePos, int64_t nSides,
                                                    const CT *__restrict__ ct, double *__restrict__ s0,
                                                    double *__restrict__ s1, double *__restrict__ s2,
                                                    double *__restrict__ s3, double *__restrict__ s4,
                                                    double *__restrict__ s5) {
    const int64_t i = xcd_block_index(gridDim.x) * TPB + threadIdx.x;
    if (i >= nSides) return;
    CT v[6];
    ct_get(ct, (int64_t)sidePos[i], v);
    if (s0) s0[i] = (double)v[0];
    if (s1) s1[i] = (double)v[1];
    if (s2) s2[i] = (double)v[2];
    if (s3) s3[i] = (double)v[3];
    if (s4) s4[i] = (double)v[4];
    if (s5) s5[i] = (double)v[5];
}

// Break prefilter thresholds, in two passes after the link build.
// Pass 1 (per link): the largest L0 (as float bits, rounded up; +inf when
// some L0 is not finite), which bounds the bend term, and the largest
// threshold T = L0 (1 + maxLoad) with per-link maxLoad, else L0 (float bits,
// rounded up), which sets the scale of the codes.
__device__ __forceinline__ float float_up(double v) {
    const float f = (float)v;
    return (double)f < v ? __uint_as_float(__float_as_uint(f) + 1u) : f;  // next float up
}

// Largest value over a workgroup, to *part as its bits.
__device__ __forceinline__ void block_max_bits(float v, uint64_t *part) {
    __shared__ uint32_t waves[TPB / 64];
    // non-negative floats order as their bit patterns
    const uint32_t bits = wave_max_u32(__float_as_uint(v));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) waves[threadIdx.x >> 6] = bits;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t m = waves[0];
        for (int w = 1; w < TPB / 64; w++) m = waves[w] > m ? waves[w] : m;
        *part = m;
    }
}

__global__ void __launch_bounds__(TPB) k_threshold_max(int64_t L, const double *__restrict__ initialLen,
                                                        const double *__restrict__ maxLoad, uint64_t *part) {
    float bigL0 = 0.0f, bigT = 0.0f;
    for (int64_t l = (int64_t)blockIdx.x * TPB + threadIdx.x; l < L; l += (int64_t)gridDim.x * TPB) {
        const double L0 = initialLen[l];
        if (L0 >= 1e-30 && L0 <= 1e300) {
            const double T = maxLoad ? L0 * (1.0 + maxLoad[l]) : L0;
            const float b = float_up(L0);
            bigL0 = b > bigL0 ? b : bigL0;
            if (T > 0.0 && T <= 1e300) {
                const float t = float_up(T);
                bigT = t > bigT ? t : bigT;
            }
        } else if (!(L0 < 1e-30)) {
            bigL0 = __builtin_inff();  // NaN or huge: no useful bound
        }
    }
    block_max_bits(bigL0, part + blockIdx.x);
    block_max_bits(bigT, part + RED_BLOCKS + blockIdx.x);
}

// Pass 2 (per side, into its wave-tile slot): a 16-bit code with
// code * scale <= T, code = floor(T / scale) held to 65535, where scale is
// the largest T / 65535 (so codes resolve T to 1.5e-5 of the largest); 0
// (never passes) when L0 is below 1e-30, not finite, or no scale exists.
// The prefilter reads 2 B per side; the exact test still reads the FP64
// initialLen and maxLoad.
__global__ void __launch_bounds__(TPB) k_side_codes(const int32_t *__restrict__ sidePos, int64_t nSides,
                                                     const double *__restrict__ initialLen,
                                                     const double *__restrict__ maxLoad, double scale,
                                                     uint16_t *__restrict__ slotThr) {
    for (int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x; i < nSides; i += (int64_t)gridDim.x * TPB) {
        const int64_t l = i >> 1;
        const double L0 = initialLen[l];
        const bool ok = L0 >= 1e-30 && L0 <= 1e300 && scale > 0.0;
        const double T = maxLoad ? L0 * (1.0 + maxLoad[l]) : L0;
        double q = ok ? floor(T / scale) : 0.0;
        if (!(q >= 0.0)) q = 0.0;  // also NaN
        if (q > 65535.0) q = 65535.0;
        slotThr[sidePos[i]] = (uint16_t)q;
    }
}

__global__ void __launch_bounds__(TPB) k_count_broken(const uint8_t *__restrict__ state, int64_t L, uint64_t *out) {
    uint32_t c = 0;
    for (int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x; i < L; i += (int64_t)gridDim.x * TPB)
        c += state[i] == 0 ? 1u : 0u;
    c = wave_sum_u32(c);
    if ((threadIdx.x & 63) == 0 && c) atomicAdd((unsigned long long *)out, (unsigned long long)c);
}

// computeActiveLinks and computeIteratedNeighbours (HiDEMLib.h:197-232): a
// particle's links with state != 0 (iterateParticleLinksCT over its slots),
// and the entries of the reference's neighbour list (the list as built plus
// the link partners it leaves out).  Sums over all particles (all are owned
// on one GPU) as finalizeTs reduces them (HiDEMLib.h:518-523).
__global__ void __launch_bounds__(TPB) k_particle_stats(const uint32_t *__restrict__ linkCount,
                                                         const int32_t *__restrict__ slotLink, int32_t width,
                                                         const uint8_t *__restrict__ state,
                                                         const int32_t *__restrict__ nbrCount,
                                                         const int32_t *__restrict__ nbrLinked, int64_t n,
                                                         int32_t *__restrict__ activeOut,
                                                         int32_t *__restrict__ nbrOut, uint64_t *sums) {
    const int64_t p = (int64_t)blockIdx.x * TPB + threadIdx.x;
    uint32_t act = 0, nb = 0;
    if (p < n) {
        const uint32_t cnt = linkCount[p];
        const int64_t base = (p >> 6) * (int64_t)64 * width + (p & 63);
        for (uint32_t k = 0; k < cnt; k++) act += state[slotLink[base + (int64_t)k * 64] & SLOT_LINK_MASK] ? 1u : 0u;
        nb = (uint32_t)nbrCount[p] + (nbrLinked ? (uint32_t)nbrLinked[p] : 0u);
        if (activeOut) activeOut[p] = (int32_t)act;
        if (nbrOut) nbrOut[p] = (int32_t)nb;
    }
    act = wave_sum_u32(act);
    nb = wave_sum_u32(nb);
    if ((threadIdx.x & 63) == 0) {
        if (act) atomicAdd((unsigned long long *)&sums[0], (unsigned long long)act);
        if (nb) atomicAdd((unsigned long long *)&sums[1], (unsigned long long)nb);
    }
}

inline int blocks_for(int64_t n) { return (int)((n + TPB - 1) / TPB); }

}  // namespace

hipError_t launch_particle_stats(Context &c, int32_t *activeLinks, int32_t *iteratedNeighbours, uint64_t *sums) {
    hipError_t e = launch_fill_u64(c.stream, sums, 0ull, 2);
    if (e != hipSuccess || c.n == 0) return e;
    hipLaunchKernelGGL(k_particle_stats, dim3(blocks_for(c.n)), dim3(TPB), 0, c.stream, c.linkCount.as<uint32_t>(),
                       c.slotLink.as<int32_t>(), c.maxLinks, c.state.as<uint8_t>(), c.nbrCount.as<int32_t>(),
                       c.nbrExcludesLinked ? c.nbrLinked.as<int32_t>() : (const int32_t *)nullptr, c.n, activeLinks,
                       iteratedNeighbours, sums);
    return hipGetLastError();
}

hipError_t launch_link_count(Context &c) {
    hipError_t e = launch_fill_u32(c.stream, c.linkCount.as<uint32_t>(), 0u, c.n);
    if (e != hipSuccess) return e;
    uint64_t *err = c.red.as<uint64_t>() + RED_LINKS + 1;
    e = launch_fill_u64(c.stream, err, 0ull, 2);   // and the partner flag
    if (e != hipSuccess) return e;
    if (c.L > 0)
        hipLaunchKernelGGL(k_link_count, dim3(blocks_for(c.L)), dim3(TPB), 0, c.stream, c.la.as<int32_t>(),
                           c.lb.as<int32_t>(), c.L, c.n, c.linkCount.as<uint32_t>(), c.sidePos.as<int32_t>(), err);
    return hipGetLastError();
}

hipError_t launch_link_fill(Context &c) {
    uint64_t *dup = c.red.as<uint64_t>() + RED_LINKS + 2;
    if (c.L > 0)
        hipLaunchKernelGGL(k_link_fill, dim3(blocks_for(c.L)), dim3(TPB), 0, c.stream, c.la.as<int32_t>(),
                           c.lb.as<int32_t>(), c.state.as<uint8_t>(), c.L, c.maxLinks, c.sidePos.as<int32_t>(),
                           c.slotLink.as<int32_t>(), c.slotOther.as<int32_t>());
    const dim3 grid((unsigned)c.tiles());
    const uint32_t *count = c.linkCount.as<uint32_t>();
    if (c.maxLinks <= LINK_LDS_WIDTH)
        hipLaunchKernelGGL(k_link_sort<true>, grid, dim3(64), sizeof(int32_t) * 128 * (size_t)c.maxLinks, c.stream, c.n,
                           c.maxLinks, count, c.slotLink.as<int32_t>(), c.slotOther.as<int32_t>(),
                           c.sidePos.as<int32_t>(), dup);
    else
        hipLaunchKernelGGL(k_link_sort<false>, grid, dim3(64), 0, c.stream, c.n, c.maxLinks, count,
                           c.slotLink.as<int32_t>(), c.slotOther.as<int32_t>(), c.sidePos.as<int32_t>(), dup);
    return hipGetLastError();
}

hipError_t launch_ct_import(Context &c) {
    int64_t nSides = 2 * c.L;
    if (nSides == 0) return hipSuccess;
    const double *s[6];
    for (int k = 0; k < 6; k++) s[k] = c.ctStage[k].as<double>();
    if (c.prec == HDM_PREC_FP64)
        hipLaunchKernelGGL(k_ct_import<double>, dim3(blocks_for(nSides)), dim3(TPB), 0, c.stream,
                           c.sidePos.as<int32_t>(), nSides, s[0], s[1], s[2], s[3], s[4], s[5], c.ct.as<double>());
    else
        hipLaunchKernelGGL(k_ct_import<float>, dim3(blocks_for(nSides)), dim3(TPB), 0, c.stream,
                           c.sidePos.as<int32_t>(), nSides, s[0], s[1], s[2], s[3], s[4], s[5], c.ct.as<float>());
    return hipGetLastError();
}

hipError_t launch_ct_export(Context &c, double *const out[6]) {
    int64_t nSides = 2 * c.L;
    if (nSides == 0) return hipSuccess;
    double *s[6];
    for (int k = 0; k < 6; k++) s[k] = out ? out[k] : c.ctStage[k].as<double>();
    if (c.prec == HDM_PREC_FP64)
        hipLaunchKernelGGL(k_ct_export<double>, dim3(blocks_for(nSides)), dim3(TPB), 0, c.stream,
                           c.sidePos.as<int32_t>(), nSides, c.ct.as<double>(), s[0], s[1], s[2], s[3], s[4], s[5]);
    else
        hipLaunchKernelGGL(k_ct_export<float>, dim3(blocks_for(nSides)), dim3(TPB), 0, c.stream,
                           c.sidePos.as<int32_t>(), nSides, c.ct.as<float>(), s[0], s[1], s[2], s[3], s[4], s[5]);
    return hipGetLastError();
}

hipError_t launch_side_thresholds(Context &c, float *l0Max, float *scale) {
    *l0Max = 0.0f;
    *scale = 0.0f;
    const int64_t nSides = 2 * c.L;
    c.partnersUnique = true;
    if (nSides == 0) return hipSuccess;
    const int cap = c.numCU > 0 ? c.numCU * 8 : 2048;
    const double *ml = c.hasMaxLoad ? c.maxLoad.as<double>() : nullptr;
    const int grid = reduce_blocks(c, c.L);
    hipLaunchKernelGGL(k_threshold_max, dim3(grid), dim3(TPB), 0, c.stream, c.L, c.initialLen.as<double>(), ml,
                       c.red.as<uint64_t>() + RED_PARTS);
    uint64_t *words = c.red.as<uint64_t>() + RED_LINKS + 2;   // partner flag, largest L0, largest threshold
    hipError_t e = launch_fold(c, grid, 2, 0u, words + 1);
    if (e != hipSuccess) return e;
    uint64_t w[3] = {0, 0, 0};
    e = read_back(c, w, words, sizeof(w));
    if (e != hipSuccess) return e;
    c.partnersUnique = w[0] == 0;
    const uint32_t b0 = (uint32_t)w[1], b1 = (uint32_t)w[2];
    float tMax;
    std::memcpy(l0Max, &b0, sizeof(float));
    std::memcpy(&tMax, &b1, sizeof(float));
    float s = tMax / 65535.0f;
    if (!(s > 0.0f && s < 3e38f)) s = 0.0f;
    *scale = s;
    const int64_t nb = blocks_for(nSides);
    hipLaunchKernelGGL(k_side_codes, dim3((unsigned)(nb < cap ? nb : cap)), dim3(TPB), 0, c.stream,
                       c.sidePos.as<int32_t>(), nSides, c.initialLen.as<double>(), ml, (double)s,
                       c.slotThr.as<uint16_t>());
    return hipGetLastError();
}

hipError_t launch_count_broken(Context &c, uint64_t *counter) {
    hipError_t e = launch_fill_u64(c.stream, counter, 0ull, 1);
    if (e != hipSuccess) return e;
    if (c.L == 0) return hipSuccess;
    int64_t nb = blocks_for(c.L);
    int cap = c.numCU > 0 ? c.numCU * 4 : 1024;
    int grid = (int)(nb < cap ? nb : cap);
    hipLaunchKernelGGL(k_count_broken, dim3(grid), dim3(TPB), 0, c.stream, c.state.as<uint8_t>(), c.L, counter);
    return hipGetLastError();
}

}  // namespace hdm
