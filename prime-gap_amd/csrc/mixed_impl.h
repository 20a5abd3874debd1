// mixed_impl.h -- numbers of several widths in one persistent, work-queue launch.
//
// Reference counterpart: the reference compiles one container width per
// binary (BITS, gap_test_gpu.cu:48-55, suggested ladder :669-686), so a
// mixed workload either runs in the widest container or in one run per
// width.  Here the numbers are grouped into size buckets.  The one-lane buckets
// below a cut that the call's sizes give (mixed.hip) are divided into tiles of one wavefront (64 numbers), tiles are queued
// widest first (longest-processing-time order), and a persistent grid of waves
// pulls tiles from an atomic counter; each wave runs the radix-2^28 variant of
// its tile's bucket.  Every wave leaves when the queue is empty.  The others run one
// number per wavefront on the matrix cores, over all their containers, widest
// first.  40% 705, 30% 2128 and 30% 4247 bits: 16411 numbers
// in 26.2 ms and 131072 in 191, against 93.2 and 309 with the wide ones on 8
// lanes each and every other bucket in one-lane tiles; 2^19 narrow ones fill
// the one-lane tiles and take 164 ms either way.
#pragma once
#include <algorithm>
#include "kernels.h"
#include "prp28.h"
#include "prp_mf.h"

namespace pgap {

// One number per lane with L digits (prp28.h).
template <int... Ls>
struct Buckets {
    static constexpr int n = sizeof...(Ls);
    static constexpr int digits[n] = {Ls...};
};
// Up to 332, 724, 1116, 1564 and 2180-bit numbers (Fermat base 2).
using MixedOneLane = Buckets<12, 26, 40, 56, 78>;
// The widest number a call takes: 160 digits of 28 bits, less 4 (Fermat) or 8.
constexpr int kMixedMaxBits = 28 * 160;
constexpr int kMixedContainers = 9;  // matrix-core containers of 1 .. 9 blocks (mont_mf.h)
static_assert(mf::max_bits(kMixedContainers) >= kMixedMaxBits, "the last container takes every number");
// Cycles of a squaring, measured at the buckets' upper widths: of a one-lane tile
// alone on its SIMD, by bucket (3311, 11001, 20056, 31691 and 38473 numbers of 330,
// 720, 1110, 1560 and 2128 bits in 0.27, 2.0, 5.4, 14.2 and 46.8 ms), and of a SIMD
// per number in mixed_mf_kernel, by blocks (the same numbers in 0.32, 2.3, 7.3, 16.8
// and 40.9 ms: two wavefronts per SIMD cost the narrow ones 20 to 30%).
constexpr double kTileCycles[MixedOneLane::n] = {2000, 6700, 11700, 21800, 52500};
constexpr double kMixedMatrixCycles[6] = {0, 740, 700, 800, 840, 1250};

// LDS park of the widest one-lane bucket (the last), one column per thread.
constexpr size_t kMixedParkBytes =
    (size_t)MixedOneLane::digits[MixedOneLane::n - 1] * r28::PARK_STRIDE * sizeof(uint32_t);

// One test of one number.  A strong-PRP launch tests one base, bases.b[0]
// (the host runs later bases on the survivors), so no loop keeps a test live
// across bases.  The kernel is scheduled for two wavefronts per SIMD, the
// batch kernels' choice for the widest bucket, so the wide squaring uses one
// chain per column.
template <int KIND, int L>
__device__ __forceinline__ uint32_t test_one(const uint32_t *nw, uint32_t limbs, const Bases &bases,
                                             uint32_t *park) {
    if (KIND == KIND_FERMAT2) return r28::fermat2<L, 1>(nw, limbs, park);
    return r28::sprp<L, 1>(nw, limbs, bases.b[0], park);
}

// One tile of a bucket in this wave: order[64 t + lane].
template <int KIND, int L>
__device__ __forceinline__ void run_tile(const uint32_t *words, const uint64_t *offset, const uint32_t *limbs,
                                         const uint32_t *order, uint32_t t, uint32_t lane, const Bases &bases,
                                         uint32_t *lds, uint8_t *out) {
    const uint32_t item = order[(size_t)t * 64 + lane];
    if (item == 0xffffffffu) return;
    out[item] = (uint8_t)test_one<KIND, L>(words + offset[item], limbs[item], bases, lds + threadIdx.x);
}

template <int KIND, int... Ls>
__device__ __forceinline__ void dispatch(int bucket, const uint32_t *words, const uint64_t *offset,
                                         const uint32_t *limbs, const uint32_t *order, uint32_t t, uint32_t lane,
                                         const Bases &bases, uint32_t *lds, uint8_t *out, Buckets<Ls...>) {
    int i = 0;
    ((bucket == i++ ? run_tile<KIND, Ls>(words, offset, limbs, order, t, lane, bases, lds, out) : (void)0), ...);
}

// Pull tiles until the queue is empty.
template <int KIND, class BL>
__device__ __forceinline__ void mixed_loop(const uint32_t *words, const uint64_t *offset, const uint32_t *limbs,
                                           const uint32_t *order, const uint8_t *tile_bucket, uint32_t ntiles,
                                           uint32_t *next_tile, const Bases &bases, uint32_t *lds, uint8_t *out) {
    const uint32_t lane = threadIdx.x & 63;
    for (;;) {
        uint32_t t = 0;
        if (lane == 0) t = atomicAdd(next_tile, 1u);
        t = (uint32_t)__shfl((int)t, 0, 64);
        if (t >= ntiles) break;
        dispatch<KIND>(tile_bucket[t], words, offset, limbs, order, t, lane, bases, lds, out, BL{});
    }
}

template <int KIND>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) mixed_kernel(const uint32_t *__restrict__ words,
                                                    const uint64_t *__restrict__ offset,
                                                    const uint32_t *__restrict__ limbs,
                                                    const uint32_t *__restrict__ order,
                                                    const uint8_t *__restrict__ tile_bucket, uint32_t ntiles,
                                                    uint32_t *__restrict__ next_tile, Bases bases,
                                                    uint8_t *__restrict__ out) {
    extern __shared__ uint32_t mixed_lds[];
    mixed_loop<KIND, MixedOneLane>(words, offset, limbs, order, tile_bucket, ntiles, next_tile, bases, mixed_lds,
                                   out);
}

// Matrix-core numbers: workgroup i (one wavefront) tests order[first + i]; end[k]
// is the end of the items of containers of more than k blocks, widest first.  Two
// wavefronts per SIMD, what the widest container's registers allow.  One test a
// wavefront and more launches instead of a loop: around the nine test bodies a
// loop takes 245 registers instead of 206 and spills 22 scalar ones.
struct MixedEnds {
    uint32_t end[kMixedContainers];
};
template <int KIND, int KB>
__device__ __forceinline__ uint32_t matrix_test(int blocks, const uint32_t *nw, uint32_t limbs, uint32_t base,
                                                uint32_t *lds) {
    if constexpr (KB > 0) {
        if (blocks != KB) return matrix_test<KIND, KB - 1>(blocks, nw, limbs, base, lds);
        if constexpr (KIND == KIND_FERMAT2)
            return mf::fermat2<KB>(nw, limbs, lds, threadIdx.x);
        else
            return mf::sprp<KB>(nw, limbs, base, lds, threadIdx.x);
    }
    return 0;
}
template <int KIND>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
mixed_mf_kernel(const uint32_t *__restrict__ words, const uint64_t *__restrict__ offset,
                const uint32_t *__restrict__ limbs, const uint32_t *__restrict__ order, MixedEnds ends, uint32_t first,
                uint32_t base, uint8_t *__restrict__ out) {
    __shared__ __align__(16) uint32_t lds[mf::buf_words(kMixedContainers)];
    const uint32_t i = first + blockIdx.x;
    int blocks = 1;
#pragma unroll
    for (int k = 1; k < kMixedContainers; ++k) blocks += i < ends.end[k];
    const uint32_t item = order[i];
    const uint32_t v =
        matrix_test<KIND, kMixedContainers>(blocks, words + offset[item], limbs[item], base, lds);
    if (threadIdx.x == 0) out[item] = (uint8_t)v;
}

// Launches the persistent kernel (mixed_fermat.hip, mixed_sprp.hip) or the
// matrix-core one (mixed_mf_fermat.hip, mixed_mf_sprp.hip) of one test kind,
// four units that compile in parallel.
struct MixedLaunch {
    const uint32_t *words;
    const uint64_t *offset;
    const uint32_t *limbs;
    const uint32_t *order;
    const uint8_t *tile_bucket;
    uint32_t ntiles;
    uint32_t *next_tile;
    Bases bases;
    uint8_t *out;
};
hipError_t launch_mixed_fermat(const MixedLaunch &a, int device, hipStream_t stream);
hipError_t launch_mixed_sprp(const MixedLaunch &a, int device, hipStream_t stream);
hipError_t launch_mixed_mf_fermat(const MixedLaunch &a, const MixedEnds &ends, hipStream_t stream);
hipError_t launch_mixed_mf_sprp(const MixedLaunch &a, const MixedEnds &ends, hipStream_t stream);

// The kernel is scheduled for two wavefronts per SIMD, which pays when every
// SIMD works through several tiles (2^19 numbers, 8192 tiles: 160.8 ms against
// 182.4 ms for the one-wave build).  With few tiles the dispatcher may place
// the first (widest) tiles two to a SIMD while other SIMDs idle (163840
// numbers, 2560 tiles: 86.5 ms against 53.1 ms), so below two tiles per
// wave slot at two waves the launch reserves enough LDS to hold one workgroup
// (one wave per SIMD) per CU.
constexpr uint32_t kMixedTilesPerCuTwoWaves = 16;
constexpr size_t kMixedOneWaveLds = 96 * 1024;  // > 160 KiB / 2: one workgroup per CU

template <int KIND>
hipError_t launch_mixed(const MixedLaunch &a, int device, hipStream_t stream) {
    int per_cu = 0, cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0)
        cus = 256;
    const bool two_waves = a.ntiles >= (uint32_t)cus * kMixedTilesPerCuTwoWaves;
    const size_t lds = two_waves ? kMixedParkBytes : std::max(kMixedParkBytes, kMixedOneWaveLds);
    (void)hipFuncSetAttribute((const void *)mixed_kernel<KIND>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, mixed_kernel<KIND>, 256, lds) != hipSuccess ||
        per_cu <= 0)
        per_cu = 1;
    const uint32_t grid = (uint32_t)std::min<size_t>((size_t)per_cu * cus, ((size_t)a.ntiles + 3) / 4);
    hipLaunchKernelGGL(mixed_kernel<KIND>, dim3(std::max(grid, 1u)), dim3(256), lds, stream, a.words, a.offset,
                       a.limbs, a.order, a.tile_bucket, a.ntiles, a.next_tile, a.bases, a.out);
    return hipGetLastError();
}

// a.order lists the matrix-core items, ends.end[0] of them.
template <int KIND>
hipError_t launch_mixed_mf(const MixedLaunch &a, const MixedEnds &ends, hipStream_t stream) {
    for (uint32_t first = 0, blocks; first < ends.end[0]; first += blocks) {
        blocks = matrix_blocks(ends.end[0] - first);
        hipLaunchKernelGGL(mixed_mf_kernel<KIND>, dim3(blocks), dim3(64), 0, stream, a.words, a.offset, a.limbs,
                           a.order, ends, first, a.bases.b[0], a.out);
        const hipError_t he = hipGetLastError();
        if (he != hipSuccess) return he;
    }
    return hipSuccess;
}

}  // namespace pgap
