// prp_mf_impl.h -- batch and scan kernels of the matrix-core tests, one
// number per wavefront (prp_mf.h); included by the prp_mf_*.hip units.
//
// One wavefront per workgroup: a small batch spreads over as many compute
// units as it has numbers.  A test costs the latency of its squarings, about
// 1090 cycles each at 1108 bits and 1660 at 2128 (a one-lane wavefront takes
// 12 and 43 thousand for its 64 numbers), until every SIMD has two wavefronts.
#pragma once
#include <algorithm>
#include "kernels.h"
#include "lucas_mf.h"

namespace pgap {

// Workgroups of a launch whose count only the device knows: two rounds of
// the wavefronts the widest width keeps resident (2 per SIMD).
constexpr uint32_t kMatrixBlocks = 4096;

template <int KB, int KIND>
__device__ __forceinline__ uint32_t prp_mf_test(const uint32_t *__restrict__ nw, uint32_t limbs, uint32_t base,
                                                uint32_t *lds) {
    if constexpr (KIND == KIND_FERMAT2)
        return mf::fermat2<KB>(nw, limbs, lds, threadIdx.x);
    else
        return mf::sprp<KB>(nw, limbs, base, lds, threadIdx.x);
}

// Wavefronts per SIMD to schedule for: the narrow widths reach four without
// spills (1108 bits: 4.34 ms for 16384 tests against 4.38 when asked for two, and
// 0.58 for one against 0.56; one, two and four blocks the same within 1%),
// the wide ones would spill (2128 bits: 36.0 against 30.8 ms).  Holding only the
// loaded fragments of N and N^-1 and spreading them at each use takes 36 to 56
// registers off, a wavefront more per SIMD, and is slower (16384 tests: 15.4 ->
// 17.8 ms at 2128 bits, 62 -> 69 at 4247): VALU issue bounds them, not waiting.
constexpr int mf_waves(int KB) { return KB <= 4 ? 4 : 2; }

template <int KB, int KIND>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(mf_waves(KB))))
prp_mf_kernel(const uint32_t *__restrict__ n, uint32_t limbs, uint32_t first, uint32_t count,
              const uint32_t *__restrict__ d_first, const uint32_t *__restrict__ d_count,
              const uint32_t *__restrict__ d_idx, uint32_t base, uint8_t *__restrict__ out) {
    __shared__ __align__(16) uint32_t lds[mf::buf_words(KB)];
    const uint32_t cnt = d_count ? min(*d_count, count) : count;
#pragma unroll 1
    for (uint32_t i = (d_first ? *d_first : first) + blockIdx.x; i < cnt; i += gridDim.x) {
        const uint32_t row = d_idx ? d_idx[i] : i;
        const uint32_t v = prp_mf_test<KB, KIND>(n + (size_t)row * limbs, limbs, base, lds);
        if (threadIdx.x == 0) out[row] = (uint8_t)v;
    }
}

template <int KB, int KIND>
hipError_t launch_mf(const uint32_t *d_n, uint32_t limbs, uint32_t first, uint32_t count, const uint32_t *d_first,
                     const uint32_t *d_count, const uint32_t *d_idx, uint32_t base, uint8_t *d_out,
                     hipStream_t stream) {
    if (first >= count) return hipSuccess;
    const uint32_t blocks = d_count ? std::min(count, kMatrixBlocks) : matrix_blocks(count - first);
    hipLaunchKernelGGL((prp_mf_kernel<KB, KIND>), dim3(blocks), dim3(64), 0, stream, d_n, limbs, first, count, d_first,
                       d_count, d_idx, base, d_out);
    return hipGetLastError();
}

// Streaming-scan round: strong Lucas items (the longest tests), strong-PRP
// confirmations, then Fermat items, in one grid.  On a stream of their own the
// Lucas tests overlap the grid only while the streams have hardware queues of
// their own: with two engines in a process they shared one, and every round of
// 1.9 to 5 ms (2128 bits) waited 2.75 ms for its Lucas batch.
template <int KB>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
scan_mf_kernel(const uint32_t *__restrict__ n, uint32_t limbs, uint32_t conf_rows, uint32_t conf_max,
               uint32_t max_items, const uint32_t *__restrict__ ctr, const uint8_t *__restrict__ base,
               uint8_t *__restrict__ out, const uint32_t *__restrict__ lnum, uint32_t nluc,
               uint8_t *__restrict__ lverd) {
    __shared__ __align__(16) uint32_t lds[mf::lucas_words(KB)];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63u;
    const uint32_t nc = min(ctr[3], conf_max), nf = min(ctr[0], max_items);
    // a Lucas test takes the workgroup, the others a wavefront each
    uint32_t i = blockIdx.x;
#pragma unroll 1
    for (; i < nluc; i += gridDim.x) {
        const uint32_t v = mf::strong_lucas<KB>(lnum + (size_t)i * limbs, limbs, lds, wave, lane);
        if (threadIdx.x == 0) lverd[i] = (uint8_t)v;
    }
    __syncthreads();
#pragma unroll 1
    for (uint32_t r = 2 * (i - nluc) + wave; r < nc + nf; r += 2 * gridDim.x) {
        const uint32_t row = r < nc ? r : conf_rows + (r - nc);
        const uint32_t *nw = n + (size_t)row * limbs;
        uint32_t *buf = lds + wave * mf::buf_words(KB);
        const uint32_t v = r < nc ? mf::sprp<KB>(nw, limbs, base[r], buf, lane) : mf::fermat2<KB>(nw, limbs, buf, lane);
        if (lane == 0) out[row] = (uint8_t)v;
    }
}

template <int KB>
hipError_t launch_scan_mf(const uint32_t *d_n, uint32_t limbs, uint32_t conf_rows, uint32_t conf_max,
                          uint32_t max_items, const uint32_t *d_ctr, const uint8_t *d_base, uint8_t *d_out,
                          const uint32_t *d_lnum, uint32_t nluc, uint8_t *d_lverd, hipStream_t stream) {
    const uint32_t blocks = std::min(nluc + (conf_max + max_items + 1) / 2, kMatrixBlocks / 2);
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((scan_mf_kernel<KB>), dim3(blocks), dim3(128), 0, stream, d_n, limbs, conf_rows, conf_max,
                       max_items, d_ctr, d_base, d_out, d_lnum, nluc, d_lverd);
    return hipGetLastError();
}

// Strong Lucas: a workgroup of two wavefronts per number.
template <int KB>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2)))
lucas_mf_kernel(const uint32_t *__restrict__ n, uint32_t limbs, uint32_t first, uint32_t count,
                const uint32_t *__restrict__ d_first, const uint32_t *__restrict__ d_count,
                const uint32_t *__restrict__ d_idx, uint8_t *__restrict__ out) {
    __shared__ __align__(16) uint32_t lds[mf::lucas_words(KB)];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63u;
    const uint32_t cnt = d_count ? min(*d_count, count) : count;
#pragma unroll 1
    for (uint32_t i = (d_first ? *d_first : first) + blockIdx.x; i < cnt; i += gridDim.x) {
        const uint32_t row = d_idx ? d_idx[i] : i;
        const uint32_t v = mf::strong_lucas<KB>(n + (size_t)row * limbs, limbs, lds, wave, lane);
        if (threadIdx.x == 0) out[row] = (uint8_t)v;
    }
}

template <int KB>
hipError_t launch_lucas_mf(const uint32_t *d_n, uint32_t limbs, uint32_t first, uint32_t count,
                           const uint32_t *d_first, const uint32_t *d_count, const uint32_t *d_idx, uint32_t,
                           uint8_t *d_out, hipStream_t stream) {
    if (first >= count) return hipSuccess;
    const uint32_t blocks = d_count ? std::min(count, kMatrixBlocks) : matrix_blocks(count - first);
    hipLaunchKernelGGL((lucas_mf_kernel<KB>), dim3(blocks), dim3(128), 0, stream, d_n, limbs, first, count, d_first,
                       d_count, d_idx, d_out);
    return hipGetLastError();
}

template <int... KBs>
struct RegisterLucasMF {
    RegisterLucasMF() {
        (register_matrix(MatrixVariant{KBs, KIND_LUCAS, mf::max_bits(KBs), &launch_lucas_mf<KBs>}), ...);
    }
};

template <int... KBs>
struct RegisterMF {
    RegisterMF() {
        (register_matrix(MatrixVariant{KBs, KIND_FERMAT2, mf::max_bits(KBs), &launch_mf<KBs, KIND_FERMAT2>}), ...);
        (register_matrix(MatrixVariant{KBs, KIND_SPRP, mf::max_bits(KBs), &launch_mf<KBs, KIND_SPRP>,
                                       &launch_scan_mf<KBs>}),
         ...);
    }
};

}  // namespace pgap
