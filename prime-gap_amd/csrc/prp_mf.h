// prp_mf.h -- Fermat base 2 and strong-PRP tests with one number per
// wavefront on the matrix cores (mont_mf.h).  Same definitions as prp28.h.
#pragma once
#include "mont_mf.h"

namespace pgap {
namespace mf {

// Words of N in lane order and its bit length; false for N even or below 2.
template <int KB>
__device__ __forceinline__ bool load_n(const uint32_t *__restrict__ nw, uint32_t limbs, uint32_t lane,
                                       uint32_t (&n)[Wave<KB>::T], uint32_t *bits) {
    uint32_t b = 0;
#pragma unroll
    for (int q = 0; q < Wave<KB>::T; ++q) {
        const uint32_t w = 64 * q + lane;
        n[q] = w < limbs && w < (uint32_t)Wave<KB>::LW ? nw[w] : 0u;
        const uint64_t nz = __ballot(n[q] != 0);
        if (nz) {
            const uint32_t top = 63u - (uint32_t)__builtin_clzll(nz);
            const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)n[q], (int)top);
            b = 32u * (64 * q + top) + 32u - (uint32_t)__builtin_clz(v);
        }
    }
    *bits = b;
    return b >= 2 && (__builtin_amdgcn_readfirstlane((int)n[0]) & 1);
}

// Fermat base 2: 2^(N-1) = 1 mod N.  The top bit of N - 1 is consumed by
// starting at 2; each further bit is a squaring, doubled when the bit is set.
template <int KB>
__device__ __forceinline__ uint32_t fermat2(const uint32_t *__restrict__ nw, uint32_t limbs, uint32_t *lds,
                                            uint32_t lane) {
    Wave<KB> w;
    uint32_t n[Wave<KB>::T], p[Wave<KB>::T], b;
    if (!load_n<KB>(nw, limbs, lane, n, &b)) return 0;
    w.init(lds, lane);
    w.setup(n, b, p);
    w.scale(n, b, 2, p);
    uint32_t ew = nw[(b - 2) >> 5];
#pragma unroll 1
    for (int i = (int)b - 2; i >= 0; --i) {
        const int32_t mult = i > 0 && ((ew >> (i & 31)) & 1u) ? 2 : 1;
        if ((i & 31) == 0 && i > 0) ew = nw[(i >> 5) - 1];
        w.square(mult, BIAS, p);
    }
    return w.classify() == 1u ? 1u : 0u;
}

// Strong probable prime test to a base below 64 (as r28::sprp).
template <int KB>
__device__ __forceinline__ uint32_t sprp(const uint32_t *__restrict__ nw, uint32_t limbs, uint32_t base, uint32_t *lds,
                                         uint32_t lane) {
    Wave<KB> w;
    uint32_t n[Wave<KB>::T], p[Wave<KB>::T], b;
    if (!load_n<KB>(nw, limbs, lane, n, &b)) return 0;
    int tz = 1;
    while (((nw[tz >> 5] >> (tz & 31)) & 1u) == 0) ++tz;
    uint32_t bb = base;
    if (b <= 32) bb = base % nw[0];
    if (bb == 0) return 0;  // x = 0 is never +-1
    w.init(lds, lane);
    w.setup(n, b, p);
    w.scale(n, b, (int32_t)bb, p);
    const uint32_t bias = bb <= 2 ? BIAS : BIAS_WIDE;
    int i = (int)b - 2;
    uint32_t ew = i >= tz ? nw[i >> 5] : 0u;
    bool high = false;  // layout of p
#pragma unroll 1
    for (; i >= tz; --i) {
        const int32_t mult = ((ew >> (i & 31)) & 1u) ? (int32_t)bb : 1;
        if ((i & 31) == 0 && i > tz) ew = nw[(i >> 5) - 1];
        w.square(mult, bias, p);
        high = true;
    }
    const uint32_t k0 = w.classify();
    if (k0 == 1 || k0 == 2) return 1;
#pragma unroll 1
    for (int c = 1; c < tz; ++c) {
        if (high)
            w.store_high(p);
        else
            w.store_low(p);
        w.square(1, BIAS, p);
        high = true;
        const uint32_t k = w.classify();
        if (k == 2) return 1;
        if (k == 1) return 0;
    }
    return 0;
}

}  // namespace mf
}  // namespace pgap
