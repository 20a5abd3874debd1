// sieve.hip -- the unknown-file producer on the device: for every m of a
// batch, the offsets x in [-SL, SL] for which m*K + x has no prime factor
// <= max_prime.
//
// Reference counterpart: combined_sieve (combined_sieve.cpp:409-750 method1,
// :2014-2447 method2) and its writers (:1261-1445).  The reference sieves
// with primesieve on the host and finds, per prime, the m's it hits with a
// modular search (modulo_search.h:33-60); here every (prime, m) pair is
// evaluated directly on the GPU:
//   1. the primes <= max_prime come from a segmented sieve of Eratosthenes,
//      one 32 KiB LDS bitmap per workgroup, survivors appended unordered;
//   2. primes <= 2*SL + 1 ("small") mark a per-m LDS bitmap, one workgroup
//      per m; those that divide K hit the same offsets for every m and are
//      marked once per call;
//   3. larger primes hit each m's interval at most once: a thread per prime
//      loops over the batch's m's, tests for a hit in 64-bit fixed point and
//      sets one bit in the m's bitmap;
//   4. the survivors are listed in outward order on the device, and the lists
//      alone are copied back.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "engine_impl.h"

namespace pgap {

// a mod p for any a < 2^64 and p < 2^62, mu = floor((2^64 - 1) / p): the
// estimated quotient is short by at most 2.
__device__ __forceinline__ uint64_t mod_b(uint64_t a, uint64_t p, uint64_t mu) {
    const uint64_t q = __umul64hi(a, mu);
    uint64_t r = a - q * p;
    r = r >= p ? r - p : r;
    return r >= p ? r - p : r;
}

// a * b mod p for a, b < p.  Below 2^32 the product fits 64 bits; above
// (p < 2^40), product = hi * 2^64 + lo with hi < 2^16, and 2^64 mod p = c64.
__device__ __forceinline__ uint64_t mulmod_b(uint64_t a, uint64_t b, uint64_t p, uint64_t mu, uint64_t c64) {
    if (p < (1ull << 32)) return mod_b(a * b, p, mu);
    const uint64_t lo = a * b, hi = __umul64hi(a, b);
    return mod_b(mod_b(lo, p, mu) + mod_b(hi * c64, p, mu), p, mu);
}

constexpr uint32_t SEG_WORDS = 8192;              // 32 KiB of LDS
constexpr uint32_t SEG_BITS = SEG_WORDS * 32;     // odd numbers per segment

// Odd primes in [3, limit]: workgroup b covers odd n = 2k+1, k in
// [b*SEG_BITS, (b+1)*SEG_BITS).
__global__ void __launch_bounds__(256) segment_primes_kernel(const uint32_t *__restrict__ small, uint32_t nsmall,
                                                             uint64_t limit, uint64_t *__restrict__ out,
                                                             uint32_t *__restrict__ count, uint32_t cap) {
    __shared__ uint32_t bits[SEG_WORDS];
    for (uint32_t i = threadIdx.x; i < SEG_WORDS; i += 256) bits[i] = 0;
    __syncthreads();
    const uint64_t k0 = (uint64_t)blockIdx.x * SEG_BITS;
    const uint64_t lo = 2 * k0 + 1, hi = 2 * (k0 + SEG_BITS) + 1;  // odd numbers in [lo, hi)
    for (uint32_t s = threadIdx.x; s < nsmall; s += 256) {
        const uint64_t p = small[s];
        uint64_t start = p * p;
        if (start < lo) start = ((lo + p - 1) / p) * p;
        if ((start & 1) == 0) start += p;
        for (uint64_t n = start; n < hi; n += 2 * p) {
            const uint32_t k = (uint32_t)((n - 1) / 2 - k0);
            atomicOr(&bits[k >> 5], 1u << (k & 31));
        }
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < SEG_WORDS; w += 256) {
        uint32_t free_bits = ~bits[w];
        const uint64_t kw = k0 + 32ull * w;
        if (kw == 0) free_bits &= ~1u;  // n = 1
        // n = 2k+1 <= limit  <=>  k <= (limit-1)/2
        const uint64_t kmax = (limit - 1) / 2;
        if (kw > kmax) free_bits = 0;
        else if (kw + 31 > kmax) free_bits &= (uint32_t)((1ull << (kmax - kw + 1)) - 1);
        const uint32_t cnt = (uint32_t)__popc(free_bits);
        if (!cnt) continue;
        uint32_t base = atomicAdd(count, cnt);
        while (free_bits) {
            const uint32_t b = (uint32_t)__ffs(free_bits) - 1;
            free_bits &= free_bits - 1;
            if (base < cap) out[base] = 2 * (kw + b) + 1;
            ++base;
        }
    }
}

__global__ void mu_kernel(const uint64_t *__restrict__ p, size_t n, uint64_t *__restrict__ mu) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) mu[i] = ~0ull / p[i];
}

// K mod p, 16 bits at a time so that r * 2^16 + digit stays below 2^64 for
// p < 2^48.
__global__ void kmod_barrett_kernel(const uint32_t *__restrict__ K, uint32_t nk, const uint64_t *__restrict__ primes,
                                    const uint64_t *__restrict__ mu, size_t np, uint64_t *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= np) return;
    const uint64_t p = primes[i], u = mu[i];
    uint64_t r = 0;
    for (int j = (int)nk - 1; j >= 0; --j) {
        r = mod_b((r << 16) | (K[j] >> 16), p, u);
        r = mod_b((r << 16) | (K[j] & 0xffffu), p, u);
    }
    out[i] = r;
}

__global__ void kmod_small_kernel(const uint32_t *__restrict__ K, uint32_t nk, const uint32_t *__restrict__ primes,
                                  const uint64_t *__restrict__ mu, uint32_t np, uint32_t *__restrict__ out) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= np) return;
    const uint64_t p = primes[i], u = mu[i];
    uint64_t r = 0;
    for (int j = (int)nk - 1; j >= 0; --j) r = mod_b((r << 32) | K[j], p, u);
    out[i] = (uint32_t)r;
}

// Offsets hit by the primes that divide K (m*K mod p = 0 for every m), one
// workgroup per SMALL_SEG words of the bitmap, a wavefront per prime.
constexpr uint32_t SMALL_SEG = 1024;
__global__ void __launch_bounds__(256) sieve_base_kernel(uint32_t SL, const uint32_t *__restrict__ primes,
                                                         const uint32_t *__restrict__ kmod, uint32_t np,
                                                         uint32_t words, uint32_t *__restrict__ base) {
    __shared__ uint32_t bm[SMALL_SEG];
    for (uint32_t i = threadIdx.x; i < SMALL_SEG; i += 256) bm[i] = 0;
    __syncthreads();
    const uint32_t lo = blockIdx.x * SMALL_SEG * 32u, hi = min(lo + SMALL_SEG * 32u, 2 * SL + 1);
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t s0 = threadIdx.x & ~63u; s0 < np; s0 += 256) {
        // 64 primes at a time; the few that divide K one after the other
        const uint32_t s = s0 + lane;
        const uint32_t mine = s < np ? primes[s] : 0u;
        for (uint64_t divide = __ballot(s < np && kmod[s] == 0); divide; divide &= divide - 1) {
            const uint32_t p = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)__builtin_ctzll(divide));
            // indexes SL mod p, ... from lo on
            const uint32_t first = lo + (SL % p + p - lo % p) % p;
            for (uint64_t i = first + (uint64_t)p * lane; i < hi; i += 64ull * p)
                atomicOr(&bm[(i - lo) >> 5], 1u << (i & 31));
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < SMALL_SEG; i += 256)
        if (blockIdx.x * SMALL_SEG + i < words) base[blockIdx.x * SMALL_SEG + i] = bm[i];
}

// One workgroup per m: the other primes <= 2SL+1 mark the m's bitmap in LDS,
// a wavefront per prime for the first nwave of them (below 4096, hundreds of
// multiples each), a thread per prime for the rest.  Bound by LDS atomics; with
// a thread per prime throughout, the thread of p = 2 walked its SL multiples
// alone: 200 m's of 1511# at SL = 40000 took 1.70 ms, now 0.053 (and 0.042 for
// the base bitmap).
__global__ void __launch_bounds__(1024) sieve_small_kernel(const uint64_t *__restrict__ m, uint32_t SL,
                                                           const uint32_t *__restrict__ primes,
                                                           const uint32_t *__restrict__ kmod,
                                                           const uint64_t *__restrict__ mu, uint32_t np,
                                                           uint32_t nwave, uint32_t words,
                                                           const uint32_t *__restrict__ base,
                                                           uint32_t *__restrict__ bitmap) {
    extern __shared__ uint32_t bm[];
    for (uint32_t i = threadIdx.x; i < words; i += 1024) bm[i] = base[i];
    __syncthreads();
    const uint64_t mi = m[blockIdx.x];
    const uint32_t W = 2 * SL + 1;
    const auto first = [&](uint32_t s) {
        const uint64_t p = primes[s], u = mu[s];
        const uint64_t r = mod_b(mod_b(mi, p, u) * kmod[s], p, u);  // m*K mod p
        // index i = SL + x with x = -r mod p
        const uint64_t a = mod_b(SL, p, u);
        return (uint32_t)(a >= r ? a - r : a + p - r);
    };
    for (uint32_t s = threadIdx.x >> 6; s < nwave; s += 16) {
        if (kmod[s] == 0) continue;
        const uint32_t p = primes[s];
        for (uint64_t i = first(s) + (uint64_t)p * (threadIdx.x & 63u); i < W; i += 64ull * p)
            atomicOr(&bm[i >> 5], 1u << (i & 31));
    }
    for (uint32_t s = nwave + threadIdx.x; s < np; s += 1024) {
        if (kmod[s] == 0) continue;
        const uint32_t p = primes[s];
        for (uint32_t i = first(s); i < W; i += p) atomicOr(&bm[i >> 5], 1u << (i & 31));
    }
    __syncthreads();
    uint32_t *o = bitmap + (size_t)blockIdx.x * words;
    for (uint32_t i = threadIdx.x; i < words; i += 1024) o[i] = bm[i];
}

// Primes > 2SL+1 (the rest of the table) hit each interval at most once: the
// offset -m*K mod p falls inside when (m*K + SL) mod p <= 2 SL.
//
// FIXED: phi = 2^64 (K mod p) / p to within two units, so v = m phi + SL 2^64 / p
// mod 2^64 is t 2^64 / p to within margin = 2 m + SL + 8 units, t = (m*K + SL)
// mod p: a pair is a hit only if the high word of v + margin is below that of
// 2 SL 2^64 / p + 2 margin, two multiply-adds and a compare per pair instead
// of two 64-bit Barrett reductions, and t = round(v p / 2^64) is exact while
// 4 margin p < 2^63 (the caller asks for 2^62 over the batch's largest m: m < 2.8
// 10^7 to 2 10^10; other batches take the exact route).  Eight m's
// share a branch and a scalar load of the m's.  Bound by the multiply-add rate:
// 200 m's of 1511# to 1e9 (10^10 pairs) take 1.19 ms against 14.0 with a Barrett
// pair each, 8.5 10^12 pairs/s; 4096 m's 23 ms against 276.
template <bool FIXED>
__global__ void __launch_bounds__(256) sieve_large_kernel(const uint64_t *__restrict__ m, const uint32_t *__restrict__ m32,
                                                          uint32_t nm, uint64_t m_max,
                                                          uint32_t SL, const uint64_t *__restrict__ primes,
                                                          const uint64_t *__restrict__ kmod,
                                                          const uint64_t *__restrict__ mu, size_t np,
                                                          uint32_t words, uint32_t *__restrict__ bitmap) {
    const uint32_t W = 2 * SL + 1;
    for (size_t s = (size_t)blockIdx.x * 256 + threadIdx.x; s < np; s += (size_t)gridDim.x * 256) {
        const uint64_t p = primes[s];
        if (p <= W) continue;  // handled by sieve_small_kernel
        const uint64_t u = mu[s], kp = kmod[s];
        const auto mark = [&](uint32_t j, uint64_t i) {
            if (i < W) atomicOr(&bitmap[(size_t)j * words + (i >> 5)], 1u << (i & 31));
        };
        if constexpr (FIXED) {
            // 2^64 = u p + c, 0 < c <= p: phi = kp u + kp c / p
            const uint64_t c = 0 - u * p;
            const uint64_t phi = kp * u + (uint64_t)((double)kp * (double)c / (double)p);
            const uint64_t margin = 2 * m_max + SL + 8;
            const uint64_t off = SL * u + margin;
            const uint32_t top = (uint32_t)((2 * SL * u + 2 * SL + 2 * margin) >> 32);
            const uint64_t half = (u >> 1) - margin;  // rounds t
            const uint32_t plo = (uint32_t)phi, phi_hi = (uint32_t)(phi >> 32);
            // v's words; the high one without the 64-bit multiply that adding
            // the two products in 64 bits would become
            const auto low = [&](uint32_t mj) { return (uint64_t)mj * plo + off; };
            const auto hit = [&](uint32_t j, uint32_t v_hi, uint32_t v_lo) {
                if (v_hi <= top) mark(j, 2 * SL - __umul64hi((((uint64_t)v_hi << 32) | v_lo) + half, p));
            };
            uint32_t j = 0;
            for (; j + 8 <= nm; j += 8) {
                uint32_t v_hi[8], v_lo[8], least = ~0u;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const uint64_t lo = low(m32[j + k]);
                    v_lo[k] = (uint32_t)lo;
                    v_hi[k] = (uint32_t)(lo >> 32) + m32[j + k] * phi_hi;
                    least = min(least, v_hi[k]);
                }
                if (least > top) continue;
#pragma unroll
                for (int k = 0; k < 8; ++k) hit(j + k, v_hi[k], v_lo[k]);
            }
            for (; j < nm; ++j) {
                const uint64_t lo = low(m32[j]);
                hit(j, (uint32_t)(lo >> 32) + m32[j] * phi_hi, (uint32_t)lo);
            }
        } else {
            uint64_t c64 = mod_b(~0ull, p, u) + 1;  // 2^64 mod p
            if (c64 == p) c64 = 0;
            for (uint32_t j = 0; j < nm; ++j) {
                const uint64_t r = mulmod_b(mod_b(m[j], p, u), kp, p, u, c64);
                mark(j, r <= SL ? SL - r : SL + p - r);
            }
        }
    }
}

// 32 distances of one side of a bitmap, nearest first: bit k is distance 32 t
// + 1 + k, set when it survives.
__device__ __forceinline__ uint32_t side_word(const uint32_t *__restrict__ bm, uint32_t words, uint32_t SL,
                                              uint32_t side, uint32_t t) {
    const int64_t lo = side ? (int64_t)SL + 1 + 32ll * t : (int64_t)SL - 32 - 32ll * t;  // lowest index
    const int64_t w = lo >> 5;  // below 0 for the last word of the prev side
    const uint32_t sh = (uint32_t)lo & 31u;
    const uint64_t a = w >= 0 && w < (int64_t)words ? bm[w] : 0u;
    const uint64_t b = w + 1 >= 0 && w + 1 < (int64_t)words ? bm[w + 1] : 0u;
    const uint32_t bits = (uint32_t)((a | (b << 32)) >> sh);
    const uint32_t left = SL - 32 * t;  // distances in range
    return (side ? ~bits : __brev(~bits)) & (left >= 32 ? ~0u : (1u << left) - 1);
}

// Survivors of every (m, side): workgroup 2 i + side.
__global__ void __launch_bounds__(256) sieve_count_kernel(const uint32_t *__restrict__ bitmap, uint32_t words,
                                                          uint32_t SL, uint32_t *__restrict__ counts) {
    __shared__ uint32_t part[4];
    const uint32_t *bm = bitmap + (size_t)(blockIdx.x >> 1) * words;
    uint32_t n = 0;
    for (uint32_t t = threadIdx.x; 32 * t < SL; t += 256)
        n += (uint32_t)__popc(side_word(bm, words, SL, blockIdx.x & 1u, t));
    for (int off = 32; off > 0; off >>= 1) n += (uint32_t)__shfl_xor((int)n, off, 64);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// Their distances, each list at offsets[workgroup] of out, or at workgroup * SL
// with its length in counts where there are no offsets: a workgroup takes 256
// words of its side at a time, scans their counts and scatters.
__global__ void __launch_bounds__(256) sieve_list_kernel(const uint32_t *__restrict__ bitmap, uint32_t words,
                                                         uint32_t SL, const uint32_t *__restrict__ offsets,
                                                         uint32_t *__restrict__ counts, int32_t *__restrict__ out) {
    __shared__ uint32_t part[4];
    const uint32_t *bm = bitmap + (size_t)(blockIdx.x >> 1) * words;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t start = offsets ? offsets[blockIdx.x] : blockIdx.x * SL;
    uint32_t done = start;
    for (uint32_t t0 = 0; 32 * t0 < SL; t0 += 256) {
        const uint32_t t = t0 + threadIdx.x;
        uint32_t w = 32 * t < SL ? side_word(bm, words, SL, blockIdx.x & 1u, t) : 0u;
        const uint32_t n = (uint32_t)__popc(w);
        uint32_t before = n;  // inclusive scan over the wavefront
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)before, off, 64);
            if (lane >= (uint32_t)off) before += o;
        }
        if (lane == 63) part[wave] = before;
        __syncthreads();
        uint32_t at = done + before - n;
        for (uint32_t k = 0; k < wave; ++k) at += part[k];
        done += part[0] + part[1] + part[2] + part[3];
        __syncthreads();
        while (w) {
            out[at++] = (int32_t)(32 * t + (uint32_t)__ffs(w));
            w &= w - 1;
        }
    }
    if (!offsets && threadIdx.x == 0) counts[blockIdx.x] = done - start;
}

}  // namespace pgap

using namespace pgap;

static void free_small(Family &f) {
    if (f.d_small) (void)hipFree(f.d_small);
    f.d_small = nullptr;
    f.small_limit = 0;
}

// Distances a call copies back at a time: the pinned staging buffer, which
// the engine keeps until it is destroyed (at least one m's 2 * 200000 fit).  It
// does not depend on the limit: freed with the prime tables at each change of it,
// two calls of 4 m's to 1e8 and 1e7 in turn took 12.1 ms.
constexpr size_t STAGE_WORDS = (size_t)8 << 20;
// Up to so many words of full lists, a batch's lists come back at their full
// length with their counts: one wait instead of a count kernel, a wait for the
// lengths and an upload of the places.  Whole calls, us, that way against the
// other: 200 words (one m, SL = 100, to 1000) 38 / 65, 32000 78 / 95, 128000 95 /
// 102, 160000 188 / 204, 480000 215 / 210, 1024000 245 / 200.
constexpr size_t DIRECT_WORDS = (size_t)1 << 18;

void pgap_engine::sieve_shutdown() {
    if (sieve_primes) (void)hipFree(sieve_primes);
    if (sieve_mu) (void)hipFree(sieve_mu);
    sieve_primes = nullptr;
    sieve_mu = nullptr;
    sieve_nprimes = 0;
    sieve_limit = 0;
    for (Family &f : families) {
        if (f.d_skmod) (void)hipFree(f.d_skmod);
        f.d_skmod = nullptr;
        f.skmod_limit = 0;
        free_small(f);
    }
}

static pgap_status sieve_tables(pgap_engine *e, Family &f, uint64_t limit) {
    hipError_t he;
    if (e->sieve_limit != limit) {
        e->sieve_shutdown();
        const uint64_t root = (uint64_t)std::sqrt((double)limit) + 2;
        std::vector<uint32_t> small;
        for (uint32_t p : primes_upto((uint32_t)root))
            if (p > 2) small.push_back(p);
        const double lg = std::log((double)std::max<uint64_t>(limit, 17));
        const uint32_t cap = (uint32_t)(1.26 * (double)limit / lg) + 64;
        uint32_t *d_small = nullptr, *d_count = nullptr;
        if ((he = hipMalloc(&e->sieve_primes, (size_t)cap * 8)) != hipSuccess ||
            (he = hipMalloc(&e->sieve_mu, (size_t)cap * 8)) != hipSuccess ||
            (he = hipMalloc(&d_small, std::max<size_t>(small.size(), 1) * 4)) != hipSuccess ||
            (he = hipMalloc(&d_count, 4)) != hipSuccess) {
            (void)hipGetLastError();
            if (d_small) (void)hipFree(d_small);
            e->sieve_shutdown();
            e->set_error("pgap_sieve: hipMalloc for primes <= %llu: %s", (unsigned long long)limit,
                         hipGetErrorString(he));
            return PGAP_E_OOM;
        }
        const uint64_t two = 2;
        const uint32_t one = 1;
        (void)hipMemcpyAsync(e->sieve_primes, &two, 8, hipMemcpyHostToDevice, e->stream);
        (void)hipMemcpyAsync(d_count, &one, 4, hipMemcpyHostToDevice, e->stream);
        (void)hipMemcpyAsync(d_small, small.data(), small.size() * 4, hipMemcpyHostToDevice, e->stream);
        const uint64_t nseg = ((limit - 1) / 2 + SEG_BITS) / SEG_BITS;
        hipLaunchKernelGGL(segment_primes_kernel, dim3((uint32_t)nseg), dim3(256), 0, e->stream, d_small,
                           (uint32_t)small.size(), limit, e->sieve_primes, d_count, cap);
        uint32_t n = 0;
        he = hipGetLastError();
        if (he == hipSuccess) he = hipMemcpyAsync(&n, d_count, 4, hipMemcpyDeviceToHost, e->stream);
        if (he == hipSuccess) he = hipStreamSynchronize(e->stream);
        (void)hipFree(d_small);
        (void)hipFree(d_count);
        if (he != hipSuccess) {
            e->sieve_shutdown();
            return e->hip_fail(he, "prime generation");
        }
        if (n > cap) {
            e->sieve_shutdown();
            e->set_error("pgap_sieve: prime table overflow (%u > %u)", n, cap);
            return PGAP_E_STATE;
        }
        hipLaunchKernelGGL(mu_kernel, dim3((n + 255) / 256), dim3(256), 0, e->stream, e->sieve_primes, (size_t)n,
                           e->sieve_mu);
        if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "mu kernel");
        e->sieve_nprimes = n;
        e->sieve_limit = limit;
    }
    if (f.skmod_limit != limit) {
        if (f.d_skmod) (void)hipFree(f.d_skmod);
        f.d_skmod = nullptr;
        if ((he = hipMalloc(&f.d_skmod, std::max<size_t>(e->sieve_nprimes, 1) * 8)) != hipSuccess) {
            (void)hipGetLastError();
            e->set_error("pgap_sieve: hipMalloc K mod p: %s", hipGetErrorString(he));
            return PGAP_E_OOM;
        }
        hipLaunchKernelGGL(kmod_barrett_kernel, dim3((uint32_t)((e->sieve_nprimes + 255) / 256)), dim3(256), 0,
                           e->stream, f.d_K, (uint32_t)f.K.size(), e->sieve_primes, e->sieve_mu, e->sieve_nprimes,
                           f.d_skmod);
        if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "kmod kernel");
        f.skmod_limit = limit;
    }
    const uint64_t W = 2ull * f.SL + 1;
    if (f.small_limit != std::min(W, limit)) {
        // primes <= 2SL+1: Barrett constants, the primes, K mod p
        free_small(f);
        const uint32_t top = (uint32_t)std::min(W, limit);
        const std::vector<uint32_t> sp = primes_upto(top);
        const size_t n = sp.size();
        std::vector<uint64_t> mu(n);
        for (size_t i = 0; i < n; ++i) mu[i] = ~0ull / sp[i];
        if ((he = hipMalloc(&f.d_small, std::max<size_t>(n, 1) * 16)) != hipSuccess) {
            (void)hipGetLastError();
            f.d_small = nullptr;
            e->set_error("pgap_sieve: hipMalloc small primes: %s", hipGetErrorString(he));
            return PGAP_E_OOM;
        }
        uint32_t *primes = (uint32_t *)(f.d_small + n);
        if ((he = hipMemcpyAsync(f.d_small, mu.data(), n * 8, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
            (he = hipMemcpyAsync(primes, sp.data(), n * 4, hipMemcpyHostToDevice, e->stream)) != hipSuccess) {
            free_small(f);
            return e->hip_fail(he, "small primes");
        }
        hipLaunchKernelGGL(kmod_small_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, e->stream, f.d_K,
                           (uint32_t)f.K.size(), primes, f.d_small, (uint32_t)n, primes + n);
        if ((he = hipGetLastError()) != hipSuccess || (he = hipStreamSynchronize(e->stream)) != hipSuccess) {
            free_small(f);
            return e->hip_fail(he, "small K mod p");
        }
        f.nsmall = (uint32_t)n;
        f.nsmall_wave = (uint32_t)(std::lower_bound(sp.begin(), sp.end(), 4096u) - sp.begin());
        f.small_limit = top;
    }
    return PGAP_OK;
}

extern "C" pgap_status pgap_sieve(pgap_engine *e, int family, const uint64_t *m, size_t count, uint64_t max_prime,
                                  int32_t *prev, uint32_t *n_prev, int32_t *next, uint32_t *n_next) {
    if (!e) return PGAP_E_ARG;
    if (!e->ready) return PGAP_E_STATE;
    Family *f = e->family(family);
    if (!f || (count && (!m || !prev || !n_prev || !next || !n_next)) || max_prime < 2 ||
        max_prime > 20000000000ull) {
        e->set_error("pgap_sieve: bad arguments (max_prime in [2, 2e10])");
        return PGAP_E_ARG;
    }
    const uint32_t SL = f->SL;
    if (SL == 0 || SL > 200000) {
        e->set_error("pgap_sieve: family sieve length %u outside [1, 200000]", SL);
        return PGAP_E_ARG;
    }
    if (count == 0) return PGAP_OK;
    (void)hipSetDevice(e->opt.device);
    pgap_status st;
    if ((st = sieve_tables(e, *f, max_prime))) return st;

    const uint32_t W = 2 * SL + 1, words = (W + 31) / 32;
    const uint32_t *sp = (const uint32_t *)(f->d_small + f->nsmall), *skm = sp + f->nsmall;
    const size_t batch = std::min<size_t>(count, 4096);
    DevBuf &bm = e->d_n;  // reuse the batch buffers: bitmaps, the base bitmap behind them
    if ((st = e->ensure(bm, (batch + 1) * words * 4, "sieve bitmaps")) ||
        (st = e->ensure(e->d_m, batch * 12, "m")) || (st = e->ensure(e->d_idx0, batch * 2 * 4, "list lengths")) ||
        (st = e->ensure(e->d_idx1, batch * 2 * 4, "list offsets")))
        return st;
    hipError_t he;
    if (!e->sieve_stage && (he = hipHostMalloc((void **)&e->sieve_stage, STAGE_WORDS * 4, 0)) != hipSuccess) {
        (void)hipGetLastError();
        e->sieve_stage = nullptr;
        e->set_error("pgap_sieve: hipHostMalloc staging: %s", hipGetErrorString(he));
        return PGAP_E_OOM;
    }
    uint32_t *base = (uint32_t *)bm.p + batch * words;
    hipLaunchKernelGGL(sieve_base_kernel, dim3((words + SMALL_SEG - 1) / SMALL_SEG), dim3(256), 0, e->stream, SL, sp,
                       skm, f->nsmall, words, base);
    if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "sieve base kernel");
    std::vector<uint32_t> len(2 * batch), at(2 * batch), up(3 * batch);  // up: the m's, then their low words
    uint32_t *d_m32 = (uint32_t *)((uint64_t *)e->d_m.p + batch);
    for (size_t off = 0; off < count; off += batch) {
        const uint32_t nb = (uint32_t)std::min(batch, count - off);
        uint64_t m_max = 0;
        for (uint32_t j = 0; j < nb; ++j) {
            m_max = std::max(m_max, m[off + j]);
            up[2 * batch + j] = (uint32_t)m[off + j];
        }
        memcpy(up.data(), m + off, nb * 8);
        if ((he = hipMemcpyAsync(e->d_m.p, up.data(), (2 * batch + nb) * 4, hipMemcpyHostToDevice, e->stream)) !=
            hipSuccess)
            return e->hip_fail(he, "sieve m upload");
        hipLaunchKernelGGL(sieve_small_kernel, dim3(nb), dim3(1024), words * 4, e->stream,
                           (const uint64_t *)e->d_m.p, SL, sp, skm, f->d_small, f->nsmall, f->nsmall_wave, words,
                           base, (uint32_t *)bm.p);
        if (e->sieve_nprimes > f->nsmall) {
            const uint32_t grid = (uint32_t)std::min<size_t>((e->sieve_nprimes + 255) / 256, 65536);
            // every m below 2^32 and 4 margin p < 2^63, see the kernel
            const bool fixed = m_max < (1ull << 32) && (double)(8 * m_max + 4 * SL + 32) * (double)max_prime < 0x1p62;
            const auto large = fixed ? &sieve_large_kernel<true> : &sieve_large_kernel<false>;
            hipLaunchKernelGGL(large, dim3(grid), dim3(256), 0, e->stream, (const uint64_t *)e->d_m.p, d_m32, nb, m_max, SL,
                               e->sieve_primes, f->d_skmod, e->sieve_mu, e->sieve_nprimes, words, (uint32_t *)bm.p);
        }
        if (const size_t full = (size_t)2 * nb * SL; full <= DIRECT_WORDS) {
            if ((st = e->ensure(e->d_x, (full + 2 * nb) * 4, "lists"))) return st;
            uint32_t *counts = (uint32_t *)e->d_x.p + full;
            hipLaunchKernelGGL(sieve_list_kernel, dim3(2 * nb), dim3(256), 0, e->stream, (const uint32_t *)bm.p, words,
                               SL, nullptr, counts, (int32_t *)e->d_x.p);
            if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "sieve kernels");
            if ((he = hipMemcpyAsync(e->sieve_stage, e->d_x.p, (full + 2 * nb) * 4, hipMemcpyDeviceToHost,
                                     e->stream)) != hipSuccess ||
                (he = hipStreamSynchronize(e->stream)) != hipSuccess)
                return e->hip_fail(he, "sieve readback");
            for (uint32_t j = 0; j < nb; ++j) {
                const size_t i = off + j;
                const uint32_t *list = e->sieve_stage + (size_t)2 * j * SL;
                n_prev[i] = e->sieve_stage[full + 2 * j];
                n_next[i] = e->sieve_stage[full + 2 * j + 1];
                memcpy(prev + i * SL, list, (size_t)n_prev[i] * 4);
                memcpy(next + i * SL, list + SL, (size_t)n_next[i] * 4);
            }
            continue;
        }
        hipLaunchKernelGGL(sieve_count_kernel, dim3(2 * nb), dim3(256), 0, e->stream, (const uint32_t *)bm.p, words,
                           SL, (uint32_t *)e->d_idx0.p);
        if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "sieve kernels");
        if ((he = hipMemcpyAsync(len.data(), e->d_idx0.p, nb * 2 * 4, hipMemcpyDeviceToHost, e->stream)) !=
                hipSuccess ||
            (he = hipStreamSynchronize(e->stream)) != hipSuccess)
            return e->hip_fail(he, "sieve counts");
        // lists of as many m's as the staging buffer holds
        for (uint32_t j0 = 0, j1 = 0; j0 < nb; j0 = j1) {
            size_t total = 0;
            while (j1 < nb && total + len[2 * j1] + len[2 * j1 + 1] <= STAGE_WORDS) {
                for (int side = 0; side < 2; ++side) {
                    at[2 * j1 + side] = (uint32_t)total;
                    total += len[2 * j1 + side];
                }
                ++j1;
            }
            if ((st = e->ensure(e->d_x, std::max<size_t>(total, 1) * 4, "lists"))) return st;
            if ((he = hipMemcpyAsync(e->d_idx1.p, at.data() + 2 * j0, (j1 - j0) * 2 * 4, hipMemcpyHostToDevice,
                                     e->stream)) != hipSuccess)
                return e->hip_fail(he, "sieve offsets");
            hipLaunchKernelGGL(sieve_list_kernel, dim3(2 * (j1 - j0)), dim3(256), 0, e->stream,
                               (const uint32_t *)bm.p + (size_t)j0 * words, words, SL,
                               (const uint32_t *)e->d_idx1.p, nullptr, (int32_t *)e->d_x.p);
            if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "sieve list kernel");
            if ((total && (he = hipMemcpyAsync(e->sieve_stage, e->d_x.p, total * 4, hipMemcpyDeviceToHost,
                                               e->stream)) != hipSuccess) ||
                (he = hipStreamSynchronize(e->stream)) != hipSuccess)
                return e->hip_fail(he, "sieve readback");
            for (uint32_t j = j0; j < j1; ++j) {
                const size_t i = off + j;
                n_prev[i] = len[2 * j];
                n_next[i] = len[2 * j + 1];
                memcpy(prev + i * SL, e->sieve_stage + at[2 * j], (size_t)n_prev[i] * 4);
                memcpy(next + i * SL, e->sieve_stage + at[2 * j + 1], (size_t)n_next[i] * 4);
            }
        }
    }
    return PGAP_OK;
}
