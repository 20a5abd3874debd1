// family.hip -- K = P#/d families and device-side candidate construction /
// trial-division screening of N = m*K + x.
//
// Reference counterparts: init_K / K_stats (gap_common.cpp:116-140) for K;
// the host batch fill mpz_mul_ui(center, K, m) + mpz_sub_ui/mpz_add_ui and
// from_mpz export (gap_test_gpu.cu:418-476, miller_rabin.h:37-52) for the
// construction; the per-prime offset test of combined_sieve for screening.
#include <algorithm>
#include <cstring>

#include "engine_impl.h"

namespace pgap {

// a mod p with mu = floor((2^64-1)/p): the quotient estimate is at most 2
// short, so two conditional subtractions finish it.
__device__ __forceinline__ uint64_t mod_barrett(uint64_t a, uint64_t p, uint64_t mu) {
    const uint64_t q = __umul64hi(a, mu);
    uint64_t r = a - q * p;
    r = r >= p ? r - p : r;
    return r >= p ? r - p : r;
}

// The trial-division test of N = m*K + x by p in 64-bit fixed point, for m <
// 2^32 and |x| < 2^31: with phi = 2^64 (K mod p) / p to within two units and mu
// = 2^64 / p to within one, m phi + x mu mod 2^64 is 2^64 (N mod p) / p to within
// 2 m + |x| < 2^34 units.  So p can divide N only if that, plus the margin 2^34,
// has a high word of at most 8: four multiply-adds and a compare instead of
// three 64-bit Barrett reductions.  For p < 2^28 that is exact: the next
// residue lies 2^64 / p >= 2^36 units away.  Larger primes pass by chance (9 in
// 2^32) and the exact residue decides.  off holds the margin less 2^31 mu, so
// that x + 2^31 enters as an unsigned word.
constexpr uint64_t kMargin = 1ull << 34;
constexpr uint32_t kMarginTop = 8;
constexpr uint32_t kFixedExact = 1u << 28;

__global__ void filter_table_kernel(const uint32_t *__restrict__ K, uint32_t nk, const uint32_t *__restrict__ primes,
                                    uint32_t np, FilterPrime *__restrict__ out) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= np) return;
    const uint64_t p = primes[i];
    uint64_t r = 0;
    for (int j = (int)nk - 1; j >= 0; --j) r = ((r << 32) | K[j]) % p;  // Horner, high to low
    const uint64_t mu = ~0ull / p, c = 0 - mu * p;                     // 2^64 = mu p + c
    FilterPrime f;
    f.phi = r * mu + (uint64_t)((double)r * (double)c / (double)p);
    f.mu = mu;
    f.off = kMargin - (mu << 31);
    f.p = (uint32_t)p;
    f.kmod = (uint32_t)r;
    out[i] = f;
}

// High word of the fixed-point residue of (m, x + 2^31).
__device__ __forceinline__ uint32_t fixed_high(uint64_t phi, uint64_t mu, uint64_t off, uint32_t m, uint32_t xs) {
    const uint64_t lo = (uint64_t)m * (uint32_t)phi + off;
    const uint64_t lo2 = (uint64_t)xs * (uint32_t)mu + lo;
    return (uint32_t)(lo2 >> 32) + m * (uint32_t)(phi >> 32) + xs * (uint32_t)(mu >> 32);
}

__device__ __forceinline__ bool divides(const FilterPrime &f, uint64_t m, int64_t x) {
    const uint64_t p = f.p, u = f.mu;
    const uint64_t ax = x < 0 ? (uint64_t)(-(x + 1)) + 1u : (uint64_t)x;
    const uint64_t mr = mod_barrett(mod_barrett(m, p, u) * f.kmod, p, u);  // m*K mod p
    const uint64_t xr = mod_barrett(ax, p, u);
    return x < 0 ? (mr == xr) : ((mr + xr == p) || (mr == 0 && xr == 0));
}

__device__ __forceinline__ bool fits_fixed(uint64_t m, int64_t x) {
    return m < (1ull << 32) && x >= -(1ll << 31) && x < (1ll << 31);
}

// The candidates of the prime-parallel stages.  The fixed-point ones fill the
// arrays from the front: (m, x + 2^31) and the row.  Those outside its range (m
// >= 2^32 or |x| >= 2^31) fill `row` from the back, `end` being its end: a
// candidate is on one of the two lists.
struct Listed {
    uint2 *pair;
    uint32_t *row, *end;
    uint32_t *n, *n_wide;
};

// Calls put(place) in the flagged threads, places counted from *n: one global
// atomic per workgroup of 1024 (a counter takes one about every 10 ns: per
// wavefront, 2^20 candidates spent 0.16 ms of the stage's 0.20 on it).
template <class Put>
__device__ __forceinline__ void append(bool flag, uint32_t *n, const Put &put) {
    __shared__ uint32_t total, base;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    const uint64_t mask = __ballot(flag);
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(&total, (uint32_t)__popcll(mask));
    at = (uint32_t)__shfl((int)at, 0, 64) + (uint32_t)__popcll(mask & ((1ull << lane) - 1));
    __syncthreads();
    if (threadIdx.x == 0) base = total ? atomicAdd(n, total) : 0u;
    __syncthreads();
    if (flag) put(base + at);
}
// Both lists; most calls have no wide candidate.
__device__ __forceinline__ void append(bool fixed, uint2 pair, bool wide, uint32_t row, const Listed &out) {
    append(fixed, out.n, [&](uint32_t at) {
        out.pair[at] = pair;
        out.row[at] = row;
    });
    if (__syncthreads_or(wide)) append(wide, out.n_wide, [&](uint32_t at) { out.end[-1 - (int64_t)at] = row; });
}

// First stage: a thread per candidate over the primes below 2^10 (table
// [0, k1), which the scalar cache holds).  Survivors are kept and listed for
// the prime-parallel stages.
__global__ void __launch_bounds__(1024) filter_first_kernel(const uint64_t *__restrict__ m, const int64_t *__restrict__ x,
                                                            uint32_t count, const FilterPrime *__restrict__ table,
                                                            uint32_t k1, uint8_t *__restrict__ keep, Listed out) {
    const uint32_t i = blockIdx.x * 1024u + threadIdx.x;
    const uint64_t mi = i < count ? m[i] : 0u;
    const int64_t xi = i < count ? x[i] : 0;
    const bool fixed = fits_fixed(mi, xi);
    const uint32_t m32 = (uint32_t)mi, xs = (uint32_t)(xi + (1ll << 31));
    bool alive = i < count;
    if (fixed) {  // four primes share a branch
        const auto high = [&](uint32_t k) {
            const FilterPrime f = table[k];
            return fixed_high(f.phi, f.mu, f.off, m32, xs);
        };
        uint32_t k = 0;
        for (; alive && k + 4 <= k1; k += 4)
            alive = min(min(high(k), high(k + 1)), min(high(k + 2), high(k + 3))) > kMarginTop;
        for (; alive && k < k1; ++k) alive = high(k) > kMarginTop;
    } else {
        for (uint32_t k = 0; alive && k < k1; ++k) alive = !divides(table[k], mi, xi);
    }
    if (i < count) keep[i] = alive ? 1 : 0;
    append(alive && fixed, make_uint2(m32, xs), alive && !fixed, i, out);
}

// The listed candidates still kept.
__global__ void __launch_bounds__(1024) filter_compact_kernel(const uint8_t *__restrict__ keep, Listed in, Listed out) {
    const uint32_t n = *in.n, nw = *in.n_wide;
    for (uint32_t c0 = blockIdx.x * 1024u; c0 < max(n, nw); c0 += gridDim.x * 1024u) {
        const uint32_t c = c0 + threadIdx.x;
        if (c0 < n) {
            const uint2 pair = c < n ? in.pair[c] : make_uint2(0, 0);
            const uint32_t row = c < n ? in.row[c] : 0u;
            append(c < n && keep[row], out.n, [&](uint32_t at) {
                out.pair[at] = pair;
                out.row[at] = row;
            });
        }
        if (c0 < nw) {
            const uint32_t row = c < nw ? in.end[-1 - (int64_t)c] : 0u;
            append(c < nw && keep[row], out.n_wide, [&](uint32_t at) { out.end[-1 - (int64_t)at] = row; });
        }
    }
}

// The other stages (primes below 2^15, then the rest): a thread per prime of
// [k0, k1), over the listed candidates (gridDim.y workgroups take groups of
// eight in turn; the candidates are scalar loads and the eight share a branch).  Of 2^20 pairs of 809#
// some 57 thousand get here, for 75 thousand primes: 4.3 10^9 tests in 0.52 ms
// (8.3 10^12 a second, the multiply-add rate); a thread per candidate with
// Barrett reductions kept 1.3 wavefronts per SIMD busy for 28.0 ms, and the
// primes below 2^15 for 1.27 ms (0.53 in fixed point, waiting for the table).
// Candidates outside the fixed-point range take three Barrett reductions a
// prime in the same split: 2^20 pairs with m above 2^33 in a call of 7.6 ms, against
// 30.2 with a thread per compacted candidate and 146 with a thread per
// candidate over the whole table.
__global__ void __launch_bounds__(256) filter_primes_kernel(const uint64_t *__restrict__ m, const int64_t *__restrict__ x,
                                                          Listed in, const FilterPrime *__restrict__ table, uint32_t k0,
                                                          uint32_t k1, uint8_t *__restrict__ keep) {
    const uint2 *__restrict__ pair = in.pair;
    const uint32_t k = k0 + blockIdx.x * 256u + threadIdx.x, n = *in.n, nw = *in.n_wide;
    if (k >= k1) return;
    const FilterPrime f = table[k];
    const auto clear = [&](uint32_t c, uint32_t high) {
        if (high <= kMarginTop && (f.p < kFixedExact || divides(f, pair[c].x, (int64_t)pair[c].y - (1ll << 31))))
            keep[in.row[c]] = 0;
    };
    for (uint32_t c = 8 * blockIdx.y; c < n; c += 8 * gridDim.y) {
        if (c + 8 > n) {
            for (uint32_t j = c; j < n; ++j) clear(j, fixed_high(f.phi, f.mu, f.off, pair[j].x, pair[j].y));
            break;
        }
        uint32_t high[8], least = ~0u;
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            high[j] = fixed_high(f.phi, f.mu, f.off, pair[c + j].x, pair[c + j].y);
            least = min(least, high[j]);
        }
        if (least > kMarginTop) continue;
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) clear(c + j, high[j]);
    }
    for (uint32_t c = blockIdx.y; c < nw; c += gridDim.y) {
        const uint32_t row = in.end[-1 - (int64_t)c];
        if (divides(f, m[row], x[row])) keep[row] = 0;
    }
}

// out[i] = m_i*K + x_i as `limbs` words; *err |= 1 on overflow or negative.
__global__ void build_kernel(const uint32_t *__restrict__ K, uint32_t nk, const uint64_t *__restrict__ m,
                             const int64_t *__restrict__ x, uint32_t count, uint32_t limbs,
                             uint32_t *__restrict__ out, uint32_t *__restrict__ err) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= count) return;
    uint32_t *o = out + (size_t)i * limbs;
    const uint64_t mi = m[i];
    const uint64_t mlo = (uint32_t)mi, mhi = mi >> 32;
    // m*K: two passes of a 32x(nk) product
    uint64_t c0 = 0, c1 = 0;  // carries of the lo and hi partial rows
    uint32_t bad = 0;
    for (uint32_t j = 0; j < limbs; ++j) {
        const uint64_t kj = j < nk ? K[j] : 0u;
        const uint64_t kj1 = (j >= 1 && j - 1 < nk) ? K[j - 1] : 0u;
        const uint64_t t0 = kj * mlo + c0;           // < 2^64
        c0 = t0 >> 32;
        const uint64_t t1 = kj1 * mhi + (t0 & 0xffffffffu) + c1;
        c1 = t1 >> 32;
        o[j] = (uint32_t)t1;
    }
    if (c0 | c1) bad = 1;
    for (uint32_t j = limbs; j < nk + 2 && !bad; ++j) {
        // words beyond `limbs` must all be zero: recompute their top part
        const uint64_t kj = j < nk ? K[j] : 0u;
        const uint64_t kj1 = (j >= 1 && j - 1 < nk) ? K[j - 1] : 0u;
        if (kj * mlo || kj1 * mhi) bad = 1;
    }
    // + x
    const int64_t xi = x[i];
    if (xi >= 0) {
        uint64_t c = (uint64_t)xi;
        for (uint32_t j = 0; j < limbs && c; ++j) {
            const uint64_t t = (uint64_t)o[j] + (c & 0xffffffffu);
            o[j] = (uint32_t)t;
            c = (c >> 32) + (t >> 32);
        }
        if (c) bad = 1;
    } else {
        uint64_t b = (uint64_t)(-(xi + 1)) + 1u;
        for (uint32_t j = 0; j < limbs && b; ++j) {
            const uint64_t sub = b & 0xffffffffu;
            const uint64_t cur = o[j];
            o[j] = (uint32_t)(cur - sub);
            b = (b >> 32) + (cur < sub ? 1u : 0u);
        }
        if (b) bad = 1;
    }
    if (bad) atomicOr(err, 1u);
}

}  // namespace pgap

using namespace pgap;

static void free_tables(Family &f) {
    if (f.d_filter) (void)hipFree(f.d_filter);
    f.d_filter = nullptr;
    f.filter_limit = 0;
}

void pgap_engine::families_shutdown() {
    for (Family &f : families) {
        if (f.d_K) (void)hipFree(f.d_K);
        f.d_K = nullptr;
        free_tables(f);
    }
    families.clear();
}

static pgap_status family_tables(pgap_engine *e, Family &f, uint32_t limit) {
    if (f.filter_limit == limit && f.d_filter) return PGAP_OK;
    free_tables(f);
    const std::vector<uint32_t> ps = primes_upto(limit);
    f.stage_end[0] = (uint32_t)(std::lower_bound(ps.begin(), ps.end(), 1u << 10) - ps.begin());
    f.stage_end[1] = (uint32_t)(std::lower_bound(ps.begin(), ps.end(), 1u << 15) - ps.begin());
    const size_t n = std::max<size_t>(ps.size(), 1);
    hipError_t he;
    pgap_status st;
    if ((st = e->ensure(e->d_idx0, n * sizeof(uint32_t), "filter primes"))) return st;
    if ((he = hipMalloc(&f.d_filter, n * sizeof(FilterPrime))) != hipSuccess) {
        (void)hipGetLastError();
        f.d_filter = nullptr;
        e->set_error("hipMalloc for %zu filter primes: %s", ps.size(), hipGetErrorString(he));
        return PGAP_E_OOM;
    }
    if (!ps.empty()) {
        he = hipMemcpyAsync(e->d_idx0.p, ps.data(), ps.size() * sizeof(uint32_t), hipMemcpyHostToDevice, e->stream);
        if (he == hipSuccess) {
            hipLaunchKernelGGL(filter_table_kernel, dim3((uint32_t)((ps.size() + 255) / 256)), dim3(256), 0,
                               e->stream, f.d_K, (uint32_t)f.K.size(), (const uint32_t *)e->d_idx0.p,
                               (uint32_t)ps.size(), f.d_filter);
            he = hipGetLastError();
        }
        if (he == hipSuccess) he = hipStreamSynchronize(e->stream);
        if (he != hipSuccess) {
            free_tables(f);
            return e->hip_fail(he, "filter primes");
        }
    }
    f.nprimes = ps.size();
    f.filter_limit = limit;
    return PGAP_OK;
}

extern "C" {

pgap_status pgap_family(pgap_engine *e, uint32_t P, uint32_t D, uint32_t sieve_length, int *family_id) {
    if (!e || !family_id) return PGAP_E_ARG;
    if (!e->ready) return PGAP_E_STATE;
    if (P < 2 || P > 1000000 || D == 0) {
        e->set_error("pgap_family: bad P=%u D=%u", P, D);
        return PGAP_E_ARG;
    }
    for (size_t i = 0; i < e->families.size(); ++i) {
        const Family &f = e->families[i];
        if (f.P == P && f.D == D && f.SL == sieve_length) {
            *family_id = (int)i;
            return PGAP_OK;
        }
    }
    Family f;
    f.P = P;
    f.D = D;
    f.SL = sieve_length;
    if (!primorial_over(P, D, f.K)) {
        e->set_error("pgap_family: d=%u must divide %u# with P#/d > 1 (gap_common.cpp:117-120)", D, P);
        return PGAP_E_ARG;
    }
    f.K_log = ln_words(f.K);
    (void)hipSetDevice(e->opt.device);
    hipError_t he = hipMalloc(&f.d_K, f.K.size() * sizeof(uint32_t));
    if (he != hipSuccess) {
        (void)hipGetLastError();
        e->set_error("hipMalloc K: %s", hipGetErrorString(he));
        return PGAP_E_OOM;
    }
    he = hipMemcpy(f.d_K, f.K.data(), f.K.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (he != hipSuccess) {
        (void)hipFree(f.d_K);
        return e->hip_fail(he, "upload K");
    }
    e->families.push_back(std::move(f));
    *family_id = (int)e->families.size() - 1;
    return PGAP_OK;
}

pgap_status pgap_build_candidates_device(pgap_engine *e, int family, const uint64_t *m, const int64_t *x,
                                         size_t count, uint32_t limbs, uint32_t *d_out) {
    if (!e) return PGAP_E_ARG;
    if (!e->ready) return PGAP_E_STATE;
    Family *f = e->family(family);
    if (!f || (count && (!m || !x || !d_out)) || limbs == 0 || count > 0xffffffffu) {
        e->set_error("pgap_build_candidates_device: bad arguments");
        return PGAP_E_ARG;
    }
    if (count == 0) return PGAP_OK;
    (void)hipSetDevice(e->opt.device);
    pgap_status st;
    if ((st = e->ensure(e->d_m, count * 8, "m")) || (st = e->ensure(e->d_x, count * 8, "x")) ||
        (st = e->ensure(e->d_small, 64, "flags")))
        return st;
    hipError_t he;
    if ((he = hipMemcpyAsync(e->d_m.p, m, count * 8, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
        (he = hipMemcpyAsync(e->d_x.p, x, count * 8, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
        (he = hipMemsetAsync(e->d_small.p, 0, 4, e->stream)) != hipSuccess)
        return e->hip_fail(he, "build upload");
    hipLaunchKernelGGL(build_kernel, dim3((uint32_t)((count + 255) / 256)), dim3(256), 0, e->stream, f->d_K,
                       (uint32_t)f->K.size(), (const uint64_t *)e->d_m.p, (const int64_t *)e->d_x.p, (uint32_t)count,
                       limbs, d_out, (uint32_t *)e->d_small.p);
    if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "build kernel");
    uint32_t err = 0;
    if ((he = hipMemcpyAsync(&err, e->d_small.p, 4, hipMemcpyDeviceToHost, e->stream)) != hipSuccess ||
        (he = hipStreamSynchronize(e->stream)) != hipSuccess)
        return e->hip_fail(he, "build sync");
    if (err) {
        e->set_error("pgap_build_candidates_device: some m*K+x does not fit %u words or is negative", limbs);
        return PGAP_E_TOO_LARGE;
    }
    return PGAP_OK;
}

pgap_status pgap_filter_candidates(pgap_engine *e, int family, const uint64_t *m, const int64_t *x, size_t count,
                                   uint32_t limit, uint8_t *keep) {
    if (!e) return PGAP_E_ARG;
    if (!e->ready) return PGAP_E_STATE;
    Family *f = e->family(family);
    if (!f || (count && (!m || !x || !keep)) || count > 0xffffffffu || limit > 2000000000u) {
        e->set_error("pgap_filter_candidates: bad arguments");
        return PGAP_E_ARG;
    }
    if (count == 0) return PGAP_OK;
    (void)hipSetDevice(e->opt.device);
    pgap_status st;
    if ((st = family_tables(e, *f, limit))) return st;
    if ((st = e->ensure(e->d_m, count * 8, "m")) || (st = e->ensure(e->d_x, count * 8, "x")) ||
        (st = e->ensure(e->d_keep, count, "keep")) || (st = e->ensure(e->d_idx0, count * 12, "index")) ||
        (st = e->ensure(e->d_idx1, count * 12, "index")) || (st = e->ensure(e->d_small, 64, "counters")))
        return st;
    hipError_t he;
    if ((he = hipMemcpyAsync(e->d_m.p, m, count * 8, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
        (he = hipMemcpyAsync(e->d_x.p, x, count * 8, hipMemcpyHostToDevice, e->stream)) != hipSuccess ||
        (he = hipMemsetAsync(e->d_small.p, 0, 16, e->stream)) != hipSuccess)
        return e->hip_fail(he, "filter upload");
    // primes < 2^10, < 2^15, the rest; survivors are compacted between them
    // (counters in d_small: [0], [1], and [2], [3] for the wide candidates)
    const uint32_t np = (uint32_t)f->nprimes;
    const uint32_t e0 = std::min(f->stage_end[0], np), e1 = std::min(f->stage_end[1], np);
    const auto listed = [&](DevBuf &b, int k) {
        uint32_t *row = (uint32_t *)((uint2 *)b.p + count), *n = (uint32_t *)e->d_small.p + k;
        return Listed{(uint2 *)b.p, row, row + count, n, n + 2};
    };
    const Listed la = listed(e->d_idx0, 0), lb = listed(e->d_idx1, 1);
    const uint64_t *d_m = (const uint64_t *)e->d_m.p;
    const int64_t *d_x = (const int64_t *)e->d_x.p;
    uint8_t *d_keep = (uint8_t *)e->d_keep.p;
    hipLaunchKernelGGL(filter_first_kernel, dim3((uint32_t)((count + 1023) / 1024)), dim3(1024), 0, e->stream, d_m, d_x,
                       (uint32_t)count, f->d_filter, e0, d_keep, la);
    if (e0 < e1)
        hipLaunchKernelGGL(filter_primes_kernel, dim3((e1 - e0 + 255) / 256, 512), dim3(256), 0, e->stream, d_m, d_x,
                           la, f->d_filter, e0, e1, d_keep);
    if (e1 < np) {
        hipLaunchKernelGGL(filter_compact_kernel, dim3((uint32_t)std::min<size_t>((count + 1023) / 1024, 512)),
                           dim3(1024), 0, e->stream, d_keep, la, lb);
        hipLaunchKernelGGL(filter_primes_kernel, dim3((np - e1 + 255) / 256, 64), dim3(256), 0, e->stream, d_m, d_x, lb,
                           f->d_filter, e1, np, d_keep);
    }
    if ((he = hipGetLastError()) != hipSuccess) return e->hip_fail(he, "filter kernels");
    if ((he = hipMemcpyAsync(keep, e->d_keep.p, count, hipMemcpyDeviceToHost, e->stream)) != hipSuccess ||
        (he = hipStreamSynchronize(e->stream)) != hipSuccess)
        return e->hip_fail(he, "filter sync");
    return PGAP_OK;
}

}  // extern "C"
