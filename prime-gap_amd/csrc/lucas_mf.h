// lucas_mf.h -- strong Lucas probable-prime test (Selfridge's method A) of one
// number per workgroup on the matrix cores (mont_mf.h).  The verdict is
// lucas_lg.h's: U_d = 0 or V_{d 2^r} = 0 (mod N) for some 0 <= r < s, with
// N + 1 = d 2^s, P = 1, Q = (1 - D) / 4.
//
// The chain runs on the sequence V'_k with parameters P' = 1 / Q - 2 and Q' =
// 1, for which V_2k = Q^k V'_k (Q is a unit: a prime dividing Q and N has U_k
// = V_k = 1 for every k > 0, so such an N fails at once).  A bit of the index then
// costs two products that share an operand, X^2 - 2 and X Y - P', instead of
// the three of the chain that carries Q^k along.  With d = 2 m + 1:
//   D U_d = V_{d+1} - Q V_{d-1} = Q^(m+1) (V'_{m+1} - V'_m),
//     V_d = V_{d+1} + Q V_{d-1} = Q^(m+1) (V'_{m+1} + V'_m),
//   V_{d 2^r} = Q^(d 2^(r-1)) V'_{d 2^(r-1)} for r > 0, V'_d = V'_m V'_{m+1} - P'.
//
// The two products of a step are independent: two wavefronts of a workgroup take
// one each and trade the results through LDS, one barrier a step, so a step has
// a squaring's latency, which is what few numbers are bound by (a scan's round
// lasts as long as its Lucas tests).  Both do the set-up and the final tests
// alike.  One wavefront per number against two, ms for 64 / 1024 / 16384
// numbers: 1108 bits 0.95 / 1.03 / 6.4 -> 0.65 / 0.85 / 7.3, 2128 bits 2.76 / 2.97 /
// 23.9 -> 1.83 / 2.54 / 28.3, 4247 bits 9.7 / 10.2 / 122 -> 6.1 / 8.6 / 98 (there
// both products' fragments spilled).  Filled up it is bound by LDS reads like a
// squaring and the A fragments are loaded by both, 15 to 25% below 3600 bits; numbers
// that get this far are few, so there is no second form for that.
#pragma once
#include "lucas_lg.h"
#include "prp_mf.h"

namespace pgap {
namespace mf {

// x^-1 mod a for gcd(x, a) = 1, 0 otherwise (a > 1).
__device__ __forceinline__ uint32_t inverse_small(uint32_t x, uint32_t a) {
    int64_t r0 = a, r1 = x % a, t0 = 0, t1 = 1;
    while (r1) {
        const int64_t q = r0 / r1, r = r0 - q * r1, t = t0 - q * t1;
        r0 = r1;
        r1 = r;
        t0 = t1;
        t1 = t;
    }
    return r0 == 1 ? (uint32_t)(t0 < 0 ? t0 + a : t0) : 0u;
}

// (rem + the number whose plain words are x, top word LW) / a, a < 2^23, word by
// word from the top in halves that a double holds exactly; returns the
// remainder and leaves the quotient's words in quot.
template <int KB>
__device__ __forceinline__ uint32_t divide_small(const uint32_t (&x)[Wave<KB>::T], uint32_t a, uint32_t lane,
                                                 uint32_t (&quot)[Wave<KB>::T]) {
    constexpr int T = Wave<KB>::T, LW = Wave<KB>::LW;
    const double inv = 1.0 / (double)a;
    uint32_t rem = 0;
#pragma unroll
    for (int q = T - 1; q >= 0; --q) {
        quot[q] = 0;
#pragma unroll 1
        for (int i = q == T - 1 ? LW - 64 * (T - 1) : 63; i >= 0; --i) {
            const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)x[q], i);
            uint32_t word = 0;
#pragma unroll
            for (int half = 1; half >= 0; --half) {
                const uint64_t cur = ((uint64_t)rem << 16) | (half ? v >> 16 : v & 0xffffu);  // < 2^39
                uint32_t d = (uint32_t)((double)cur * inv);
                int32_t left = (int32_t)((uint32_t)cur - d * a);  // within [-a, 2a)
                if (left < 0) {
                    --d;
                    left += (int32_t)a;
                } else if (left >= (int32_t)a) {
                    ++d;
                    left -= (int32_t)a;
                }
                rem = (uint32_t)left;
                word = (word << 16) + d;
            }
            if ((int)lane == i) quot[q] = word;
        }
    }
    return rem;
}

// Selfridge's parameter: the first D = 5, -7, 9, ... with Jacobi(D/N) = -1,
// or 0 when N is proved composite on the way (lucas_lg.h has the rules).  The
// lanes try 64 values at a time.
template <int KB>
__device__ __forceinline__ int32_t selfridge(const uint32_t *__restrict__ nw, uint32_t limbs, uint32_t b,
                                             uint32_t lane) {
    constexpr int S = 32 * words(KB) / (16 * lg::RB) + 1;  // digits of a 16-lane row that hold N
    const uint32_t nwords = (b + 31) / 32;
    for (uint32_t a0 = 5; a0 < lg::kLucasMaxD; a0 += 128) {
        const uint32_t a = a0 + 2 * lane;
        const int j = lg::jacobi(lg::words_mod(nw, nwords, a), a);
        const bool factor = j == 0 && !(b <= 25 && a % nw[0] == 0);
        uint64_t minus = __ballot(j < 0), zero = __ballot(factor);
        if (a0 == 5) {
            const uint64_t early = (1ull << lg::kLucasSquareCheck) - 1;
            if (!((minus | zero) & early)) {
                uint32_t n[S];
                lg::load_digits<S, 16>(nw, limbs, lane & 15u, n);
                if (lg::is_square<S, 16>(n, b, lane & 15u)) return 0;
            }
        }
        const uint64_t stop = minus | zero;
        if (stop) {
            const uint32_t k = (uint32_t)__builtin_ctzll(stop), d = a0 + 2 * k;
            if ((zero >> k) & 1) return 0;
            return (d & 2u) ? -(int32_t)d : (int32_t)d;
        }
    }
    return 0;
}

// LDS of a test: (V'_j, V'_{j+1}) twice, for reading and writing, and a work
// buffer per wavefront.
constexpr int lucas_words(int KB) { return 6 * buf_words(KB); }

// x y R^-1 - c into out's buffer (c: the high tiles' per-word constants with
// the subtrahend taken off); w's buffer is overwritten.
template <int KB>
__device__ __forceinline__ void lucas_product(const Wave<KB> &w, const Wave<KB> &x, const Wave<KB> &y,
                                              const Wave<KB> &out, const int64_t (&c)[Wave<KB>::T]) {
    typedef Wave<KB> W;
    constexpr int T = W::T;
    v4i hi[T], lo[T], a[W::NA], bl[W::NB], bh[W::NBH];
    uint32_t p[T];
    int64_t s[T];
    x.load_a_all(a);
    if constexpr (!W::L::shared) y.load_b_high(bh);
    y.load_b_low(bl);
    W::mul_low(lo, a, bl);
    W::high_of(hi, lo, a, bl, bh);
    w.columns(lo, Weights(1), w.k_low(BIAS), W::k_rest(BIAS), s);
    w.carry(s, p);
    w.store_low(p);
    w.load_b_low(bl);
    W::mul_low(lo, w.ni, bl);
    w.columns(lo, Weights(-1), w.k_low(BIAS), W::k_rest(BIAS), s);
    w.carry(s, p);
    w.store_low(p);
    w.load_b_high(bh);
    W::mul_high(hi, w.nf, bh);
    const Weights one(1);
#pragma unroll
    for (int q = 0; q < T; ++q) s[q] = W::column(hi[q], one, c[q]);
    w.template carry<W::G0>(s, p);
    out.store_high(p);
}

// A test by a workgroup of two wavefronts (`wave` 0 and 1), every thread in it.
template <int KB>
__device__ __forceinline__ uint32_t strong_lucas(const uint32_t *__restrict__ nw, uint32_t limbs, uint32_t *lds,
                                                 uint32_t wave, uint32_t lane) {
    typedef Wave<KB> W;
    constexpr int T = W::T, LW = W::LW;
    constexpr int BW = buf_words(KB);
    W w;
    uint32_t n[T], p[T], b;
    if (!load_n<KB>(nw, limbs, lane, n, &b)) return b == 2 && (nw[0] & 1u) == 0 ? 1u : 0u;  // 2 passes
    const int32_t D = selfridge<KB>(nw, limbs, b, lane);
    if (D == 0) return 0;
    const int32_t Q = (1 - D) / 4;
    const uint32_t qa = Q < 0 ? (uint32_t)(-Q) : (uint32_t)Q;
    const uint32_t ninv = qa > 1 ? inverse_small(lg::words_mod(nw, (b + 31) / 32, qa), qa) : 1u;
    if (ninv == 0) return 0;  // a prime divides Q and N

    // buffers 2 par + i: V'_{j+i}; 4 + wave: work
    __syncthreads();  // the workgroup's previous test has been read
    w.init(lds + wave * BW, lane);  // the wavefront's own V' is stored before the next barrier
    w.init(lds + (2 + wave) * BW, lane);
    w.init(lds + (4 + wave) * BW, lane);
    w.setup(n, b, p);  // R mod N
    int64_t s[T], c[T];
    uint32_t one[T];
#pragma unroll
    for (int q = 0; q < T; ++q) one[q] = p[q];
    w.scale(n, b, 2, p);  // V'_0 = 2
#pragma unroll
    for (int q = 0; q < T; ++q) {
        const int i = w.high_word(q);
        c[q] = (q == 0 ? w.k_high(BIAS) : W::k_rest(BIAS)) - (i >= 0 && i < LW ? value(w.buf[i]) : 0);
    }
    // 1 / |Q|: (R mod N + k N) / |Q| with k making the division exact
    if (qa > 1) {
        uint32_t quot[T];
#pragma unroll 1
        for (uint32_t k = 1, pass = 0; pass < 2; ++pass) {
            // one += k N, as plain words
#pragma unroll
            for (int q = 0; q < T; ++q)
                s[q] = (pass ? (int64_t)one[q] : value(one[q])) + (int64_t)k * (int64_t)n[q] +
                       ((int64_t)BIAS_DIV << 32) - (q == 0 && lane == 0 ? 0 : (int64_t)BIAS_DIV);
            w.carry(s, one);
#pragma unroll
            for (int q = 0; q < T; ++q) one[q] ^= FLIP;
            const uint32_t r = divide_small<KB>(one, qa, lane, quot);
            k = (uint32_t)((uint64_t)(qa - r) * ninv % qa);
        }
        // balanced words of the quotient (below 2 N)
#pragma unroll
        for (int q = 0; q < T; ++q) s[q] = (int64_t)quot[q] + (q == 0 ? w.k_low(BIAS) : W::k_rest(BIAS));
        w.carry(s, one);
    }
    // V'_1 = P' = 1 / Q - 2, reduced
#pragma unroll
    for (int q = 0; q < T; ++q)
        s[q] = (Q < 0 ? -value(one[q]) : value(one[q])) - value(p[q]) + (q == 0 ? w.k_low(BIAS) : W::k_rest(BIAS));
    uint32_t v1[T];
    w.carry(s, v1);
    w.scale(n, b, 1, v1);
    // what this wavefront subtracts: 2 from X^2, P' from X Y
#pragma unroll
    for (int q = 0; q < T; ++q) {
        const int i = w.high_word(q);
        const int64_t cp = (q == 0 ? w.k_high(BIAS) : W::k_rest(BIAS)) - (i >= 0 && i < LW ? value(w.buf[i]) : 0);
        c[q] = wave ? cp : c[q];
    }

    // (V'_j, V'_{j+1}) from j = 0 over the bits of m = N >> (tz + 1): X = V'_{j+bit}
    uint32_t tz = 0;  // N + 1 = d 2^tz
    while (tz < b && ((nw[tz >> 5] >> (tz & 31)) & 1u)) ++tz;
    W x, y, out;
    x.attach(lds + wave * BW, lane);
    if (wave == 0)
        x.store_low(p);  // V'_0
    else
        x.store_low(v1);  // V'_1
    uint32_t par = 0;
    const auto step = [&](uint32_t bit) {
        __syncthreads();
        x.attach(lds + (2 * par + bit) * BW, lane);
        y.attach(lds + (2 * par + (wave ? 1 - bit : bit)) * BW, lane);
        par ^= 1;
        // X^2 - 2 is V'_{2j} (bit 0) or V'_{2j+2} (bit 1), X Y - P' is V'_{2j+1}
        out.attach(lds + (2 * par + (wave ? 1 - bit : bit)) * BW, lane);
        lucas_product<KB>(w, x, y, out, c);
    };
#pragma unroll 1
    for (int i = (int)b - 1; i > (int)tz; --i) step((nw[i >> 5] >> (i & 31)) & 1u);
    __syncthreads();
    // V'_{m+1} -+ V'_m
    uint32_t v0[T];
    const auto state = [&](uint32_t i, uint32_t (&v)[T]) {
        const uint32_t *buf = lds + (2 * par + i) * BW + PAD;
#pragma unroll
        for (int q = 0; q < T; ++q) v[q] = 64 * q + (int)lane < LW ? buf[64 * q + lane] : 0u;
    };
    state(0, v0);
    state(1, v1);
#pragma unroll
    for (int sign = 0; sign < 2; ++sign) {
#pragma unroll
        for (int q = 0; q < T; ++q)
            s[q] = value(v1[q]) + (sign ? value(v0[q]) : -value(v0[q])) + (q == 0 ? w.k_low(BIAS) : W::k_rest(BIAS));
        w.carry(s, p);
        w.store_low(p);
        if (w.classify() == 3) return 1;
    }
    if (tz < 2) return 0;
    // V'_d = V'_m V'_{m+1} - P' (bit 0 writes it as V'_{j+1}), then V'_2k = V'_k^2 -
    // 2, wavefront 0's product with X = V'_k (bit 1 writes it as V'_{j+1} too)
    step(0);
#pragma unroll 1
    for (uint32_t r = 1;; ++r) {
        __syncthreads();
        state(1, v1);
        w.store_low(v1);
        if (w.classify() == 3) return 1;
        if (r + 1 >= tz) return 0;
        step(1);
    }
}

}  // namespace mf
}  // namespace pgap
