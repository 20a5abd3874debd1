// mont_mf.h -- Montgomery arithmetic on the matrix cores, one number per
// wavefront: numbers are byte strings, and the three products of a Montgomery
// squaring are convolutions of bytes that v_mfma_i32_16x16x64_i8 sums exactly.
//
// Representation.  x is LW words (16 KB - 1 or 16 KB + 1) of four balanced bytes (digits in
// [-128, 127], the operand type of the instruction), 4 LW digits of base 256;
// R = 2^(32 LW).  A word of balanced bytes p has the value (p ^ 0x80808080) -
// 0x80808080, so adding 0x80808080 to every word of a column sum, carrying
// in base 2^32 and flipping the sign bits of the bytes turns any column sum
// into balanced words: digits need no per-byte carries.  Values are residues
// of either sign: a Montgomery product of |a|, |b| <= 40 N is below 0.62 N in
// magnitude for N < R / 2^16 (the quotient's digits are balanced too), so
// nothing is ever reduced conditionally.
//
// Products.  c_k = sum_i a_i b_{k-i} over a tile of 256 consecutive k is a
// 16 x 16 matrix D = A B: k = 4 base + f(row) + 4 col with f(row) = 64 (row / 4)
// + row % 4, A[row][t] = a_{4 base + f(row) - t}, B[t][col] = b_{4 col + t}.  With
// the accumulator layout (lane holds column lane % 16 and rows 4 (lane / 16) +
// 0..3) lane l holds the four bytes of word base + l: words stay in lane order.
// t runs in blocks of 64 (one instruction): block c starts at word 16 c - 15
// for the tiles of the low half (bases 0, 64, ...) and 16 c + HOFF for those of
// the high half (bases HB, HB + 64, ...).  With HB = HOFF + 15 mod 16 the A
// fragments of both are one family, words 15 + 16 u + 16 (row / 4) - 4 (lane
// / 16) downwards: A for block c of low tile q is fragment u = 4 q - c, of high
// tile q it is u = UH + 4 q - c.  N (high tiles) and N^-1 mod R (low tiles)
// stay in registers as A fragments; B is read from the wave's LDS buffer.
// Two layouts: HB = LW - 1 and HOFF = -1, the fewest instructions for LW = 15
// mod 16; or HB a multiple of 16 and HOFF = -15, whose high tiles read the B
// fragments of the low ones, and where HB is a multiple of 64 its first high
// tile is the last low tile of the same product.  Layout gives each width the
// one measured faster.
//
// Reduction.  T = a b; q = -T N^-1 mod R from the low tiles; (T + q N) / R from
// the high tiles alone: everything beneath the word below R, word LW - 1, adds
// less than 2^24 units of it, so rounding there is exact.  The high columns of T
// are never carried: q N accumulates onto them.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pgap {
namespace mf {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v4iu __attribute__((ext_vector_type(4), aligned(4)));

constexpr uint32_t FLIP = 0x80808080u;
// HB and HOFF of a width, see above.  Measured with both layouts, tests/s: 1108
// bits (3 blocks) 3.67 -> 3.89 M with shared B fragments, 4247 (9) 232 -> 241 k;
// 2128 (5) the same, where LW - 1 has the lower latency; one and two blocks 2 to 6%
// fewer (4096 of 450 bits 0.31 against 0.33 ms, 9000 of 705 1.33 against 1.39; one
// number 1 to 4% sooner).  Four and eight blocks would need a tile more for their
// word 16 KB, and at six and seven the high tiles from 64 reach past two (the
// static assertion in Wave).
constexpr bool shared_layout(int KB) { return KB == 3 || KB == 9; }
template <int KB>
struct Layout {
    static constexpr bool shared = shared_layout(KB);
    static constexpr int LW = shared ? 16 * KB + 1 : 16 * KB - 1;
    static constexpr int HB = shared ? (KB < 4 ? 16 * KB : KB / 4 * 64) : LW - 1;
    static constexpr int HOFF = shared ? -15 : -1;
};
constexpr int words(int KB) { return shared_layout(KB) ? 16 * KB + 1 : 16 * KB - 1; }
// Bits a width takes: 16 below R for the lazy bounds (bases up to 63).
constexpr int max_bits(int KB) { return 32 * words(KB) - 16; }

// LDS words of a wave: the number's, with zeros on both sides where fragments
// reach past it (49 words below, 49 above), and one word that masked lanes
// write to.
constexpr int PAD = 64;
constexpr int buf_words(int KB) { return PAD + 16 * KB + 64; }

// Orders a wave's LDS accesses in the compiler; the hardware keeps the LDS
// operations of one wave in order.
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// lane l <- lane l - 1 of the whole wavefront, lane 0 <- lane 63.
__device__ __forceinline__ uint32_t wave_ror(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x13C, 0xF, 0xF, false);
}

__device__ __forceinline__ int64_t value(uint32_t p) { return (int64_t)(p ^ FLIP) - (int64_t)FLIP; }

// Weights of a column's four bytes: the product times `mult` (which may be
// negative), |mult| <= 63.
struct Weights {
    int32_t w0, w1, w2, w3;
    __device__ __forceinline__ explicit Weights(int32_t mult)
        : w0(mult), w1(mult * 256), w2(mult * 65536), w3(mult * 16777216) {
        // opaque, so that a column is four v_mad_i64_i32 and not shifts and
        // 64-bit adds of sign-extended bytes (15 instructions a word)
        asm("" : "+s"(w0), "+s"(w1), "+s"(w2), "+s"(w3));
    }
};

// Bias that keeps the carries out of words non-negative: above the largest
// column sum's value over 2^32 (two products of 580 digits: 2^16.2 times mult).
constexpr uint32_t BIAS = 1u << 18;       // mult 1 or 2
constexpr uint32_t BIAS_WIDE = 1u << 24;  // mult up to 63
constexpr uint32_t BIAS_DIV = 1u << 24;   // words plus a multiple below 2^23 of words

template <int KB>
struct Wave {
    typedef Layout<KB> L;
    static constexpr int LW = L::LW, HB = L::HB;
    static constexpr int T = (LW + 63) / 64;                   // low tiles, and high ones
    static constexpr int UMAX = LW / 16, NA = UMAX + 4;        // A fragments u = -3 .. UMAX
    static constexpr int UH = (HB - L::HOFF - 15) / 16;
    static constexpr int NB = (LW + 14) / 16 + 1;              // B blocks of the low tiles
    static constexpr int NBH = (LW - 1 - L::HOFF) / 16 + 1;    // ... of the high ones
    static constexpr int G0 = LW - 1 - HB;                     // lane of word LW - 1 in the first high tile
    static_assert((2 * LW - HB + 63) / 64 == T, "as many high tiles as low ones");
    static_assert((HB - L::HOFF) % 16 == 15 && 15 + 16 * (UMAX / 4 * 4) + 48 < 16 * KB + 60, "fragments");
    uint32_t *buf;                // word 0 of the wave's operand
    const uint32_t *pa, *pb;      // this lane's A and B fragment origins
    uint32_t *st_lo, *st_hi0, *st_hi;  // store addresses of the last low tile, the first and last high tile
    uint32_t sel, lane;
    v4i nf[NA];  // N as A fragments (those the high tiles use)
    v4i ni[NA];  // N^-1 mod R (the low tiles)

    __device__ __forceinline__ void init(uint32_t *lds, uint32_t l) {
        attach(lds, l);
        for (int i = (int)l; i < buf_words(KB); i += 64) lds[i] = 0;
        lds_order();
    }
    __device__ __forceinline__ void attach(uint32_t *lds, uint32_t l) {
        lane = l;
        buf = lds + PAD;
        const uint32_t m = l & 15u, h = l >> 4;
        pa = buf + 16 * (m >> 2) - 4 * h;
        pb = buf + m + 4 * h;
        sel = 0x01020304u + (m & 3u) * 0x01010101u;
        uint32_t *dummy = buf + 16 * KB + 60;
        const int last = 64 * (T - 1);
        st_lo = (int)l + last < LW ? buf + l + last : dummy;
        const int hi = (int)l + last - G0 - 1, hi0 = (int)l - G0 - 1;
        st_hi = hi >= 0 && hi < LW ? buf + hi : dummy;
        st_hi0 = hi0 >= 0 ? buf + hi0 : dummy;
    }

    // A fragment u of the number in the buffer.
    __device__ __forceinline__ v4i load_a(int u) const {
        const v4i v = *(const v4i *)(pa + 12 + 16 * u);
        const uint32_t lo = pa[11 + 16 * u];
        v4i f;
        f.x = (int)__builtin_amdgcn_perm((uint32_t)v.w, (uint32_t)v.z, sel);
        f.y = (int)__builtin_amdgcn_perm((uint32_t)v.z, (uint32_t)v.y, sel);
        f.z = (int)__builtin_amdgcn_perm((uint32_t)v.y, (uint32_t)v.x, sel);
        f.w = (int)__builtin_amdgcn_perm((uint32_t)v.x, lo, sel);
        return f;
    }
    // Lane 16 h + 4 g + j of fragment u holds piece u + g of the number (16
    // words; pieces outside 0 .. UMAX are zero), so one load in four is
    // enough: the fragments between are its rows moved by 4 lanes a step, at
    // 1 or 2 moves a word against 1.2 words loaded and a permute.  The
    // kernel is bound by LDS reads (a squaring read 159 cycles of them at 1108
    // bits, 109 now) as much as by the vector ALU: 3.06 -> 3.90 M tests/s at 1108
    // bits, 1.0 -> 1.07 at 2128, 237 -> 248 k at 4247.  Moving words for the B
    // fragments too (2 moves each) costs more than the reads they replace.
    __device__ __forceinline__ void load_a_all(v4i (&a)[NA]) const {
#pragma unroll
        for (int b = 0; b <= UMAX; b += 4) a[b + 3] = load_a(b);
#pragma unroll
        for (int u = -3; u <= UMAX; ++u) {
            if (u >= 0 && u % 4 == 0) continue;
            const v4i z = {0, 0, 0, 0};
            if (u < 0) {
                a[u + 3] = u == -1 ? shift<0x114>(z, a[3]) : u == -2 ? shift<0x118>(z, a[3]) : shift<0x11C>(z, a[3]);
            } else {
                const int b = u / 4 * 4, r = u % 4;
                v4i up = z;
                if (b + 4 <= UMAX) {
                    const v4i &f = a[b + 7];
                    up = r == 1 ? shift<0x11C>(z, f) : r == 2 ? shift<0x118>(z, f) : shift<0x114>(z, f);
                }
                const v4i &f = a[b + 3];
                a[u + 3] = r == 1 ? shift<0x104>(up, f) : r == 2 ? shift<0x108>(up, f) : shift<0x10C>(up, f);
            }
        }
    }
    // Rows of 16 lanes moved by a DPP shift; lanes without a source keep old.
    template <int CTRL>
    __device__ __forceinline__ static int shift(int old, int v) {
        return __builtin_amdgcn_update_dpp(old, v, CTRL, 0xF, 0xF, false);
    }
    template <int CTRL>
    __device__ __forceinline__ static v4i shift(const v4i &old, const v4i &v) {
        return v4i{shift<CTRL>(old.x, v.x), shift<CTRL>(old.y, v.y), shift<CTRL>(old.z, v.z), shift<CTRL>(old.w, v.w)};
    }

    // Every B fragment of the number in the buffer, for its low or high tiles.
    // The barrier keeps the loads together: left to itself the compiler loads
    // two blocks at a time and the matrix core idles for an LDS latency
    // between them.
    __device__ __forceinline__ void load_b_low(v4i (&b)[NB]) const {
#pragma unroll
        for (int c = 0; c < NB; ++c) b[c] = *(const v4iu *)(pb + 16 * c - 15);
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void load_b_high(v4i (&b)[NBH]) const {
#pragma unroll
        for (int c = 0; c < NBH; ++c) b[c] = *(const v4iu *)(pb + 16 * c + L::HOFF);
        __builtin_amdgcn_sched_barrier(0);
    }

    // Low tiles of A times B (columns of words 0 ..).
    __device__ __forceinline__ static void mul_low(v4i (&acc)[T], const v4i (&a)[NA], const v4i (&b)[NB]) {
#pragma unroll
        for (int q = 0; q < T; ++q) acc[q] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
            for (int q = 0; q < T; ++q)
                if (4 * q - c >= -3 && 4 * q - c <= UMAX)
                    acc[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[4 * q - c + 3], b[c], acc[q], 0, 0, 0);
    }
    // High tiles q0 .. (columns of words HB + 64 q ..), added to acc.
    __device__ __forceinline__ static void mul_high(v4i (&acc)[T], const v4i (&a)[NA], const v4i (&b)[NBH],
                                                    int q0 = 0) {
#pragma unroll
        for (int c = 0; c < NBH; ++c)
#pragma unroll
            for (int q = 0; q < T; ++q)
                if (q >= q0 && UH + 4 * q - c >= -3 && UH + 4 * q - c <= UMAX)
                    acc[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[UH + 4 * q - c + 3], b[c], acc[q], 0, 0, 0);
    }
    // The high tiles of a product whose low tiles are lo and low B fragments bl.
    __device__ __forceinline__ static void high_of(v4i (&hi)[T], const v4i (&lo)[T], const v4i (&a)[NA],
                                                   const v4i (&bl)[NB], const v4i (&bh)[NBH]) {
#pragma unroll
        for (int q = 0; q < T; ++q) hi[q] = v4i{0, 0, 0, 0};
        if constexpr (L::shared) {
            if constexpr (HB % 64 == 0) {
                hi[0] = lo[HB / 64];
                mul_high(hi, a, bl, 1);
            } else {
                mul_high(hi, a, bl);
            }
        } else {
            mul_high(hi, a, bh);
        }
    }

    // Base-2^32 carries over the T x 64 words of s (every true carry plus the
    // bias is non-negative), then balanced bytes.
    // G: the lowest word's lane (lanes below it hold nothing).
    template <int G = 0>
    __device__ __forceinline__ void carry(const int64_t (&s)[T], uint32_t (&p)[T]) const {
        uint32_t prev = 0;
        uint64_t cy[T], any = 0;
#pragma unroll
        for (int q = 0; q < T; ++q) {
            const uint32_t rot = wave_ror((uint32_t)((uint64_t)s[q] >> 32));
            const uint32_t in = lane <= (q == 0 ? G : 0) ? prev : rot;
            prev = rot;
            p[q] = (uint32_t)s[q] + in;
            cy[q] = __ballot(p[q] < in);
            if (q == 0) cy[q] &= ~0ull << G;
            any |= cy[q];
        }
        // a carry out of a word is rare: its addend is below 2^19 (2^25 with
        // a large base)
        while (__builtin_expect(any != 0, 0)) {
            uint64_t top = 0;
            any = 0;
#pragma unroll
            for (int q = 0; q < T; ++q) {
                const uint64_t in = (cy[q] << 1) | top;
                top = cy[q] >> 63;
                const uint32_t one = (uint32_t)(in >> lane) & 1u;
                p[q] += one;
                cy[q] = __ballot(p[q] < one);
                if (q == 0) cy[q] &= ~0ull << G;
                any |= cy[q];
            }
        }
#pragma unroll
        for (int q = 0; q < T; ++q) p[q] ^= FLIP;
    }
    // Per-word constants: the balancing and the bias a word passes up and the
    // one it receives (the lowest word receives none; the lowest word of the
    // high tiles is rounded away instead of balanced).
    __device__ __forceinline__ static int64_t k_rest(uint32_t bias) {
        return ((int64_t)bias << 32) + FLIP - bias;
    }
    __device__ __forceinline__ int64_t k_low(uint32_t bias) const {
        return lane == 0 ? ((int64_t)bias << 32) + FLIP : k_rest(bias);
    }
    __device__ __forceinline__ int64_t k_high(uint32_t bias) const {
        return lane == G0 ? ((int64_t)bias << 32) + 0x80000000u : k_rest(bias);
    }
    __device__ __forceinline__ static int64_t column(const v4i &a, const Weights &w, int64_t k) {
        return k + (int64_t)a.x * w.w0 + (int64_t)a.y * w.w1 + (int64_t)a.z * w.w2 + (int64_t)a.w * w.w3;
    }
    __device__ __forceinline__ void columns(const v4i (&acc)[T], const Weights &w, int64_t k0, int64_t k,
                                            int64_t (&s)[T]) const {
#pragma unroll
        for (int q = 0; q < T; ++q) s[q] = column(acc[q], w, q == 0 ? k0 : k);
    }

    // The number's word that lane l of high tile q holds.
    __device__ __forceinline__ int high_word(int q) const { return 64 * q + (int)lane - G0 - 1; }

    // Balanced words into the buffer: low tiles hold words 0 .., high tiles
    // high_word().
    __device__ __forceinline__ void store_low(const uint32_t (&p)[T]) const {
        lds_order();
#pragma unroll
        for (int q = 0; q < T - 1; ++q) buf[64 * q + lane] = p[q];
        *st_lo = p[T - 1];
        lds_order();
    }
    __device__ __forceinline__ void store_high(const uint32_t (&p)[T]) const {
        lds_order();
#pragma unroll
        for (int q = 0; q < T - 1; ++q) *(q == 0 ? st_hi0 : buf + high_word(q)) = p[q];
        *st_hi = p[T - 1];
        lds_order();
    }

    // The number in the buffer holds T mod R (low words): leaves q = -T N^-1
    // mod R there.
    __device__ __forceinline__ void quotient() const {
        v4i acc[T];
        int64_t s[T];
        uint32_t p[T];
        v4i b[NB];
        load_b_low(b);
        mul_low(acc, ni, b);
        columns(acc, Weights(-1), k_low(BIAS), k_rest(BIAS), s);
        carry(s, p);
        store_low(p);
    }

    // buffer <- buffer^2 R^-1 mult mod N; p: the result's words (high layout).
    __device__ __forceinline__ void square(int32_t mult, uint32_t bias, uint32_t (&p)[T]) const {
        v4i hi[T], lo[T], bh[NBH], bl[NB], a[NA];
        int64_t s[T];
        load_a_all(a);
        if constexpr (!L::shared) load_b_high(bh);
        load_b_low(bl);
        mul_low(lo, a, bl);
        // the high columns of T are summed while its low words are carried
        high_of(hi, lo, a, bl, bh);
        columns(lo, Weights(1), k_low(BIAS), k_rest(BIAS), s);
        carry(s, p);
        store_low(p);
        // q = -T N^-1 mod R
        load_b_low(bl);
        mul_low(lo, ni, bl);
        columns(lo, Weights(-1), k_low(BIAS), k_rest(BIAS), s);
        carry(s, p);
        store_low(p);
        load_b_high(bh);
        mul_high(hi, nf, bh);
        columns(hi, Weights(mult), k_high(bias), k_rest(bias), s);
        carry<G0>(s, p);
        store_high(p);
    }

    // 1 if the number in the buffer, times R^-1, is 1 mod N, 2 if it is -1, 3
    // if it is 0, else 0 (leaves the buffer overwritten).  Its reduction (x +
    // q N) / R is within 0.51 N of zero, so 1, -1 and 0 show as themselves; x
    // itself adds less than 2^22 below the rounding word.
    __device__ __forceinline__ uint32_t classify() const {
        v4i hi[T];
        int64_t s[T];
        uint32_t p[T];
        quotient();
#pragma unroll
        for (int q = 0; q < T; ++q) hi[q] = v4i{0, 0, 0, 0};
        v4i b[NBH];
        load_b_high(b);
        mul_high(hi, nf, b);
        columns(hi, Weights(1), k_high(BIAS), k_rest(BIAS), s);
        carry<G0>(s, p);
        bool rest = false;  // some word above the lowest is not zero
#pragma unroll
        for (int q = 0; q < T; ++q) {
            const int w = high_word(q);
            rest |= w >= 1 && w < LW && p[q] != 0;
        }
        if (__ballot(rest) != 0) return 0;
        const uint32_t w0 = (uint32_t)__builtin_amdgcn_readlane((int)p[0], G0 + 1);
        return w0 == 1u ? 1u : (w0 == 0xffu ? 2u : (w0 == 0u ? 3u : 0u));
    }

    // Loads N (odd, b bits, words in n[] in lane order), its inverse mod R,
    // and leaves R mod N in the buffer as balanced words p (low layout).
    // `nd` and `tw`: N's top as a double in units of its top word tw.
    __device__ __forceinline__ void setup(const uint32_t (&n)[T], uint32_t b, uint32_t (&p)[T]) {
        int64_t s[T];
#pragma unroll
        for (int q = 0; q < T; ++q) s[q] = (int64_t)n[q] + (q == 0 ? k_low(BIAS) : k_rest(BIAS));
        carry(s, p);
        store_low(p);
        load_a_all(ni);  // N for now
#pragma unroll
        for (int u = 0; u < NA; ++u) nf[u] = ni[u];
        // N^-1 by Newton's iteration y <- y (2 - N y), 30 bits to start
        const uint32_t n0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)n[0]);
        uint32_t y0 = n0;
#pragma unroll
        for (int i = 0; i < 4; ++i) y0 *= 2u - n0 * y0;
#pragma unroll
        for (int q = 0; q < T; ++q) p[q] = q == 0 && lane == 0 ? (((y0 & 0x3fffffffu) + FLIP) ^ FLIP) : 0u;
        store_low(p);
#pragma unroll 1
        for (int prec = 30; prec < 32 * LW; prec *= 2) {
            v4i y[NA], bl[NB], acc[T];
            load_a_all(y);
            load_b_low(bl);
            mul_low(acc, ni, bl);
            columns(acc, Weights(-1), k_low(BIAS) + (lane == 0 ? 2 : 0), k_rest(BIAS), s);
            carry(s, p);
            store_low(p);
            load_b_low(bl);
            mul_low(acc, y, bl);
            columns(acc, Weights(1), k_low(BIAS), k_rest(BIAS), s);
            carry(s, p);
            store_low(p);
        }
        load_a_all(ni);
        // R mod N: 2^(b-2) times 2 until 2^(32 LW), 16 bits a step
        const uint32_t bit = b - 2;
#pragma unroll
        for (int q = 0; q < T; ++q)
            s[q] = (q == 0 ? k_low(BIAS) : k_rest(BIAS)) +
                   (64 * q + lane == (bit >> 5) ? (int64_t)1 << (bit & 31) : 0);
        carry(s, p);
        uint32_t left = 32 * LW - bit;
#pragma unroll 1
        while (left) {
            const uint32_t k = left < 16 ? left : 16;
            scale(n, b, 1 << k, p);
            left -= k;
        }
    }

    // p <- p * mult mod N (low layout, |p| <= N, mult <= 2^16), |result| <=
    // 0.51 N; the quotient comes from the tops of p and N in double precision.
    // Leaves the result in the buffer.
    __device__ __forceinline__ void scale(const uint32_t (&n)[T], uint32_t b, int32_t mult, uint32_t (&p)[T]) const {
        const int tw = (int)((b - 1) >> 5);
        constexpr double w32 = 1.0 / 4294967296.0;
        uint32_t plain[T];
#pragma unroll
        for (int q = 0; q < T; ++q) plain[q] = n[q];
        // N's top words through the buffer, then p's (words below 0 and
        // above LW read zeros)
        store_low(plain);
        const double nd = (double)buf[tw] + ((double)buf[tw - 1] + (double)buf[tw - 2] * w32) * w32;
        store_low(p);
        const double xd = (double)value(buf[tw + 1]) * 4294967296.0 + (double)value(buf[tw]) +
                          ((double)value(buf[tw - 1]) + (double)value(buf[tw - 2]) * w32) * w32;
        const int32_t quo = (int32_t)__builtin_rint(xd * (double)mult / nd);
        int64_t s[T];
#pragma unroll
        for (int q = 0; q < T; ++q)
            s[q] = value(p[q]) * mult - (int64_t)quo * (int64_t)n[q] + (q == 0 ? k_low(BIAS_WIDE) : k_rest(BIAS_WIDE));
        carry(s, p);
        store_low(p);
    }
};

}  // namespace mf
}  // namespace pgap
