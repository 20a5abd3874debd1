// Carries through chunks of 64 words (prime-gap_amd/csrc/carry.h) as a scan
// forms N = centre + x or centre - x, against word-by-word arithmetic: centres of
// 1 to 150 words whose runs of ones (zeros for a borrow) end at and around
// every chunk boundary.  Prints "ok" and exits 0 when every case agrees.
#include <cstdio>
#include <random>
#include <vector>

#include "../../prime-gap_amd/csrc/carry.h"

typedef std::vector<uint32_t> Words;

static Words serial(const Words &c, bool add, uint32_t x) {
    Words o(c);
    uint64_t carry = x;
    for (size_t j = 0; j < c.size() && carry; ++j) {
        const uint64_t v = add ? (uint64_t)c[j] + carry : (uint64_t)c[j] - carry;
        o[j] = (uint32_t)v;
        carry = add ? v >> 32 : (v >> 32 ? 1 : 0);
    }
    return o;
}

static Words chunked(const Words &c, bool add, uint32_t x) {
    Words o(c.size());
    uint64_t in = 0;
    for (size_t base = 0; base < c.size(); base += 64) {
        uint64_t pass = 0;
        for (size_t k = 0; k < 64; ++k) {  // words past the centre are zero
            const uint32_t w = base + k < c.size() ? c[base + k] : 0u;
            if (base + k && w == (add ? ~0u : 0u)) pass |= 1ull << k;
        }
        const uint32_t first = add ? c[0] + x : c[0] - x;
        if (base == 0) in = (add ? first < x : c[0] < x) ? 2 : 0;
        const pgap::CarryChunk ch = pgap::carry_chunk(pass, in);
        for (size_t k = 0; k < 64 && base + k < c.size(); ++k) {
            const uint32_t one = (uint32_t)(ch.got >> k) & 1u;
            o[base + k] = base + k == 0 ? first : add ? c[base + k] + one : c[base + k] - one;
        }
        in = ch.out;
    }
    return o;
}

int main() {
    std::mt19937 rng(1);
    for (size_t words : {1, 2, 63, 64, 65, 66, 127, 128, 129, 130, 150})
        for (int run : {0, 1, 2, 62, 63, 64, 65, 126, 127, 128, 129, 149})
            for (int side = 0; side < 2; ++side)
                for (uint32_t x : {0u, 1u, 2u, 0x80000000u, 0xffffffffu}) {
                    Words c(words);
                    for (auto &w : c) w = (uint32_t)rng() | 2u;  // neither all zeros nor (below) all ones
                    for (auto &w : c) w &= ~4u;
                    c[0] = side ? 0xffffffffu : 0u;  // x > 0 carries out of word 0
                    for (int j = 1; j <= run && j < (int)words; ++j) c[(size_t)j] = side ? ~0u : 0u;
                    if (serial(c, side, x) != chunked(c, side, x)) {
                        printf("words %zu run %d side %d x %u\n", words, run, side, x);
                        return 1;
                    }
                }
    printf("ok\n");
    return 0;
}
