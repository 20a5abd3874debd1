// carry.h -- carries through 64 words at a time (plain C++: a constexpr function
// is host and device code).
#pragma once
#include <stdint.h>

namespace pgap {

// Words 0..63 of a chunk, bit k of `pass` set when word k hands an incoming
// carry on (all ones; all zeros for a borrow).  Adding the carries that enter (1
// into word 0, or 2 into word 1) to `pass` flips exactly the bits of the words
// that receive one.
struct CarryChunk {
    uint64_t got;  // words that receive a carry
    uint64_t out;  // 1 when one leaves word 63
};
constexpr CarryChunk carry_chunk(uint64_t pass, uint64_t in) {
    return CarryChunk{pass ^ (pass + in), pass + in < pass ? 1u : 0u};
}

}  // namespace pgap
