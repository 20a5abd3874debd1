// Instantiation unit: matrix-core variants of up to 4560 bits.
#include "prp_mf_impl.h"
namespace pgap {
static RegisterMF<7, 8, 9> registered_mf_1;
}
