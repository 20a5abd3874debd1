// Instantiation unit: matrix-core variants of up to 3024 bits.
#include "prp_mf_impl.h"
namespace pgap {
static RegisterMF<1, 2, 3, 4, 5, 6> registered_mf_0;
}
