// Instantiation unit: matrix-core strong Lucas variants of up to 3024 bits.
#include "prp_mf_impl.h"
namespace pgap {
static RegisterLucasMF<1, 2, 3, 4, 5, 6> registered_lucas_mf_0;
}
