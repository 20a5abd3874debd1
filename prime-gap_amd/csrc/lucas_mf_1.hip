// Instantiation unit: matrix-core strong Lucas variants of up to 4560 bits.
#include "prp_mf_impl.h"
namespace pgap {
static RegisterLucasMF<7, 8, 9> registered_lucas_mf_1;
}
