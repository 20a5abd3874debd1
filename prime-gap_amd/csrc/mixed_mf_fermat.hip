// Instantiation unit: mixed-width matrix-core kernel, Fermat base 2.
#include "mixed_impl.h"
namespace pgap {
hipError_t launch_mixed_mf_fermat(const MixedLaunch &a, const MixedEnds &ends, hipStream_t stream) {
    return launch_mixed_mf<KIND_FERMAT2>(a, ends, stream);
}
}  // namespace pgap
