// Instantiation unit: mixed-width matrix-core kernel, strong PRP.
#include "mixed_impl.h"
namespace pgap {
hipError_t launch_mixed_mf_sprp(const MixedLaunch &a, const MixedEnds &ends, hipStream_t stream) {
    return launch_mixed_mf<KIND_SPRP>(a, ends, stream);
}
}  // namespace pgap
