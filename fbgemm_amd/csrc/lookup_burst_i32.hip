// The burst kernel's instances for 32-bit indices.
#include "lookup_burst.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_BURST_LAUNCH(launch_lookup_burst_i32, int32_t)
} // namespace fbgemm_amd
