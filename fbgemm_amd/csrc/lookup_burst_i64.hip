// The burst kernel's instances for 64-bit indices.
#include "lookup_burst.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_BURST_LAUNCH(launch_lookup_burst_i64, int64_t)
} // namespace fbgemm_amd
