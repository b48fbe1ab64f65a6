// One instance of the general pooled-lookup kernel.
#include "lookup_general.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_LAUNCH(launch_lookup_i32, int32_t, false, false)
} // namespace fbgemm_amd
