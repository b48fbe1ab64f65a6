// One instance of the general pooled-lookup kernel: checked forwards.
#include "lookup_general.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_LAUNCH(launch_lookup_i32_checked, int32_t, false, true)
} // namespace fbgemm_amd
