// One instance of the general pooled-lookup kernel: checked forwards.
#include "lookup_general.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_LAUNCH(launch_lookup_i64_checked, int64_t, false, true)
} // namespace fbgemm_amd
