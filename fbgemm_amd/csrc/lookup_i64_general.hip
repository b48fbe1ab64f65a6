// One instance of the general pooled-lookup kernel.
#include "lookup_general.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_LAUNCH(launch_lookup_i64_general, int64_t, true, false)
} // namespace fbgemm_amd
