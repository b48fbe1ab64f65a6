// One instance of the launch of both pooled-lookup kernels: checked forwards.
#include "lookup_both.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_BOTH_LAUNCH(launch_lookup_both_i32_checked, int32_t, true, true)
} // namespace fbgemm_amd
