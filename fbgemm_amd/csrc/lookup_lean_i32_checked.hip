// lookup_lean_kernel and lookup_lean_wide4_kernel of checked forwards, int32 indices
#include "lookup_lean.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LEAN_LAUNCH(launch_lookup_lean_i32_checked, int32_t, true, false, true)
FBGEMM_AMD_DEFINE_LEAN_WIDE4_LAUNCH(launch_lookup_lean_i32_checked_w4, int32_t, true, true)
} // namespace fbgemm_amd
