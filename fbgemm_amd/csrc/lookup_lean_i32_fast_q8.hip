// One instance of the lean pooled-lookup kernel: the one that writes the 8-bit pooled output.
#include "lookup_lean.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LEAN_LAUNCH(launch_lookup_lean_i32_fast_q8, int32_t, false, true, false)
} // namespace fbgemm_amd
