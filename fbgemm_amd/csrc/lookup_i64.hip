// One instance of the general pooled-lookup kernel.
//
// With the paired conversion this instance, and no other, compiles to 608 KB of code instead of 390, and takes 8 to 12 %
// longer whatever its output is: 78 tables x 52 bags x 39 of all row types 54.4 -> 58.9 us, 76 x 33 x 19 to fp16 26.8 ->
// 29.1. The lean kernel and the launch of both kernels gain by it (27 x 1791 x 12 to fp16, exact: 108 -> 102 us).
#define FBGEMM_AMD_HALVES_APART
#include "lookup_general.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_LOOKUP_LAUNCH(launch_lookup_i64, int64_t, false, false)
} // namespace fbgemm_amd
