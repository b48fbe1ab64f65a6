// int32_t indices: see lookup_matrix.h
#include "lookup_matrix.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_MATRIX_LAUNCH(launch_lookup_matrix_i32, int32_t)
} // namespace fbgemm_amd
