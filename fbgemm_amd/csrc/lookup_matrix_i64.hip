// int64_t indices: see lookup_matrix.h
#include "lookup_matrix.h"

namespace fbgemm_amd {
FBGEMM_AMD_DEFINE_MATRIX_LAUNCH(launch_lookup_matrix_i64, int64_t)
} // namespace fbgemm_amd
