// Table-batched forwards with tables for both lookup kernels, in one launch: the first workgroups are the general
// kernel's (lookup_general.h), the others the lean kernel's (lookup_lean.h), each with its own work list.
//
// What bounds such a forward, unless it is large, is that neither kernel fills the device: 27 general and 13 lean tables
// of 1000 bags x 12 are 7776 and 544 waves, which one behind the other took 43.7 and 18.8 us. Both kernels run at 3 waves
// per SIMD and one wave per workgroup, so a launch of both has the registers of the larger and the LDS of the larger.
// The general kernel's waves take longer and come first.
#pragma once
#include "lookup_general.h"
#include "lookup_lean.h"

namespace fbgemm_amd {

// One instance per index type and arithmetic, and those of checked forwards. `a` carries the general tables' list, `lean` the other one.
template <typename index_t, bool EXACT, bool CHECKED>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(FBGEMM_AMD_MIN_WAVES, 8))) void lookup_both_kernel(const LookupArgs a, const WorkRun lean,
                                                                                                                     unsigned general_blocks) {
  constexpr int ROW_WORDS = MAX_GROUPS * MAX_ROUND * (int)sizeof(StageRow) / 4, MUL_WORDS = MAX_GROUPS * MAX_ROUND * (int)sizeof(StageMul) / 4;
  static_assert(ROW_WORDS + MUL_WORDS <= LEAN_LDS_WORDS, "the general kernel's staging fits the lean kernel's LDS");
  __shared__ __attribute__((aligned(16))) uint32_t lds[LEAN_LDS_WORDS + MAX_GROUPS];
  const int lane = (int)threadIdx.x;
  const bool general = blockIdx.x < general_blocks;
  const unsigned block = general ? blockIdx.x : blockIdx.x - general_blocks;
  const int64_t* xcd_start = general ? a.xcd_start : lean.xcd_start;
  const WaveWork* work = general ? a.work : lean.work;
  // general_blocks is a multiple of 8: a list's run x stays with XCD x
  const int64_t first = xcd_start[block & 7], item = first + (int64_t)(block >> 3);
  if (item >= xcd_start[(block & 7) + 1]) return;
  const WaveWork ww = work[item];
  const TableDesc d = a.tables[ww.table];
  if (general) {
    StageRow* stage_row = reinterpret_cast<StageRow*>(lds);
    StageMul* stage_mul = reinterpret_cast<StageMul*>(lds + ROW_WORDS);
    run_table<index_t, false, CHECKED>(a, d, ww.table, ww.first_bag, lane, stage_row, stage_mul);
  } else {
    lean_dispatch<index_t, EXACT, false, CHECKED>(a, d, ww.table, ww.first_bag, lane, lds);
  }
}

#define FBGEMM_AMD_DEFINE_LOOKUP_BOTH_LAUNCH(FN, INDEX_T, EXACT, CHECKED)                                                         \
  hipError_t FN(const LookupArgs& a, const WorkRun& lean, unsigned general_blocks, unsigned blocks, hipStream_t stream) {         \
    hipLaunchKernelGGL((lookup_both_kernel<INDEX_T, EXACT, CHECKED>), dim3(blocks), dim3(64), 0, stream, a, lean, general_blocks); \
    return hipGetLastError();                                                                                                     \
  }

} // namespace fbgemm_amd
