// gfx950 kernels around the pooled lookup: the bag scheduler, lengths ->
// offsets, the status block, pruned_array_lookup, and
// the launchers the C ABI calls. The lookup kernels themselves are in
// lookup_general.h (any shape) and compiled one instance per translation unit.
#include "launchers.h"
#include "lookup_device.h"

namespace fbgemm_amd {

// ---- bag scheduler -------------------------------------------------------------
//
// One workgroup per window of SORT_WINDOW consecutive bags of a table orders them
// by length, longest first (counting sort over lengths, lengths >= SORT_BINS - 1
// share the first bin). Waves then take consecutive runs of the order, so the
// bags a wave pools side by side need the same number of rounds and no lane
// idles behind a long neighbour. Ties are placed in arrival order of the LDS
// atomics: the order may differ between runs, the results cannot (each bag is
// summed on its own). Windows for tables of many bags: a launch of many rounds of
// waves runs as fast over bags ordered inside windows of a few thousand as over
// tables ordered as a whole, and many workgroups order a table at once.
constexpr int SORT_BINS = 1024;
constexpr int SORT_WINDOW = 2048;
constexpr int SORT_WHOLE_TABLE = 8192;

// A forward waits for this launch, whose 16 waves a workgroup wait for themselves: all offsets are asked for at once (PER
// bags per thread) and kept, a bag's place among those of its length is what its one atomic returns, a wave whose
// bags all have one length makes one atomic, and the waves before a thread's own are added up from 16 reads in flight. With
// offsets read and lengths counted twice, and that sum one read behind the other: 64 tables x 2048 bags 6.4 us, 32 x 4096
// 8.9; now 5.4 and 6.4.
template <int PER>
__global__ __launch_bounds__(1024) void bag_order_kernel(const void* offsets, int off64, int32_t B_table, int32_t window,
                                                         BagEntry* order) {
  __shared__ int bins[SORT_BINS];
  __shared__ __attribute__((aligned(16))) int partial[16];
  // workgroup t * windows + w orders bags w * window .. of table t among themselves
  const int windows = (B_table + window - 1) / window;
  const int t = blockIdx.x / windows;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int first = (blockIdx.x - t * windows) * window;
  const int B = B_table - first < window ? B_table - first : window;
  const int64_t ob = (int64_t)t * B_table + first;
  int64_t o0[PER], o1[PER];
  auto load = [&](auto* p) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int b = min(tid + k * 1024, B - 1);
      o0[k] = (int64_t)p[ob + b];
      o1[k] = (int64_t)p[ob + b + 1];
    }
  };
  if (off64) load(reinterpret_cast<const int64_t*>(offsets));
  else load(reinterpret_cast<const int32_t*>(offsets));
  bins[tid] = 0;
  __syncthreads();
  // bin of a bag: SORT_BINS - 1 - min(length, SORT_BINS - 1), so that the longest come first
  int bin[PER], rank[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t len = o1[k] - o0[k];
    bin[k] = SORT_BINS - 1 - (int)(len < 0 ? 0 : (len > SORT_BINS - 1 ? SORT_BINS - 1 : len));
    rank[k] = 0;
    if (tid + k * 1024 < B) {
      const uint64_t here = __builtin_amdgcn_ballot_w64(true);
      const int common = __builtin_amdgcn_readfirstlane(bin[k]);
      if (__builtin_amdgcn_ballot_w64(bin[k] != common) == 0ull) {
        int at = 0;
        if (lane == 0) at = atomicAdd(&bins[common], (int)__builtin_popcountll(here)); // lane 0 has the smallest bag: it is here
        rank[k] = __builtin_amdgcn_readfirstlane(at) + lane;
      } else {
        rank[k] = atomicAdd(&bins[bin[k]], 1);
      }
    }
  }
  __syncthreads();
  // exclusive scan of the SORT_BINS (== blockDim) counters: inside each wave
  // through lane shuffles, then over the 16 wave totals
  const int mine = bins[tid];
  int incl = mine;
#pragma unroll
  for (int step = 1; step < 64; step <<= 1) {
    const int v = __shfl_up(incl, step, 64);
    if (lane >= step) incl += v;
  }
  if (lane == 63) partial[wave] = incl;
  __syncthreads();
  int before = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) before += w < wave ? partial[w] : 0;
  bins[tid] = before + incl - mine;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int b = tid + k * 1024;
    if (b >= B) break;
    const int64_t exact = o1[k] - o0[k];
    BagEntry be;
    be.o0 = o0[k];
    be.len = (exact < 0 || exact > 0x7fffffffLL) ? -1 : (int32_t)exact;
    be.bag = first + b;
    order[ob + bins[bin[k]] + rank[k]] = be;
  }
}

// ---- helpers ----------------------------------------------------------------

// lengths -> offsets (exclusive prefix sum). Used when the caller passes Caffe2-style lengths instead
// of offsets. One launch without scratch: a workgroup owns a run of lengths, adds up everything before
// it itself (from the caches, 16 loads in flight per thread) and scans its own run 1024 at a time, with one barrier
// a turn. One workgroup walking the whole array took 12.2 us for 10 000 lengths, 8 loads in flight under a
// condition each and four barriers 7.0, this 6.0. At most LENGTHS_MAX_BLOCKS runs, which bounds what is read
// twice (512 bytes per length).
constexpr int LENGTHS_BLOCK = 1024;
constexpr int LENGTHS_MAX_BLOCKS = 256;
template <typename T>
__global__ __launch_bounds__(LENGTHS_BLOCK) void lengths_to_offsets_kernel(const T* lengths, int64_t n, int64_t run, int64_t* offsets) {
  constexpr int WAVES = LENGTHS_BLOCK / 64;
  __shared__ int64_t sums[WAVES], ends[2][WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t first = (int64_t)blockIdx.x * run, end = first + run < n ? first + run : n;
  int64_t mine = first + tid < end ? (int64_t)(int)lengths[first + tid] : 0; // in flight beside the sums
  int64_t sum = 0;
  for (int64_t i0 = tid; i0 < first; i0 += 16 * LENGTHS_BLOCK) {
    int v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) { // every load is made: those past the sum read a length that counts as zero
      const int64_t i = i0 + u * LENGTHS_BLOCK;
      v[u] = (int)lengths[i < first ? i : 0];
      v[u] = i < first ? v[u] : 0;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) sum += v[u];
  }
  if (first > 0) {
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) sum += __shfl_xor(sum, step, 64);
    if (lane == 0) sums[wave] = sum;
  }
  int64_t carry = 0;
  int turn = 0; // which of the two arrays of wave ends: one barrier a turn, the other array may still be read
  for (int64_t i = first + tid; i - tid < end; i += LENGTHS_BLOCK, turn ^= 1) {
    int64_t upto = mine;
#pragma unroll
    for (int step = 1; step < 64; step <<= 1) {
      const int64_t o = __shfl_up(upto, step, 64);
      if (lane >= step) upto += o;
    }
    if (lane == 63) ends[turn][wave] = upto;
    __syncthreads();
    if (i - tid == first && first > 0) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) carry += sums[w];
    }
    int64_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      before += w < wave ? ends[turn][w] : 0;
      all += ends[turn][w];
    }
    if (i < end) offsets[i] = carry + before + upto - mine;
    carry += all;
    mine = i + LENGTHS_BLOCK < end ? (int64_t)(int)lengths[i + LENGTHS_BLOCK] : 0;
  }
  if (end == n && tid == 0) offsets[n] = carry;
}

// what a call finds wrong before it launches anything
__global__ void status_report_kernel(Status* st, int32_t bits) { status_or(st, bits); }

__global__ void status_clear_kernel(Status* st, int32_t mark) {
  st->bits = 0;
  st->pad = mark;
  st->first_bad_pos = ~0ull;
}

// `word` is pinned host memory: a host that reads `number` there sees what the stream did before.
__global__ void status_done_kernel(int32_t* word, int32_t number) {
  __hip_atomic_store(word, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void status_counted_kernel(FlaggedStatus* st, int64_t* warning) {
  if (warning) *warning = (int64_t)st->counted;
  st->counted = 0;
}

// dense[i] = remap[remap_offsets[t] + idx[i]] for tables with a mapping, a copy
// otherwise (…/embedding_forward_quantized_cpu_template.cpp:605-659).
template <typename index_t, typename remap_t>
__global__ __launch_bounds__(256) void pruned_array_lookup_kernel(
    const index_t* indices, const index_t* offsets, const remap_t* remap,
    const int64_t* remap_offsets, int32_t B, int32_t T, index_t* dense) {
  const int t = blockIdx.y;
  const int64_t rs = remap_offsets[t], re = remap_offsets[t + 1];
  const int64_t is = offsets[(int64_t)t * B], ie = offsets[(int64_t)(t + 1) * B];
  const bool mapped = re - rs > 0;
  for (int64_t i = is + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ie; i += (int64_t)gridDim.x * blockDim.x) {
    index_t v = indices[i];
    // an id outside the mapping reads nothing (the reference reads out of bounds there)
    if (mapped) v = (v >= 0 && (int64_t)v < re - rs) ? (index_t)remap[rs + v] : (index_t)-1;
    dense[i] = v;
  }
}

// ---- launchers (called from the C ABI) ---------------------------------------

hipError_t launch_lookup_i64(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_i32(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_i64_general(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_i32_general(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_i64_checked(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_i32_checked(const LookupArgs& a, unsigned blocks, hipStream_t stream);

hipError_t launch_lookup_lean_i64_exact(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_exact(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i64_fast(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_fast(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i64_exact_w4(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_exact_w4(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i64_fast_w4(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_fast_w4(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i64_checked(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_checked(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i64_checked_w4(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_checked_w4(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i64_exact_q8(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_exact_q8(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i64_fast_q8(const LookupArgs& a, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_lean_i32_fast_q8(const LookupArgs& a, unsigned blocks, hipStream_t stream);

// The lean kernel (lookup_lean.h) over a work list (or a single table) whose tables all
// have a lean shape. `exact` selects the reference's sequence of roundings; `wide4`: every table
// of the launch has the shape lookup_lean_wide4_kernel takes.
hipError_t launch_lookup_lean(const LookupArgs& a, bool idx64, bool exact, bool wide4, hipStream_t stream) {
  if (a.num_waves <= 0) return hipSuccess;
  const int64_t blocks = a.xcd_start ? 8 * a.num_waves : a.num_waves;
  if (blocks > 0x7fffffffLL || a.positional) return hipErrorInvalidValue;
  if (a.check_rows) {
    if (!exact || a.out_ty == ST_INT8 || !a.tables) return hipErrorInvalidValue;
    if (wide4 && (!a.redo || !a.redo_count)) return hipErrorInvalidValue;
    if (wide4) return idx64 ? launch_lookup_lean_i64_checked_w4(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_checked_w4(a, (unsigned)blocks, stream);
    return idx64 ? launch_lookup_lean_i64_checked(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_checked(a, (unsigned)blocks, stream);
  }
  if (a.out_ty == ST_INT8) { // the instances whose output stage quantizes the pooled vectors (lean_store_q8)
    if (exact) return idx64 ? launch_lookup_lean_i64_exact_q8(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_exact_q8(a, (unsigned)blocks, stream);
    return idx64 ? launch_lookup_lean_i64_fast_q8(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_fast_q8(a, (unsigned)blocks, stream);
  }
  if (wide4) { // two launches: the kernel, and the one that pools what it has queued
    if (!a.redo || !a.redo_count || !a.tables) return hipErrorInvalidValue;
    if (exact) return idx64 ? launch_lookup_lean_i64_exact_w4(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_exact_w4(a, (unsigned)blocks, stream);
    return idx64 ? launch_lookup_lean_i64_fast_w4(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_fast_w4(a, (unsigned)blocks, stream);
  }
  if (exact) return idx64 ? launch_lookup_lean_i64_exact(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_exact(a, (unsigned)blocks, stream);
  return idx64 ? launch_lookup_lean_i64_fast(a, (unsigned)blocks, stream) : launch_lookup_lean_i32_fast(a, (unsigned)blocks, stream);
}

hipError_t launch_lookup_matrix_i64(const LookupArgs& a, bool int4, bool wide, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_matrix_i32(const LookupArgs& a, bool int4, bool wide, unsigned blocks, hipStream_t stream);

// The matrix kernel (lookup_matrix.h) over a work list of `wave_bags` bags a wave whose tables it takes.
hipError_t launch_lookup_matrix(const LookupArgs& a, bool idx64, bool int4, bool wide, hipStream_t stream) {
  if (a.num_waves <= 0) return hipSuccess;
  const int64_t blocks = 8 * a.num_waves;
  if (blocks > 0x7fffffffLL || (a.wave_bags != 8 && a.wave_bags != 16) || !a.tables || !a.work || !a.xcd_start || !a.out_aligned || a.sample_weights || a.remap || a.check_rows || a.check_total || a.index_size > MATRIX_MAX_RUN ||
      a.out_ty == ST_INT8)
    return hipErrorInvalidValue;
  return idx64 ? launch_lookup_matrix_i64(a, int4, wide, (unsigned)blocks, stream) : launch_lookup_matrix_i32(a, int4, wide, (unsigned)blocks, stream);
}

hipError_t launch_lookup(const LookupArgs& a, bool idx64, hipStream_t stream) {
  if (a.num_waves <= 0) return hipSuccess;
  const int64_t blocks = a.xcd_start ? 8 * a.num_waves : a.num_waves;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const bool general = a.remap || a.positional || a.check_total;
  if (a.check_rows) {
    if (general || !a.tables) return hipErrorInvalidValue;
    return idx64 ? launch_lookup_i64_checked(a, (unsigned)blocks, stream) : launch_lookup_i32_checked(a, (unsigned)blocks, stream);
  }
  if (general) return idx64 ? launch_lookup_i64_general(a, (unsigned)blocks, stream) : launch_lookup_i32_general(a, (unsigned)blocks, stream);
  return idx64 ? launch_lookup_i64(a, (unsigned)blocks, stream) : launch_lookup_i32(a, (unsigned)blocks, stream);
}

hipError_t launch_lookup_both_i64_exact(const LookupArgs& a, const WorkRun& lean, unsigned general_blocks, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_both_i64_fast(const LookupArgs& a, const WorkRun& lean, unsigned general_blocks, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_both_i32_exact(const LookupArgs& a, const WorkRun& lean, unsigned general_blocks, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_both_i32_fast(const LookupArgs& a, const WorkRun& lean, unsigned general_blocks, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_both_i64_checked(const LookupArgs& a, const WorkRun& lean, unsigned general_blocks, unsigned blocks, hipStream_t stream);
hipError_t launch_lookup_both_i32_checked(const LookupArgs& a, const WorkRun& lean, unsigned general_blocks, unsigned blocks, hipStream_t stream);

// Both kernels in one launch (lookup_both.h): `a` with the general tables' list, `lean` the lean tables'.
hipError_t launch_lookup_both(const LookupArgs& a, const WorkRun& lean, bool idx64, bool exact, hipStream_t stream) {
  const int64_t general = 8 * a.num_waves, blocks = general + 8 * lean.num_waves;
  if (blocks <= 0) return hipSuccess;
  if (!lookup_both_fits(a.num_waves, lean.num_waves) || !a.tables || !a.work || !a.xcd_start || !lean.work || !lean.xcd_start || a.remap || a.positional || a.check_total ||
      a.out_ty == ST_INT8 || (a.check_rows && !exact))
    return hipErrorInvalidValue;
  if (a.check_rows) return idx64 ? launch_lookup_both_i64_checked(a, lean, (unsigned)general, (unsigned)blocks, stream) : launch_lookup_both_i32_checked(a, lean, (unsigned)general, (unsigned)blocks, stream);
  if (exact) return idx64 ? launch_lookup_both_i64_exact(a, lean, (unsigned)general, (unsigned)blocks, stream) : launch_lookup_both_i32_exact(a, lean, (unsigned)general, (unsigned)blocks, stream);
  return idx64 ? launch_lookup_both_i64_fast(a, lean, (unsigned)general, (unsigned)blocks, stream) : launch_lookup_both_i32_fast(a, lean, (unsigned)general, (unsigned)blocks, stream);
}

hipError_t launch_lookup_burst_i64(const LookupArgs& a, dim3 grid, bool four_waves, int lds_bytes, hipStream_t stream);
hipError_t launch_lookup_burst_i32(const LookupArgs& a, dim3 grid, bool four_waves, int lds_bytes, hipStream_t stream);

// The burst kernel (lookup_burst.h): a workgroup per bag and window of 256 columns. max_D, max_bits: the
// widest table and row type of the launch; waves: 1 or 4 per workgroup; lds_bytes: what a workgroup's
// staged rows may take, at least 8 rows of the widest window.
hipError_t launch_lookup_burst(const LookupArgs& a, bool idx64, int32_t max_D, int32_t max_bits, int waves, int lds_bytes, hipStream_t stream) {
  if (a.B <= 0 || a.T <= 0) return hipSuccess;
  const int windows = (max_D + BURST_COLS - 1) / BURST_COLS;
  if (a.T > 65535 || windows > 65535 || !burst_fits(max_D, max_bits, lds_bytes) || (waves != 1 && waves != 4)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)a.B, (unsigned)a.T, (unsigned)windows);
  return idx64 ? launch_lookup_burst_i64(a, grid, waves == 4, lds_bytes, stream) : launch_lookup_burst_i32(a, grid, waves == 4, lds_bytes, stream);
}

hipError_t launch_bag_order(const void* offsets, bool off64, int32_t B, int32_t T, BagEntry* order, hipStream_t stream) {
  if (T <= 0 || B <= 0) return hipSuccess;
  // Tables of up to SORT_WHOLE_TABLE bags are ordered as a whole: their launches are a few rounds of
  // waves, and longest-first over the whole table is what keeps the drain of such a launch short
  // (32 tables x 4 096 bags of 5..50 rows: 88 us ordered whole, 100 us in windows of 2 048).
  const int window = B <= SORT_WHOLE_TABLE ? B : SORT_WINDOW;
  const int64_t blocks = (int64_t)((B + window - 1) / window) * T;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  const auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(1024), 0, stream, offsets, off64 ? 1 : 0, B, window, order); };
  static_assert(SORT_WHOLE_TABLE <= 8 * 1024 && SORT_WINDOW <= SORT_WHOLE_TABLE, "eight bags per thread at most");
  if (window <= 1024) launch(bag_order_kernel<1>);
  else if (window <= 2048) launch(bag_order_kernel<2>);
  else if (window <= 4096) launch(bag_order_kernel<4>);
  else launch(bag_order_kernel<8>);
  return hipGetLastError();
}

hipError_t launch_lengths_to_offsets(const void* lengths, bool is64, int64_t n, int64_t* offsets, hipStream_t stream) {
  const int64_t tiles = n > 0 ? (n + LENGTHS_BLOCK - 1) / LENGTHS_BLOCK : 1;
  const int64_t run = (tiles + LENGTHS_MAX_BLOCKS - 1) / LENGTHS_MAX_BLOCKS * LENGTHS_BLOCK;
  const unsigned blocks = (unsigned)(n > 0 ? (n + run - 1) / run : 1);
  if (is64) hipLaunchKernelGGL(lengths_to_offsets_kernel<int64_t>, dim3(blocks), dim3(LENGTHS_BLOCK), 0, stream, (const int64_t*)lengths, n, run, offsets);
  else hipLaunchKernelGGL(lengths_to_offsets_kernel<int32_t>, dim3(blocks), dim3(LENGTHS_BLOCK), 0, stream, (const int32_t*)lengths, n, run, offsets);
  return hipGetLastError();
}

hipError_t launch_status_report(Status* st, int32_t bits, hipStream_t stream) {
  hipLaunchKernelGGL(status_report_kernel, dim3(1), dim3(1), 0, stream, st, bits);
  return hipGetLastError();
}

hipError_t launch_status_clear(Status* st, int32_t mark, hipStream_t stream) {
  hipLaunchKernelGGL(status_clear_kernel, dim3(1), dim3(1), 0, stream, st, mark);
  return hipGetLastError();
}

hipError_t launch_status_done(int32_t* word, int32_t number, hipStream_t stream) {
  hipLaunchKernelGGL(status_done_kernel, dim3(1), dim3(1), 0, stream, word, number);
  return hipGetLastError();
}

hipError_t launch_status_counted(FlaggedStatus* st, int64_t* warning, hipStream_t stream) {
  hipLaunchKernelGGL(status_counted_kernel, dim3(1), dim3(1), 0, stream, st, warning);
  return hipGetLastError();
}

hipError_t launch_pruned_array_lookup(const void* indices, const void* offsets, bool idx64, const void* remap,
                                      bool remap64, const int64_t* remap_offsets, int32_t B, int32_t T,
                                      void* dense, hipStream_t stream) {
  if (T <= 0 || B <= 0) return hipSuccess;
  dim3 grid(64, (unsigned)T), block(256);
  if (idx64 && remap64)
    hipLaunchKernelGGL((pruned_array_lookup_kernel<int64_t, int64_t>), grid, block, 0, stream, (const int64_t*)indices, (const int64_t*)offsets, (const int64_t*)remap, remap_offsets, B, T, (int64_t*)dense);
  else if (idx64)
    hipLaunchKernelGGL((pruned_array_lookup_kernel<int64_t, int32_t>), grid, block, 0, stream, (const int64_t*)indices, (const int64_t*)offsets, (const int32_t*)remap, remap_offsets, B, T, (int64_t*)dense);
  else if (remap64)
    hipLaunchKernelGGL((pruned_array_lookup_kernel<int32_t, int64_t>), grid, block, 0, stream, (const int32_t*)indices, (const int32_t*)offsets, (const int64_t*)remap, remap_offsets, B, T, (int32_t*)dense);
  else
    hipLaunchKernelGGL((pruned_array_lookup_kernel<int32_t, int32_t>), grid, block, 0, stream, (const int32_t*)indices, (const int32_t*)offsets, (const int32_t*)remap, remap_offsets, B, T, (int32_t*)dense);
  return hipGetLastError();
}

} // namespace fbgemm_amd
