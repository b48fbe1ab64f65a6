// gfx950 kernels of the index operators that run before the lookup:
// bounds_check_indices and pruned_hashmap_lookup.
//
// bounds_check_indices follows the reference's CPU operator
// (fbgemm_gpu/codegen/utils/embedding_bounds_check_host_cpu.cpp:76-219), whose
// loop over the bags is sequential: repairing a bag writes both of its offsets,
// and the next bag starts from the repaired value. Carried through, the offsets
// it leaves are the running maximum of the original offsets clamped to
// [0, num_indices] (the last one replaced by num_indices first), and a bag is
// "bad" (one warning) when the running maximum at its start exceeds its
// original end, or that end exceeds num_indices, or the very first offset is
// negative. A running maximum is a scan, so the GPU computes exactly what the
// sequential loop does, independent of scheduling. (The reference's own GPU
// kernel lets neighbouring bags race on the shared offset.)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "lookup_common.h"

namespace fbgemm_amd {

namespace {

constexpr int SCAN_THREADS = 1024;
constexpr int SCAN_ITEMS = 4; // offsets per thread
constexpr int SCAN_BLOCK = SCAN_THREADS * SCAN_ITEMS;

__device__ __forceinline__ int64_t read_index(const void* p, bool is64, int64_t i) {
  return is64 ? reinterpret_cast<const int64_t*>(p)[i] : (int64_t) reinterpret_cast<const int32_t*>(p)[i];
}
__device__ __forceinline__ void write_index(void* p, bool is64, int64_t i, int64_t v) {
  if (is64) reinterpret_cast<int64_t*>(p)[i] = v;
  else reinterpret_cast<int32_t*>(p)[i] = (int32_t)v;
}

// offsets[k] as the scan sees it: the last one is num_indices, all are clamped
__device__ __forceinline__ int64_t clamped_offset(const void* offsets, bool is64, int64_t k, int64_t total_B, int64_t N) {
  int64_t v = k == total_B ? N : read_index(offsets, is64, k);
  v = v < N ? v : N;
  return v > 0 ? v : 0;
}

__device__ __forceinline__ int64_t block_max(int64_t v, int64_t* lds) {
  const int tid = threadIdx.x;
  lds[tid] = v;
  __syncthreads();
  for (int step = SCAN_THREADS / 2; step > 0; step >>= 1) {
    if (tid < step) lds[tid] = lds[tid] > lds[tid + step] ? lds[tid] : lds[tid + step];
    __syncthreads();
  }
  const int64_t r = lds[0];
  __syncthreads();
  return r;
}

// pass 1: maximum of the clamped offsets of every block of SCAN_BLOCK offsets
__global__ __launch_bounds__(SCAN_THREADS) void bounds_partial_max_kernel(
    const void* offsets, int is64, int64_t total_B, int64_t N, int64_t* partial, int64_t* warning, int mode) {
  __shared__ int64_t lds[SCAN_THREADS];
  if (mode == 1 && blockIdx.x == 0 && threadIdx.x == 0) warning[0] = 0; // WARNING mode starts from zero
  const int64_t base = (int64_t)blockIdx.x * SCAN_BLOCK + (int64_t)threadIdx.x * SCAN_ITEMS;
  int64_t m = 0;
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    const int64_t k = base + i;
    if (k <= total_B) {
      const int64_t v = clamped_offset(offsets, is64, k, total_B, N);
      m = v > m ? v : m;
    }
  }
  m = block_max(m, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = m;
}

// pass 2 (one workgroup): partial[b] becomes the maximum of all blocks before b
__global__ __launch_bounds__(SCAN_THREADS) void bounds_carry_kernel(int64_t* partial, int64_t nblocks) {
  __shared__ int64_t lds[SCAN_THREADS];
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < nblocks; b0 += SCAN_THREADS) {
    const int64_t b = b0 + threadIdx.x;
    const int64_t mine = b < nblocks ? partial[b] : 0;
    lds[threadIdx.x] = mine;
    __syncthreads();
    for (int step = 1; step < SCAN_THREADS; step <<= 1) {
      const int64_t v = (int)threadIdx.x >= step ? lds[threadIdx.x - step] : 0;
      __syncthreads();
      lds[threadIdx.x] = lds[threadIdx.x] > v ? lds[threadIdx.x] : v;
      __syncthreads();
    }
    const int64_t before = threadIdx.x > 0 ? lds[threadIdx.x - 1] : 0;
    const int64_t total = lds[SCAN_THREADS - 1];
    __syncthreads();
    if (b < nblocks) partial[b] = carry > before ? carry : before;
    carry = carry > total ? carry : total;
  }
}

// pass 3: the repaired offsets (into `fixed`), the count of bad bags, the
// conditions a FATAL run reports
__global__ __launch_bounds__(SCAN_THREADS) void bounds_fix_offsets_kernel(
    const void* offsets, int is64, int64_t total_B, int64_t N, const int64_t* carry_in, int carry_is_prefix,
    int64_t* fixed, int mode, int64_t* warning, Status* status) {
  __shared__ int64_t lds[SCAN_THREADS];
  __shared__ int bad_count;
  if (threadIdx.x == 0) bad_count = 0;
  // what the blocks before this one leave: either pass 2 has made it (carry_is_prefix), or, with at most
  // SCAN_THREADS blocks, every block takes the maximum of the earlier blocks' maxima itself and pass 2 is not run
  int64_t carry;
  if (carry_is_prefix) {
    carry = carry_in[blockIdx.x];
  } else {
    carry = block_max(threadIdx.x < blockIdx.x ? carry_in[threadIdx.x] : 0, lds);
  }
  const int64_t base = (int64_t)blockIdx.x * SCAN_BLOCK + (int64_t)threadIdx.x * SCAN_ITEMS;
  int64_t v[SCAN_ITEMS];
  int64_t local = 0;
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    const int64_t k = base + i;
    v[i] = k <= total_B ? clamped_offset(offsets, is64, k, total_B, N) : 0;
    local = v[i] > local ? v[i] : local;
  }
  // running maximum of the threads' local maxima before this thread: inside each wave through lane
  // shuffles, then over the 16 wave maxima (two workgroup barriers instead of twenty)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t incl = local;
  for (int step = 1; step < 64; step <<= 1) {
    const int64_t o = __shfl_up(incl, step, 64);
    if (lane >= step) incl = incl > o ? incl : o;
  }
  int64_t run = __shfl_up(incl, 1, 64); // exclusive inside the wave (values are >= 0)
  if (lane == 0) run = 0;
  __syncthreads(); // lds is free again (the carry above may have used it)
  if (lane == 63) lds[wave] = incl;
  __syncthreads();
  for (int w = 0; w < wave; ++w) run = run > lds[w] ? run : lds[w];
  run = run > carry ? run : carry;
  int bad = 0, err = 0;
  for (int i = 0; i < SCAN_ITEMS; ++i) {
    const int64_t k = base + i;
    if (k > total_B) break;
    run = v[i] > run ? v[i] : run; // repaired offsets[k]
    fixed[k] = run;
    if (k == total_B) {
      if (read_index(offsets, is64, total_B) != N) {
        ++bad; // "the last element in offsets is incorrect"
        err |= ERR_LENGTH_MISMATCH;
      }
    } else {
      // bag k: starts at the repaired offsets[k], ends at the original offsets[k + 1]
      const int64_t end = k + 1 == total_B ? N : read_index(offsets, is64, k + 1);
      const bool first_negative = k == 0 && read_index(offsets, is64, 0) < 0;
      // a first offset beyond num_indices is bad whatever follows it
      const bool first_high = k == 0 && read_index(offsets, is64, 0) > N;
      if (first_negative || first_high || run > end || end > N) {
        ++bad;
        err |= ERR_BAG_OVERRUN;
      }
    }
  }
  if (mode == 1 && bad) atomicAdd(&bad_count, bad);
  if (mode == 0 && err) status_or(status, err);
  __syncthreads();
  if (mode == 1 && threadIdx.x == 0 && bad_count) atomicAdd(reinterpret_cast<unsigned long long*>(warning), (unsigned long long)bad_count);
}

// pass 4: one group of 16 lanes per bag checks the bag's indices against its
// table's row count and (WARNING, IGNORE) writes the repairs back
constexpr int BAG_LANES = 16;
__global__ __launch_bounds__(256) void bounds_check_bags_kernel(
    const int64_t* rows_per_table, int32_t T, void* indices, void* offsets, int is64, int64_t total_B,
    int64_t B, const int32_t* B_offsets, const int64_t* fixed, int mode, int64_t* warning, Status* status) {
  __shared__ int bad_count;
  if (threadIdx.x == 0) bad_count = 0;
  __syncthreads();
  const int sub = threadIdx.x % BAG_LANES;
  const int64_t groups = (int64_t)gridDim.x * (blockDim.x / BAG_LANES);
  int bad = 0;
  for (int64_t bag = (int64_t)blockIdx.x * (blockDim.x / BAG_LANES) + threadIdx.x / BAG_LANES; bag < total_B; bag += groups) {
    int32_t t;
    if (B_offsets) {
      int32_t lo = 0, hi = T; // largest t with B_offsets[t] <= bag
      while (hi - lo > 1) {
        const int32_t mid = (lo + hi) / 2;
        if ((int64_t)B_offsets[mid] <= bag) lo = mid;
        else hi = mid;
      }
      t = lo;
    } else {
      t = (int32_t)(bag / B);
    }
    const int64_t num_rows = rows_per_table[t];
    const int64_t start = fixed[bag], end = fixed[bag + 1];
    for (int64_t i = start + sub; i < end; i += BAG_LANES) {
      const int64_t idx = read_index(indices, is64, i);
      if (idx == -1) continue; // pruned row
      if (idx < 0 || idx >= num_rows) {
        if (mode == 0) {
          status_index(status, i);
        } else {
          ++bad;
          write_index(indices, is64, i, 0);
        }
      }
    }
    if (mode != 0 && sub == 0) {
      write_index(offsets, is64, bag, start);
      if (bag == total_B - 1) write_index(offsets, is64, total_B, end);
    }
  }
  if (mode == 1) {
    if (bad) atomicAdd(&bad_count, bad);
    __syncthreads();
    if (threadIdx.x == 0 && bad_count) atomicAdd(reinterpret_cast<unsigned long long*>(warning), (unsigned long long)bad_count);
  }
}

// ---- bounds check and pruned-row mapping in one pass, out of place --------------------
//
// What a serving forward does to its indices before the lookup (WARNING and IGNORE mode): with
// plain tables one bounds check; with array-pruned tables a check against the logical rows, the
// mapping, and a check against the physical rows. Done by the operators one after the other that
// is two copies (the caller's tensors stay as they are), up to six launches and five passes over
// the indices. Here the inputs are read once and the checked (and mapped) indices and the repaired
// offsets written once. A workgroup owns 256 bags (gridDim.y workgroups share their indices): it
// makes the running maximum of their offsets, which decides what the bags are, and then walks
// their indices as one range, 8 loads in flight per thread: the mapping is a random gather, bound
// by round trips unless many of them overlap.
//   64 tables x 32 bags x 30 entries: 16 us of copies and check -> 9.5 us (its chain of five round
//   trips). 32 pruned tables x 4096 bags x 27: 121 us of copies, check, mapping (64.6) and check ->
//   78 us: the random 4-byte reads of 256 MB of mappings, a line each, 6 TB/s of lines. With the
//   compact mappings (RANKED, 8 bytes per 32 logical rows, 16 MB) 55 us.
// Workgroups take the bags in their order and so go round the XCDs. An eighth of the bags per XCD, whose
// L2 would then hold its tables' records, takes 33 us there, but as long as the longest eighth takes:
// 64 tables x 2048 bags x 30 with 50 times longer bags in the first 8 tables 25 -> 54 us without a
// mapping, 117 -> 379 with the array, 88 -> 274 with records.
// The warning counter is what the last of the separate checks leaves there: with a mapping the
// second check's, which starts from zero and whose offsets are already in order.
//
// What a workgroup needs of the bags before its own is the maximum of their offsets. Up to 16
// workgroups read those offsets themselves. With more, a kernel before this one leaves the maximum of
// every 512 offsets in out_offsets, at the place of the last of them, and at every sixteenth such place
// that of all 8192 up to there, so that the call needs no memory but its own outputs. A workgroup
// combines the 8192s and the 512s before its own bags, a line each but few, with the rest of the
// offsets. The workgroup that owns a place overwrites it with the running maximum up to there while
// others may still read it, which comes to the same: a later workgroup's maximum is over everything
// before its own bags whichever of the two values it finds. Unmapped checks of 32 x 4096, 64 x 8192,
// 64 x 16384 and 128 x 16640 bags take 18.7, 28.1, 49.3 and 109 us (with every workgroup's maximum in
// an array of the library's, which two calls at a time would share: 17.4, 26.5, 49.3 and 111).
constexpr int CR_BAGS = 256; // bags of a workgroup, one per thread
constexpr int CR_LOADS = 8;
constexpr int CR_ONE_LAUNCH_BLOCKS = 16; // up to here every workgroup reads the offsets before its own itself
constexpr int CR_GROUP = 2 * CR_BAGS;         // offsets to a maximum that the kernel before leaves
constexpr int CR_SUPER = 16;                  // groups to a maximum of the second level
constexpr int64_t CR_OWN_CARRY_SUPERS = 1024; // up to here every workgroup goes over those before its own itself

__device__ __forceinline__ int64_t cr_block_max(int64_t v, int64_t* lds) {
  for (int m = 32; m > 0; m >>= 1) {
    const int64_t o = __shfl_xor(v, m, 64);
    v = v > o ? v : o;
  }
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  int64_t r = lds[0];
  for (int w = 1; w < CR_BAGS / 64; ++w) r = r > lds[w] ? r : lds[w];
  __syncthreads();
  return r;
}

// where the maximum of the offsets of group g is left
__device__ __forceinline__ int64_t cr_place(int64_t g) { return (g + 1) * CR_GROUP - 1; }

template <typename index_t>
__global__ __launch_bounds__(CR_BAGS) void check_remap_partial_kernel(const index_t* offsets, int64_t total_B, int64_t N, index_t* out_offsets,
                                                                      int64_t* warning, int mode) {
  constexpr int PER = CR_GROUP / CR_BAGS; // offsets per thread and group
  __shared__ int64_t lds[CR_BAGS / 64];
  if (mode == 1 && blockIdx.x == 0 && threadIdx.x == 0) warning[0] = 0;
  const int64_t place = cr_place(blockIdx.x);
  if (place >= total_B) return; // nobody comes after it
  int64_t m = 0;
  auto take = [&](auto n) { // the last n offsets per thread up to the place, all in flight together
    constexpr int COUNT = decltype(n)::value;
    index_t v[COUNT];
#pragma unroll
    for (int u = 0; u < COUNT; ++u) v[u] = offsets[place + 1 - (u + 1) * CR_BAGS + threadIdx.x];
#pragma unroll
    for (int u = 0; u < COUNT; ++u) m = m > (int64_t)v[u] ? m : (int64_t)v[u];
  };
  if ((blockIdx.x + 1) % CR_SUPER == 0) take(std::integral_constant<int, PER * CR_SUPER>{});
  else take(std::integral_constant<int, PER>{});
  m = cr_block_max(m < N ? m : N, lds); // of offsets clamped to 0 .. N
  if (threadIdx.x == 0) out_offsets[place] = (index_t)m;
}

// One workgroup: the first `n` maxima of the second level become running maxima.
__global__ __launch_bounds__(SCAN_THREADS) void check_remap_carry_kernel(void* out_offsets, int is64, int64_t n) {
  __shared__ int64_t lds[SCAN_THREADS / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < n; b0 += SCAN_THREADS) {
    const int64_t b = b0 + threadIdx.x;
    int64_t run = b < n ? read_index(out_offsets, is64, cr_place(b * CR_SUPER + CR_SUPER - 1)) : 0;
    for (int step = 1; step < 64; step <<= 1) {
      const int64_t o = __shfl_up(run, step, 64);
      if (lane >= step) run = run > o ? run : o;
    }
    if (lane == 63) lds[wave] = run;
    __syncthreads();
    int64_t before = carry;
    for (int w = 0; w < SCAN_THREADS / 64; ++w) {
      if (w < wave) before = before > lds[w] ? before : lds[w];
      carry = carry > lds[w] ? carry : lds[w];
    }
    run = run > before ? run : before;
    if (b < n) write_index(out_offsets, is64, cr_place(b * CR_SUPER + CR_SUPER - 1), run);
    __syncthreads(); // lds is free again
  }
}

template <typename index_t, typename remap_t, bool RANKED>
__global__ __launch_bounds__(CR_BAGS) void check_remap_kernel(CheckRemapArgs a) {
  constexpr bool IS64 = sizeof(index_t) == 8;
  __shared__ int64_t fixed[CR_BAGS + 1];
  __shared__ int64_t t_rows[CR_BAGS], t_logical[CR_BAGS], t_remap[CR_BAGS], t_cap[CR_BAGS];
  __shared__ int64_t t_rank[RANKED ? CR_BAGS : 1];
  __shared__ int64_t lds[CR_BAGS / 64];
  __shared__ int bad_count;
  const int tid = threadIdx.x;
  const int64_t k0 = (int64_t)blockIdx.x * CR_BAGS;
  const int nb = (int)(a.total_B - k0 < CR_BAGS ? a.total_B - k0 : CR_BAGS);
  // every load the walk over the offsets needs, before anything waits: this bag's offset, the one
  // behind the last bag, and what the bags before these leave
  const int64_t mine = tid < nb ? clamped_offset(a.offsets, IS64, k0 + tid, a.total_B, a.N) : 0;
  const int64_t behind = clamped_offset(a.offsets, IS64, k0 + nb, a.total_B, a.N);
  int64_t carry = 0;
  if (a.carry) {
    const index_t* place = reinterpret_cast<const index_t*>(a.out_offsets);
    const int64_t groups = k0 / CR_GROUP, supers = groups / CR_SUPER;
    const int64_t rest = groups * CR_GROUP + tid;
    if (rest < k0) carry = clamped_offset(a.offsets, IS64, rest, a.total_B, a.N);
    const int64_t first = a.carry == 2 && supers > 0 ? supers - 1 : 0; // running maxima: the last says it all
    for (int64_t j = first + tid; j < supers + groups % CR_SUPER; j += CR_BAGS) {
      const int64_t g = j < supers ? j * CR_SUPER + CR_SUPER - 1 : supers * CR_SUPER + (j - supers);
      const int64_t v = (int64_t)__hip_atomic_load(place + cr_place(g), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      carry = carry > v ? carry : v;
    }
  } else {
#pragma unroll
    for (int u = 0; u < CR_ONE_LAUNCH_BLOCKS - 1; ++u) {
      const int64_t k = tid + u * CR_BAGS;
      const int64_t v = k < k0 ? clamped_offset(a.offsets, IS64, k, a.total_B, a.N) : 0;
      carry = carry > v ? carry : v;
    }
  }
  // the tables of these bags, at most one per bag
  const bool small = a.total_B <= 0xffffffffll;
  auto table_of = [&](int64_t k) { return small ? (int64_t)((uint32_t)k / (uint32_t)a.B) : k / a.B; };
  const int64_t t0 = table_of(k0);
  const int nt = (int)(table_of(k0 + nb - 1) - t0) + 1;
  if (tid == 0) bad_count = 0;
  if (tid < nt) {
    t_rows[tid] = a.rows[t0 + tid];
    if (a.remap_offsets) {
      t_logical[tid] = a.logical_rows[t0 + tid];
      t_remap[tid] = a.remap_offsets[t0 + tid];
      t_cap[tid] = a.remap_offsets[t0 + tid + 1] - t_remap[tid];
      if (RANKED) t_rank[tid] = a.rank_offsets[t0 + tid];
    }
  }
  carry = cr_block_max(carry, lds);
  carry = carry < a.N ? carry : a.N; // it is; whatever else may have been there leads to no index that is not
  // running maximum: the repaired offsets
  int64_t run = mine;
  for (int step = 1; step < 64; step <<= 1) {
    const int64_t o = __shfl_up(run, step, 64);
    if ((tid & 63) >= step) run = run > o ? run : o;
  }
  if ((tid & 63) == 63) lds[tid >> 6] = run;
  __syncthreads();
  for (int w = 0; w < (tid >> 6); ++w) run = run > lds[w] ? run : lds[w];
  run = run > carry ? run : carry;
  if (tid < nb) fixed[tid] = run;
  if (tid == nb - 1) fixed[nb] = run > behind ? run : behind;
  __syncthreads();
  int bad = 0;
  if (blockIdx.y == 0) {
    if (tid < nb) {
      const int64_t k = k0 + tid;
      write_index(a.out_offsets, IS64, k, run);
      // see bounds_fix_offsets_kernel
      const int64_t end = k + 1 == a.total_B ? a.N : read_index(a.offsets, IS64, k + 1);
      const int64_t first = k == 0 ? read_index(a.offsets, IS64, 0) : 0;
      if (first < 0 || first > a.N || run > end || end > a.N) ++bad;
      if (k + 1 == a.total_B) {
        write_index(a.out_offsets, IS64, a.total_B, fixed[nb]);
        if (read_index(a.offsets, IS64, a.total_B) != a.N) ++bad;
      }
    }
    if (a.remap_offsets) bad = 0; // the second check starts from zero, and from offsets that are in order
  }
  // the indices of these bags; what lies before the first bag is nobody's and passes through
  const int64_t lo0 = blockIdx.x == 0 ? 0 : fixed[0], hi0 = fixed[nb], own = fixed[0];
  const int64_t share = (hi0 - lo0 + gridDim.y - 1) / gridDim.y;
  const int64_t lo = lo0 + share * blockIdx.y;
  const int64_t hi = lo + share < hi0 ? lo + share : hi0;
  const index_t* in = reinterpret_cast<const index_t*>(a.indices);
  const remap_t* remap = reinterpret_cast<const remap_t*>(a.remap);
  index_t* out = reinterpret_cast<index_t*>(a.out_indices);
  for (int64_t i0 = lo + tid; i0 < hi; i0 += CR_LOADS * CR_BAGS) {
    index_t v[CR_LOADS];
    int t[CR_LOADS];
    bool gather[CR_LOADS];
#pragma unroll
    for (int u = 0; u < CR_LOADS; ++u) {
      const int64_t i = i0 + u * CR_BAGS;
      v[u] = i < hi ? in[i] : 0;
    }
#pragma unroll
    for (int u = 0; u < CR_LOADS; ++u) {
      const int64_t i = i0 + u * CR_BAGS;
      // the last of the tables that starts at or before i
      int l = 0, h = nt;
      while (h - l > 1) {
        const int mid = (l + h) >> 1;
        if (fixed[(t0 + mid) * a.B - k0] <= i) l = mid;
        else h = mid;
      }
      t[u] = l;
      gather[u] = false;
      if (a.remap_offsets && i < hi && i >= own) {
        if (v[u] != (index_t)-1 && (v[u] < 0 || (int64_t)v[u] >= t_logical[l])) v[u] = 0;
        if (t_cap[l] > 0) {
          gather[u] = v[u] >= 0 && (int64_t)v[u] < t_cap[l];
          if (!gather[u]) v[u] = (index_t)-1;
        }
      }
    }
    if (a.remap_offsets) {
      remap_t m[CR_LOADS];
      RankRecord rec[CR_LOADS];
      bool ranked[CR_LOADS];
#pragma unroll
      for (int u = 0; u < CR_LOADS; ++u) {
        ranked[u] = false;
        if (gather[u]) {
          const int64_t rank = RANKED ? t_rank[t[u]] : -1;
          ranked[u] = rank >= 0;
          if (RANKED && ranked[u]) rec[u] = a.rank_records[rank + ((int64_t)v[u] >> 5)];
          else m[u] = remap[t_remap[t[u]] + (int64_t)v[u]];
        }
      }
#pragma unroll
      for (int u = 0; u < CR_LOADS; ++u) {
        if (RANKED && ranked[u]) { // the rank among the kept rows (remap_rank_kernels.hip)
          const uint32_t bit = (uint32_t)v[u] & 31u;
          v[u] = ((rec[u].bits >> bit) & 1u) ? (index_t)(rec[u].before + (uint32_t)__builtin_popcount(rec[u].bits & ((1u << bit) - 1u))) : (index_t)-1;
        } else if (gather[u]) {
          v[u] = (index_t)m[u];
        }
      }
    }
#pragma unroll
    for (int u = 0; u < CR_LOADS; ++u) {
      const int64_t i = i0 + u * CR_BAGS;
      if (i < hi) {
        if (i >= own && v[u] != (index_t)-1 && (v[u] < 0 || (int64_t)v[u] >= t_rows[t[u]])) {
          v[u] = 0;
          ++bad;
        }
        out[i] = v[u];
      }
    }
  }
  if (a.mode != 1) return;
  if (bad) atomicAdd(&bad_count, bad);
  __syncthreads();
  if (tid != 0) return;
  unsigned long long* warning = reinterpret_cast<unsigned long long*>(a.warning);
  if (a.carry) { // the kernel before this one has set the counter to zero
    if (bad_count) atomicAdd(warning, (unsigned long long)bad_count);
    return;
  }
  // one launch: the workgroups add up in a counter that is this call's until the call says that it is
  // zero again: their number in the low 16 bits, what they found above; the last one hands the sum
  // over. One atomic and no fence. 64 tables x 32 bags: 11.5 us, with two launches 13.9.
  const unsigned long long had = atomicAdd(a.counter, ((unsigned long long)bad_count << 16) + 1ull);
  if ((had & 0xffffull) + 1 == (unsigned long long)gridDim.x * gridDim.y) {
    *warning = (had >> 16) + (unsigned long long)bad_count;
    const unsigned long long sum = atomicExch(a.counter, 0ull); // not zero, and here once the counter is
    __hip_atomic_store(a.counter_taken, sum == 0ull ? 1 : 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// MurmurHash3 finalizers, as the reference hashes sparse ids
// (embedding_forward_quantized_cpu_template.cpp:102-120)
__device__ __forceinline__ uint32_t pruned_hash(uint32_t h) {
  h ^= h >> 16;
  h *= 0x85ebca6bu;
  h ^= h >> 13;
  h *= 0xc2b2ae35u;
  h ^= h >> 16;
  return h;
}
__device__ __forceinline__ uint64_t pruned_hash(uint64_t k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

// dense[i] = value of key indices[i] in its table's open-addressing map (linear
// probing, -1 = empty slot = not there), a copy for tables without a map
// (embedding_forward_quantized_cpu_template.cpp:524-603). One lane per index.
// A probe sequence ends after one trip round the table (the reference would
// not return from a full table that lacks the key).
template <typename index_t, typename hash_t>
__global__ __launch_bounds__(256) void pruned_hashmap_lookup_kernel(
    const index_t* indices, const index_t* offsets, const hash_t* hash_table, const int64_t* hash_table_offsets,
    int32_t B, index_t* dense) {
  using uidx_t = typename std::conditional<sizeof(index_t) == 8, uint64_t, uint32_t>::type;
  const int t = blockIdx.y;
  const int64_t table_start = hash_table_offsets[t];
  const int64_t capacity = hash_table_offsets[t + 1] - table_start;
  const int64_t is = offsets[(int64_t)t * B], ie = offsets[(int64_t)(t + 1) * B];
  for (int64_t i = is + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ie; i += (int64_t)gridDim.x * blockDim.x) {
    const index_t idx = indices[i];
    if (capacity == 0) {
      dense[i] = idx;
      continue;
    }
    int64_t slot;
    if (sizeof(index_t) == 8) slot = (int64_t)(pruned_hash((uint64_t)(uidx_t)idx) % (uint64_t)capacity);
    else slot = (int64_t)pruned_hash((uint32_t)(uidx_t)idx) % capacity;
    index_t out = (index_t)-1;
    for (int64_t probes = 0; probes < capacity; ++probes) {
      const hash_t* entry = hash_table + 2 * (table_start + slot);
      const hash_t key = entry[0];
      if (key == (hash_t)-1) break;
      if ((int64_t)key == (int64_t)idx) {
        out = (index_t)entry[1];
        break;
      }
      slot = slot + 1 == capacity ? 0 : slot + 1;
    }
    dense[i] = out;
  }
}

} // namespace

hipError_t launch_bounds_check(const int64_t* rows_per_table, int32_t T, void* indices, void* offsets, bool is64,
                               int64_t num_indices, int64_t total_B, int64_t B, const int32_t* B_offsets, int mode,
                               int64_t* warning, int64_t* fixed, int64_t* partial, Status* status, hipStream_t stream) {
  const int64_t n = total_B + 1;
  const int64_t nblocks = (n + SCAN_BLOCK - 1) / SCAN_BLOCK;
  hipLaunchKernelGGL(bounds_partial_max_kernel, dim3((unsigned)nblocks), dim3(SCAN_THREADS), 0, stream, offsets,
                     is64 ? 1 : 0, total_B, num_indices, partial, warning, mode);
  const int own_carry = nblocks <= SCAN_THREADS; // up to 4 M offsets: one launch less
  if (!own_carry) hipLaunchKernelGGL(bounds_carry_kernel, dim3(1), dim3(SCAN_THREADS), 0, stream, partial, nblocks);
  hipLaunchKernelGGL(bounds_fix_offsets_kernel, dim3((unsigned)nblocks), dim3(SCAN_THREADS), 0, stream, offsets,
                     is64 ? 1 : 0, total_B, num_indices, partial, own_carry ? 0 : 1, fixed, mode, warning, status);
  if (total_B > 0) {
    const int64_t per_block = 256 / BAG_LANES;
    int64_t blocks = (total_B + per_block - 1) / per_block;
    if (blocks > 256 * 64) blocks = 256 * 64;
    hipLaunchKernelGGL(bounds_check_bags_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, rows_per_table, T,
                       indices, offsets, is64 ? 1 : 0, total_B, B, B_offsets, fixed, mode, warning, status);
  }
  return hipGetLastError();
}

int64_t bounds_check_partials(int64_t total_B) { return (total_B + 1 + SCAN_BLOCK - 1) / SCAN_BLOCK; }

bool check_remap_counts(int64_t total_B, int mode) { return mode == 1 && total_B <= CR_ONE_LAUNCH_BLOCKS * CR_BAGS; }

hipError_t launch_check_remap(CheckRemapArgs a, bool is64, bool remap64, hipStream_t stream) {
  const int64_t blocks = (a.total_B + CR_BAGS - 1) / CR_BAGS;
  if (a.total_B <= 0 || a.B <= 0 || blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  a.carry = 0;
  if (blocks > CR_ONE_LAUNCH_BLOCKS || (a.mode == 1 && !a.counter)) {
    a.carry = 1;
    const int64_t groups = (a.total_B + CR_GROUP - 1) / CR_GROUP, supers = a.total_B / (CR_GROUP * CR_SUPER);
    if (is64)
      hipLaunchKernelGGL(check_remap_partial_kernel<int64_t>, dim3((unsigned)groups), dim3(CR_BAGS), 0, stream, (const int64_t*)a.offsets,
                         a.total_B, a.N, (int64_t*)a.out_offsets, a.warning, a.mode);
    else
      hipLaunchKernelGGL(check_remap_partial_kernel<int32_t>, dim3((unsigned)groups), dim3(CR_BAGS), 0, stream, (const int32_t*)a.offsets,
                         a.total_B, a.N, (int32_t*)a.out_offsets, a.warning, a.mode);
    if (supers > CR_OWN_CARRY_SUPERS) {
      a.carry = 2;
      hipLaunchKernelGGL(check_remap_carry_kernel, dim3(1), dim3(SCAN_THREADS), 0, stream, a.out_offsets, is64 ? 1 : 0, supers);
    }
  }
  // a workgroup per 2048 indices (one turn of 8 loads per thread), per 512 where that leaves the device half empty
  const int64_t per = a.N < (int64_t)256 * CR_LOADS * CR_BAGS ? 2 * CR_BAGS : CR_LOADS * CR_BAGS;
  int64_t shares = (a.N / blocks + per - 1) / per;
  shares = shares < 1 ? 1 : (shares > 1024 ? 1024 : shares);
  const dim3 grid((unsigned)blocks, (unsigned)shares), block(CR_BAGS);
  const bool ranked = a.remap_offsets && a.rank_records && a.rank_offsets;
#define FBGEMM_AMD_CHECK_REMAP(INDEX_T, REMAP_T)                                                                          \
  do {                                                                                                                    \
    if (ranked) hipLaunchKernelGGL((check_remap_kernel<INDEX_T, REMAP_T, true>), grid, block, 0, stream, a);              \
    else hipLaunchKernelGGL((check_remap_kernel<INDEX_T, REMAP_T, false>), grid, block, 0, stream, a);                    \
  } while (0)
  if (is64 && remap64) FBGEMM_AMD_CHECK_REMAP(int64_t, int64_t);
  else if (is64) FBGEMM_AMD_CHECK_REMAP(int64_t, int32_t);
  else if (remap64) FBGEMM_AMD_CHECK_REMAP(int32_t, int64_t);
  else FBGEMM_AMD_CHECK_REMAP(int32_t, int32_t);
#undef FBGEMM_AMD_CHECK_REMAP
  return hipGetLastError();
}

hipError_t launch_pruned_hashmap_lookup(const void* indices, const void* offsets, bool idx64, const void* hash_table,
                                        bool hash64, const int64_t* hash_table_offsets, int32_t B, int32_t T,
                                        void* dense, hipStream_t stream) {
  if (T <= 0 || B <= 0) return hipSuccess;
  dim3 grid(64, (unsigned)T), block(256);
  if (idx64 && hash64)
    hipLaunchKernelGGL((pruned_hashmap_lookup_kernel<int64_t, int64_t>), grid, block, 0, stream, (const int64_t*)indices, (const int64_t*)offsets, (const int64_t*)hash_table, hash_table_offsets, B, (int64_t*)dense);
  else if (idx64)
    hipLaunchKernelGGL((pruned_hashmap_lookup_kernel<int64_t, int32_t>), grid, block, 0, stream, (const int64_t*)indices, (const int64_t*)offsets, (const int32_t*)hash_table, hash_table_offsets, B, (int64_t*)dense);
  else if (hash64)
    hipLaunchKernelGGL((pruned_hashmap_lookup_kernel<int32_t, int64_t>), grid, block, 0, stream, (const int32_t*)indices, (const int32_t*)offsets, (const int64_t*)hash_table, hash_table_offsets, B, (int32_t*)dense);
  else
    hipLaunchKernelGGL((pruned_hashmap_lookup_kernel<int32_t, int32_t>), grid, block, 0, stream, (const int32_t*)indices, (const int32_t*)offsets, (const int32_t*)hash_table, hash_table_offsets, B, (int32_t*)dense);
  return hipGetLastError();
}

} // namespace fbgemm_amd
