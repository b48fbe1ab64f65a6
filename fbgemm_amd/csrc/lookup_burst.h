// The burst kernel: pooled lookups too small to fill the device.
//
// What bounds such a launch is the chain of memory round trips behind one bag (offsets, indices,
// rows, and again indices and rows for every round of 8 rows), each of them 1 to 2 us on rows that
// are nowhere near the caches or the TLBs; bytes and arithmetic do not show. So one workgroup owns
// one bag (and up to 256 of its columns) and asks for ALL of it at once: a thread per entry reads
// the index, the weight and the row's scale and bias, then every thread copies 16-byte pieces of
// different rows into LDS with 4 or 8 loads in flight, and only then are the rows added up, each
// column by one lane, in index order: the sequence of roundings is the reference's, bit for bit.
// A bag needs three round trips instead of two and one per 8 rows.
//
// WAVES = 1: a wave per bag, a lane owns 4 columns (64 lanes * 4 = the 256 columns), up to 64 rows
// at a time in 4, 8 or 16 KB of LDS. Large launches are bound by how many workgroups are resident, so
// this form keeps 4 loads per thread and adds 4 rows per turn, which fits 5 waves per SIMD without
// spills: 5000 bags x 25 of a 4-bit table in 14.6 us. With 8 loads and 8 rows it needs 128 registers, 4
// waves per SIMD: 16.0; held to 6 and to 8 waves per SIMD it spills: 16.8 and 16.0. WAVES = 4: four waves per bag, a lane
// owns one column, up to 256 rows at a time in 32 KB: for fewer bags than compute units have room
// for, whose rows one wave would need many loads each for, and whose summing loop (a dependent add
// and fma per row and column) is the longest part left. Which of them, and from where on the other
// lookup kernels take over, is decided in c_api.cpp (plan_burst), with the figures.
#pragma once
#include "lookup_device.h"

namespace fbgemm_amd {

// What a row's window of columns looks like in memory and in LDS: np pieces of `size` bytes, piece
// k at byte k * size of the window, the last one at `last` (which is less where a whole piece there
// would leave the row: it then overlaps its neighbour). In LDS the pieces lie end to end.
struct BurstWindow {
  int size, np, last, pitch;
};

// `first`: the window's first byte in row 0; `room`: bytes from there to the end of what may be read
// of a row.
__device__ __forceinline__ BurstWindow burst_window(const TableDesc& d, const uint8_t* first, int64_t room, int wb) {
  BurstWindow w;
  const bool a4 = (((uintptr_t)first | (uintptr_t)d.row_stride) & 3) == 0;
  const int wb16 = (wb + 15) & ~15, wb4 = (wb + 3) & ~3;
  if (a4 && wb16 <= room) { // what follows in the row takes the overhang
    w.size = 16;
    w.np = wb16 >> 4;
    w.last = wb16 - 16;
  } else if (a4 && wb >= 16 && wb == wb4) {
    w.size = 16;
    w.np = wb16 >> 4;
    w.last = wb - 16;
  } else if (a4 && (wb == wb4 || wb4 <= room)) {
    w.size = 4;
    w.np = wb4 >> 2;
    w.last = wb4 - 4;
  } else {
    w.size = 1;
    w.np = wb;
    w.last = wb - 1;
  }
  w.pitch = wb16;
  return w;
}

// K columns of one row from their bytes in LDS, added to the accumulators. `shift`: where the one
// column of a lane (K = 1) sits inside its byte, for the types below 8 bits.
template <int TY, int K>
__device__ __forceinline__ void burst_add(float (&acc)[K], const uint8_t* p, int shift, StageMul m, int fp8_shift, float fp8_mult) {
  constexpr int BITS = type_bits(TY);
  constexpr int BYTES = K * BITS / 8 > 0 ? K * BITS / 8 : 1;
  uint32_t raw[(BYTES + 3) / 4];
  if constexpr (BYTES == 16) {
    const Dwordx4 v = *reinterpret_cast<const Dwordx4*>(p);
    raw[0] = v.v[0]; raw[1] = v.v[1]; raw[2] = v.v[2]; raw[3] = v.v[3];
  } else if constexpr (BYTES == 8) {
    const Dwordx2 v = *reinterpret_cast<const Dwordx2*>(p);
    raw[0] = v.v[0]; raw[1] = v.v[1];
  } else if constexpr (BYTES == 4) {
    raw[0] = *reinterpret_cast<const uint32_t*>(p);
  } else if constexpr (BYTES == 2) {
    raw[0] = *reinterpret_cast<const uint16_t*>(p);
  } else {
    raw[0] = *p;
  }
#pragma unroll
  for (int e = 0; e < K; ++e) {
    if constexpr (TY == ST_FP32) {
      acc[e] = __builtin_fmaf(m.scale, bits_to_float(raw[e]), acc[e]);
    } else if constexpr (TY == ST_FP16) {
      acc[e] = __builtin_fmaf(m.scale, (e & 1) ? half_hi(raw[e / 2]) : half_lo(raw[e / 2]), acc[e]);
    } else if constexpr (TY == ST_BF16) {
      acc[e] = __builtin_fmaf(m.scale, bits_to_float((e & 1) ? (raw[e / 2] & 0xffff0000u) : (raw[e / 2] << 16)), acc[e]);
    } else if constexpr (TY == ST_FP8) {
      const uint32_t b = (raw[e / 4] >> (8 * (e % 4))) & 0xffu;
      const float mag = bits_to_float((b & 0x7fu) << fp8_shift) * fp8_mult;
      acc[e] = __builtin_fmaf(m.scale, bits_to_float(float_to_bits(mag) | ((b & 0x80u) << 24)), acc[e]);
    } else {
      const uint32_t q = (raw[(e * BITS) / 32] >> (K == 1 ? shift : (e * BITS) % 32)) & ((1u << BITS) - 1u);
      acc[e] = __builtin_fmaf(m.scale, (float)q, acc[e] + m.bias);
    }
  }
}

// `rows` staged rows (a multiple of 8: holes carry the multiplier (-0, -0) and zeros, which leave an
// accumulator as it is) added up in order.
template <int TY, int K, int R>
__device__ __forceinline__ void burst_sum(float (&acc)[K], const uint8_t* col, int pitch, int shift, const StageMul* mul, int rows,
                                          int fp8_shift, float fp8_mult) {
#pragma unroll 1
  for (int r = 0; r < rows; r += R) {
#pragma unroll
    for (int u = 0; u < R; ++u) burst_add<TY, K>(acc, col + (r + u) * pitch, shift, mul[r + u], fp8_shift, fp8_mult);
  }
}

// The pieces of `rows` rows into LDS: S lanes (a power of two) take the pieces of a row, the
// workgroup as many rows per load instruction as it has such groups, U loads per thread in flight.
template <int SIZE, int THREADS, int U>
__device__ __forceinline__ void burst_copy(const uint8_t* base, const StageRow* off, int rows, const BurstWindow& w, uint8_t* lds) {
  constexpr int NW = SIZE == 16 ? 4 : 1;
  int log = 0;
  while ((1 << log) < w.np && log < 6) ++log;
  const int S = 1 << log;
  const int sub = threadIdx.x & (S - 1), group = threadIdx.x >> log, groups = THREADS >> log;
#pragma unroll 1
  for (int k = sub; k < w.np; k += S) { // one turn, but for single bytes
    const int from = k * SIZE < w.last ? k * SIZE : w.last;
#pragma unroll 1
    for (int r0 = group; r0 < rows; r0 += U * groups) {
      uint32_t v[U][NW];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = r0 + u * groups;
#pragma unroll
        for (int i = 0; i < NW; ++i) v[u][i] = 0;
        if (r < rows) {
          const int64_t o = off[r].off;
          if (o >= 0) load_raw<SIZE>(v[u], base + o + from);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = r0 + u * groups;
        if (r < rows) {
          uint8_t* p = lds + r * w.pitch + k * SIZE;
          if constexpr (SIZE == 16) *reinterpret_cast<uint4*>(p) = make_uint4(v[u][0], v[u][1], v[u][2], v[u][3]);
          else if constexpr (SIZE == 4) *reinterpret_cast<uint32_t*>(p) = v[u][0];
          else *p = (uint8_t)v[u][0];
        }
      }
    }
  }
}

template <int K>
__device__ __forceinline__ void burst_store(const LookupArgs& a, const float (&acc)[K], int64_t pos, int n) {
  if (n <= 0) return;
  const bool bf = a.out_ty == ST_BF16;
  if (a.out_ty == ST_FP32) {
    float* o = reinterpret_cast<float*>(a.out) + pos;
    if constexpr (K == 4) {
      if (n >= 4 && ((uintptr_t)o & 15) == 0) {
        *reinterpret_cast<float4*>(o) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        return;
      }
    }
#pragma unroll
    for (int e = 0; e < K; ++e)
      if (e < n) o[e] = acc[e];
  } else {
    uint16_t* o = reinterpret_cast<uint16_t*>(a.out) + pos;
    if constexpr (K == 4) {
      if (n >= 4 && ((uintptr_t)o & 7) == 0) {
        *reinterpret_cast<uint2*>(o) = bf ? make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]))
                                          : make_uint2(pack_half2(acc[0], acc[1]), pack_half2(acc[2], acc[3]));
        return;
      }
    }
#pragma unroll
    for (int e = 0; e < K; ++e)
      if (e < n) o[e] = (uint16_t)(bf ? to_bf16_bits(acc[e]) : to_half_bits(acc[e]));
  }
}

// The sum of the first `bag` lengths, for the whole workgroup: 16 loads in flight per thread.
template <int WAVES, typename T>
__device__ __forceinline__ int64_t burst_lengths_before(const T* lengths, int bag, int tid, int64_t* lds) {
  constexpr int THREADS = 64 * WAVES;
  int64_t sum = 0;
  for (int i0 = 0; i0 < bag; i0 += 16 * THREADS) {
    int v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) { // those past the bag read a length that does not count
      const int i = i0 + u * THREADS + tid;
      v[u] = (int)lengths[i < bag ? i : 0];
      v[u] = i < bag ? v[u] : 0;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) sum += v[u];
  }
#pragma unroll
  for (int step = 32; step > 0; step >>= 1) sum += __shfl_xor(sum, step, 64);
  if constexpr (WAVES > 1) {
    if ((tid & 63) == 0) lds[tid >> 6] = sum;
    __syncthreads();
    sum = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) sum += lds[w];
    __syncthreads(); // the rows' places are staged where the sums were
  }
  return sum;
}

// blockIdx: (bag, table, window of columns)
// CHECKED: a checked forward's launch (LookupArgs::check_rows); the other instance keeps its registers and its time.
// LENGTHS: a single table's launch that is handed lengths (LookupArgs::lengths): a workgroup adds up those in front of its bag.
template <typename index_t, int WAVES, bool CHECKED, bool LENGTHS>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(WAVES == 1 ? 5 : 4, 8))) void lookup_burst_kernel(const LookupArgs a, int lds_bytes) {
  constexpr int THREADS = 64 * WAVES;
  constexpr int K = BURST_COLS / THREADS; // columns per lane
  constexpr int LOADS = WAVES == 1 ? 4 : 8;   // in flight per thread
  constexpr int UNROLL = WAVES == 1 ? 4 : 8;  // rows added up per turn
  extern __shared__ __align__(16) uint8_t burst_lds[];
  StageRow* st_row = reinterpret_cast<StageRow*>(burst_lds);
  StageMul* st_mul = reinterpret_cast<StageMul*>(burst_lds + THREADS * sizeof(StageRow));
  uint8_t* lds = burst_lds + THREADS * (sizeof(StageRow) + sizeof(StageMul));
  const int table = blockIdx.y;
  const TableDesc d = a.tables ? a.tables[table] : a.single;
  const int col0 = (int)blockIdx.z * BURST_COLS;
  if (col0 >= d.D) return;
  const int tid = threadIdx.x;
  const int bag = blockIdx.x;
  const bool quant = d.ty == ST_INT8 || d.ty == ST_INT4 || d.ty == ST_INT2;

  // the bag, judged like the other lookup kernels judge it
  const int64_t ob = (int64_t)table * a.B;
  int64_t o0, o1, base = 0;
  if constexpr (LENGTHS) {
    o0 = a.off64 ? burst_lengths_before<WAVES>(reinterpret_cast<const int64_t*>(a.offsets), bag, tid, reinterpret_cast<int64_t*>(burst_lds))
                 : burst_lengths_before<WAVES>(reinterpret_cast<const int32_t*>(a.offsets), bag, tid, reinterpret_cast<int64_t*>(burst_lds));
    o1 = o0 + (int64_t)(int)read_offset(a.offsets, a.off64, bag);
  } else {
    o0 = read_offset(a.offsets, a.off64, ob + bag);
    o1 = read_offset(a.offsets, a.off64, ob + bag + 1);
    if (a.check_total) base = read_offset(a.offsets, a.off64, ob);
  }
  const int64_t pos0 = o0 - base;
  int64_t len = o1 - o0;
  if (len < 0) {
    if (tid == 0) report(a.status, ERR_NEGATIVE_LENGTH);
    len = 0;
  }
  if (len > 0x7fffffffLL || pos0 < 0 || pos0 + len > a.index_size) {
    if (tid == 0) report(a.status, ERR_BAG_OVERRUN);
    len = 0;
  }
  if (a.check_total && bag == a.B - 1 && o1 - base != a.index_size && tid == 0) report(a.status, ERR_LENGTH_MISMATCH);
  if (CHECKED && table == a.T - 1 && bag == a.B - 1 && tid == 0) check_end(a, o1);
  const int n = (int)len;
  const int64_t row_bound = index_bound<CHECKED>(a, d, table, tid == 0);
  const int64_t logical = CHECKED && a.remap ? a.logical_rows[table] : 0;
  int counted = 0; // a checked forward: this thread's indices outside the table

  int64_t remap_base = 0, remap_cap = 0, rank_base = -1;
  bool remapped = false;
  if (a.remap) {
    remapped = true;
    remap_cap = a.remap_rows;
    if (a.remap_offsets) {
      remap_base = a.remap_offsets[table];
      remap_cap = a.remap_offsets[table + 1] - remap_base;
      remapped = remap_cap > 0;
      if (a.rank_records) rank_base = a.rank_offsets[table];
    }
  }

  const int bits = type_bits(d.ty);
  const uint8_t* wbase = (d.placement ? a.weights[1] : a.weights[0]) + d.weights_offset;
  const int64_t in_row = (int64_t)d.data_off + (int64_t)col0 * bits / 8;
  const uint8_t* first = wbase + in_row;
  const int cols = d.D - col0 < BURST_COLS ? d.D - col0 : BURST_COLS;
  // a row of a table batch owns its whole stride; of a single table (whose last row may end with its
  // last element) only the elements and the scale and bias are known to be there
  int64_t row_end = d.row_stride;
  if (!a.tables) {
    row_end = (int64_t)d.data_off + d.data_bytes;
    if (quant) row_end = max(row_end, (int64_t)d.sb_off + (d.sb_fp32 ? 8 : 4));
  }
  const BurstWindow w = burst_window(d, first, row_end - in_row, (cols * bits + 7) >> 3);
  // a multiple of 8, and 8 at least (burst_fits)
  const int cap = min(lds_bytes / w.pitch, THREADS) & ~7;

  // this lane's columns: their bytes inside a staged row
  const int lane_col = tid * K;
  const bool mine = lane_col < cols;
  int at = mine ? (lane_col * bits) >> 3 : 0;
  const int shift = (lane_col * bits) & 7;
  if (w.size == 16 && at >= w.last) at += (w.np - 1) * 16 - w.last;

  float acc[K];
#pragma unroll
  for (int e = 0; e < K; ++e) acc[e] = 0.0f;

  const index_t* idx = reinterpret_cast<const index_t*>(a.indices);
  int64_t row = 0;
  float wt = 1.0f;
  auto load_entry = [&](int i) {
    if (tid < cap && i < n) {
      row = (int64_t)idx[pos0 + i];
      if (a.sample_weights) wt = a.sample_weights[a.positional ? (int64_t)i : pos0 + i];
    }
  };
  load_entry(tid);
  for (int r0 = 0; r0 < n; r0 += cap) {
    const int left = n - r0 < cap ? n - r0 : cap;
    const int rows = (left + 7) & ~7;
    // entry r0 + tid: where its row is, what to multiply it with
    if (tid < rows) {
      int64_t off = -1;
      if (tid < left) {
        const int64_t pos = pos0 + r0 + tid;
        bool ok = true;
        if (CHECKED && a.remap) row = logical_index(row, logical);
        if (remapped) {
          if (row < 0 || row >= remap_cap) {
            if (!CHECKED) report_index(a.status, pos);
            ok = false;
          } else {
            if (rank_base >= 0) {
              const RankRecord rec = a.rank_records[rank_base + (row >> 5)];
              const uint32_t bit = (uint32_t)row & 31u;
              row = ((rec.bits >> bit) & 1u) ? (int64_t)(rec.before + (uint32_t)__builtin_popcount(rec.bits & ((1u << bit) - 1u))) : -1;
            } else {
              row = a.remap64 ? reinterpret_cast<const int64_t*>(a.remap)[remap_base + row]
                              : (int64_t) reinterpret_cast<const int32_t*>(a.remap)[remap_base + row];
              if (CHECKED) row = checked_entry<index_t>(row);
            }
            ok = row != -1;
          }
        } else if (d.skip_minus_one && row == -1) {
          ok = false;
        }
        if (ok && (row < 0 || row >= row_bound)) {
          if (CHECKED) {
            ++counted;
            row = 0;
          } else {
            report_index(a.status, pos);
            ok = false;
          }
        }
        if (ok) off = row * d.row_stride;
      }
      st_row[tid].off = off;
      StageMul m;
      m.scale = off >= 0 ? wt : -0.0f;
      m.bias = -0.0f;
      if (quant && off >= 0) {
        const uint8_t* p = wbase + off + d.sb_off;
        float s, b;
        load_scale_bias(p, d.sb_fp32 != 0, ((uintptr_t)p & 3) == 0, s, b);
        m.scale = wt * s;
        m.bias = wt * b;
      }
      st_mul[tid] = m;
    }
    load_entry(r0 + cap + tid);
    __syncthreads();
    if (w.size == 16) burst_copy<16, THREADS, LOADS>(first, st_row, rows, w, lds);
    else if (w.size == 4) burst_copy<4, THREADS, LOADS>(first, st_row, rows, w, lds);
    else burst_copy<1, THREADS, LOADS>(first, st_row, rows, w, lds);
    __syncthreads();
    if (mine) {
#define FBGEMM_AMD_BURST_SUM(TY) \
  case TY: burst_sum<TY, K, UNROLL>(acc, lds + at, w.pitch, shift, st_mul, rows, a.fp8_shift, a.fp8_mult); break;
      switch (d.ty) {
        FBGEMM_AMD_BURST_SUM(ST_INT4)
        FBGEMM_AMD_BURST_SUM(ST_INT8)
        FBGEMM_AMD_BURST_SUM(ST_FP16)
        FBGEMM_AMD_BURST_SUM(ST_INT2)
        FBGEMM_AMD_BURST_SUM(ST_FP32)
        FBGEMM_AMD_BURST_SUM(ST_BF16)
        FBGEMM_AMD_BURST_SUM(ST_FP8)
        default: break;
      }
#undef FBGEMM_AMD_BURST_SUM
    }
    if (r0 + cap < n) __syncthreads(); // the staged rows are free again
  }
  if (CHECKED && counted && a.warning && blockIdx.z == 0) status_count(a.status, counted);
  if (a.normalize && n > 0) {
    const float inv = 1.0f / (float)n;
#pragma unroll
    for (int e = 0; e < K; ++e) acc[e] *= inv;
  }
  if (mine) burst_store<K>(a, acc, (int64_t)bag * a.out_stride + d.out_col + col0 + lane_col, cols - lane_col);
}

// Defines the launcher of the instances for one index type. 16 bytes of LDS more than the rows take:
// a lane past the last column of a shifted piece reads up to 12 bytes behind it.
#define FBGEMM_AMD_DEFINE_LOOKUP_BURST_LAUNCH(FN, INDEX_T)                                                  \
  hipError_t FN(const LookupArgs& a, dim3 grid, bool four_waves, int lds_bytes, hipStream_t stream) {       \
    const unsigned lds = (unsigned)((four_waves ? 256 : 64) * (sizeof(StageRow) + sizeof(StageMul)) + lds_bytes + 16); \
    if (a.check_rows) {                                                                                     \
      if (four_waves) hipLaunchKernelGGL((lookup_burst_kernel<INDEX_T, 4, true, false>), grid, dim3(256), lds, stream, a, lds_bytes); \
      else hipLaunchKernelGGL((lookup_burst_kernel<INDEX_T, 1, true, false>), grid, dim3(64), lds, stream, a, lds_bytes); \
    } else if (a.lengths) {                                                                                 \
      if (four_waves) hipLaunchKernelGGL((lookup_burst_kernel<INDEX_T, 4, false, true>), grid, dim3(256), lds, stream, a, lds_bytes); \
      else hipLaunchKernelGGL((lookup_burst_kernel<INDEX_T, 1, false, true>), grid, dim3(64), lds, stream, a, lds_bytes); \
    } else if (four_waves) {                                                                                \
      hipLaunchKernelGGL((lookup_burst_kernel<INDEX_T, 4, false, false>), grid, dim3(256), lds, stream, a, lds_bytes); \
    } else {                                                                                                \
      hipLaunchKernelGGL((lookup_burst_kernel<INDEX_T, 1, false, false>), grid, dim3(64), lds, stream, a, lds_bytes); \
    }                                                                                                       \
    return hipGetLastError();                                                                               \
  }

} // namespace fbgemm_amd
