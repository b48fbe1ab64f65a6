// gfx950 kernel of PoolingMode.NONE for rows on 16-byte boundaries (what the table-batched layout
// gives at its usual row alignment) and output in whole 16-byte pieces; everything else takes
// sequence_lookup_kernel (sequence_kernels.hip), which says what the mode computes.
//
// What bounds it is the traffic: a row's lines in, D elements out. A wave takes 4, 16 or 32 consecutive
// positions (fewer where its LDS holds fewer rows), in segments of one table. A lane per position turns its index into a row offset; the
// wave then copies those rows, headers included, as consecutive 16-byte pieces into LDS, all of a
// lane's pieces in flight at once (2.5 KB a wave for 32 rows of 4 bits x 128, where four rows per
// group of lanes are 1 KB). The decoding lanes take the output's 16-byte pieces in order, so that a
// store instruction writes 1 KB in a row whatever the width, and unpack through half-precision
// denormals as the pooled kernels do: 52 vector instructions per piece, all told, where
// sequence_lookup_kernel spends 174. Waves of one segment and no more: a grid of resident waves that fetched the next rows
// behind the current ones took 300 us where this takes 281.
//   32 tables x 1 M rows of 4 bits x 128, 3.5 M positions to fp16: 431 -> 281 us; to fp32 453 us;
//   4-bit, 8-bit and fp16 tables mixed 440 -> 315 us; 442 368 positions 56 -> 23 us, 65 536 14.8 -> 6.8.
// Over 278 forwards of all row types but bf16, 8 to 4000 columns, to fp16 and fp32, 2 to 262 144 positions, it takes 0.63
// of sequence_lookup_kernel's time on average and 0.98 at most: 262 144 positions of fp32 x 256 to fp32 105.6 -> 93.7,
// of 4 bits x 512 to fp32 114.4 -> 109.3; 8192 of 2 bits x 4000 to fp32 35.5 -> 28.3; 4096 of 4 bits x 8 to fp16 7.0 -> 3.6.
#include <hip/hip_runtime.h>

#include "launchers.h"
#include "lookup_device.h"

namespace fbgemm_amd {

namespace {

constexpr int SS_WAVES = 4;             // per workgroup
constexpr int SS_PAD = 64;              // a run of a row's last columns may be read past its last piece
constexpr int ss_wave_bytes(int steps) { return steps * 1024 + SS_PAD + 64 * (int)sizeof(int64_t); }

typedef stream_u32x4 Piece;

struct StreamArgs {
  const TableDesc* tables;
  const uint8_t* weights[2];
  const void* indices;
  const void* offsets;
  void* out;
  Status* status;
  int64_t total_L;
  int64_t chunks; // of `rows` positions
  int32_t is64;   // indices and offsets are int64 (else int32)
  int32_t B, T, D;
  int32_t rows;   // positions a wave takes at a time, at most 64; rows * pieces of a row <= 64 STEPS
  int32_t fp8_shift;
  float fp8_mult;
};

// BYTES of LDS from `p` (4-byte aligned from 4 on, 2-byte for 2) into w[], little end first
template <int BYTES>
__device__ __forceinline__ void run_words(const uint8_t* p, uint32_t (&w)[8]) {
  if constexpr (BYTES == 1) w[0] = *p;
  else if constexpr (BYTES == 2) w[0] = *reinterpret_cast<const uint16_t*>(p);
  else {
#pragma unroll
    for (int i = 0; i < BYTES / 4; ++i) w[i] = reinterpret_cast<const uint32_t*>(p)[i];
  }
}

// Columns [run * C, run * C + C) of a row in LDS, as a bag of one (see sequence_kernels.hip): fma(scale, q, 0 + bias)
// for quantised rows, fma(1, x, 0) for the others. The table-batched header is two halfs, so scale * 2^24 cannot overflow.
template <int TY, int C>
__device__ __forceinline__ void run_values(const uint8_t* row, int run, int fp8_shift, float fp8_mult, float (&v)[C]) {
  constexpr int bits = type_bits(TY);
  constexpr bool quant = TY == ST_INT8 || TY == ST_INT4 || TY == ST_INT2;
  constexpr int run_bytes = C * bits / 8;
  uint32_t w[8];
  run_words<run_bytes>(row + (quant ? 4 : 0) + run * run_bytes, w);
  float scale = 1.0f, bias = 0.0f;
  if constexpr (quant) {
    const uint32_t hdr = *reinterpret_cast<const uint32_t*>(row);
    scale = half_lo(hdr);
    bias = 0.0f + half_hi(hdr);
  }
  if constexpr (TY == ST_INT4) {
    const float s24 = scale * 0x1p24f, s20 = scale * 0x1p20f;
    const uint32_t a0 = w[0] & 0x000f000fu, a1 = w[0] & 0x00f000f0u; // nibbles 0, 4 and 1, 5 (times 16)
    const uint32_t a2 = (w[0] >> 8) & 0x000f000fu, a3 = (w[0] >> 8) & 0x00f000f0u;
    v[0] = __builtin_fmaf(s24, half_lo(a0), bias);
    v[1] = __builtin_fmaf(s20, half_lo(a1), bias);
    v[2] = __builtin_fmaf(s24, half_lo(a2), bias);
    v[3] = __builtin_fmaf(s20, half_lo(a3), bias);
    if constexpr (C == 8) {
      v[4] = __builtin_fmaf(s24, half_hi(a0), bias);
      v[5] = __builtin_fmaf(s20, half_hi(a1), bias);
      v[6] = __builtin_fmaf(s24, half_hi(a2), bias);
      v[7] = __builtin_fmaf(s20, half_hi(a3), bias);
    }
  } else if constexpr (TY == ST_INT8) {
    const float s24 = scale * 0x1p24f;
#pragma unroll
    for (int i = 0; i < C / 4; ++i) {
      const uint32_t lo = __builtin_amdgcn_perm(0u, w[i], 0x0c010c00u), hi = __builtin_amdgcn_perm(0u, w[i], 0x0c030c02u);
      v[4 * i] = __builtin_fmaf(s24, half_lo(lo), bias);
      v[4 * i + 1] = __builtin_fmaf(s24, half_hi(lo), bias);
      v[4 * i + 2] = __builtin_fmaf(s24, half_lo(hi), bias);
      v[4 * i + 3] = __builtin_fmaf(s24, half_hi(hi), bias);
    }
  } else {
#pragma unroll
    for (int k = 0; k < C; ++k) {
      if constexpr (TY == ST_INT2) v[k] = __builtin_fmaf(scale, (float)((w[0] >> (2 * k)) & 3u), bias);
      else if constexpr (TY == ST_FP32) v[k] = __builtin_fmaf(1.0f, bits_to_float(w[k]), 0.0f);
      else if constexpr (TY == ST_FP16) v[k] = __builtin_fmaf(1.0f, (k & 1) ? half_hi(w[k / 2]) : half_lo(w[k / 2]), 0.0f);
      else if constexpr (TY == ST_BF16) v[k] = __builtin_fmaf(1.0f, bits_to_float((k & 1) ? w[k / 2] & 0xffff0000u : w[k / 2] << 16), 0.0f);
      else {
        const uint32_t b = (w[k / 4] >> (8 * (k % 4))) & 0xffu;
        const float mag = bits_to_float((b & 0x7fu) << fp8_shift) * fp8_mult;
        v[k] = __builtin_fmaf(1.0f, bits_to_float(float_to_bits(mag) | ((b & 0x80u) << 24)), 0.0f);
      }
    }
  }
}

// Rows 0 .. n-1 from LDS to the output, a 16-byte piece per lane and step. Bit r of `ok`: row r is there (else zeros).
template <int TY, int OUT_TY>
__device__ __forceinline__ void write_rows(const uint8_t* lds, int pitch, int n, uint64_t ok, int D, uint8_t* out, int lane,
                                           int fp8_shift, float fp8_mult) {
  constexpr int C = OUT_TY == ST_FP32 ? 4 : 8; // columns of an output piece
  const int R = D / C, total = n * R;
  int row = lane / R, run = lane - row * R;
  const int row_step = 64 / R, run_step = 64 - row_step * R;
  const bool all = (ok | (n < 64 ? ~0ull << n : 0ull)) == ~0ull;
  auto piece = [&](int q) {
    float v[C];
    run_values<TY, C>(lds + row * pitch, run, fp8_shift, fp8_mult, v);
    if (!all && !((ok >> row) & 1)) {
#pragma unroll
      for (int k = 0; k < C; ++k) v[k] = 0.0f;
    }
    uint8_t* o = out + (uint32_t)q * 16u;
    if constexpr (OUT_TY == ST_FP32) stream_store16(o, v[0], v[1], v[2], v[3]);
    else if constexpr (OUT_TY == ST_FP16) stream_store16(o, pack_half2(v[0], v[1]), pack_half2(v[2], v[3]), pack_half2(v[4], v[5]), pack_half2(v[6], v[7]));
    else stream_store16(o, pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
    row += row_step;
    run += run_step;
    if (run >= R) {
      run -= R;
      ++row;
    }
  };
  const int full = total >> 6;
#pragma unroll 4
  for (int s = 0; s < full; ++s) piece(s * 64 + lane);
  if (full * 64 + lane < total) piece(full * 64 + lane);
}

__device__ __forceinline__ void wave_lds_order() { // a wave's LDS operations complete in order: this keeps the compiler to it
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int OUT_TY, int STEPS>
__global__ __launch_bounds__(64 * SS_WAVES) void sequence_stream_kernel(StreamArgs a) {
  __shared__ __align__(16) uint8_t smem[SS_WAVES][ss_wave_bytes(STEPS)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint8_t* rows_lds = smem[wave];
  int64_t* off_lds = reinterpret_cast<int64_t*>(rows_lds + STEPS * 1024 + SS_PAD);
  // Workgroup b runs on XCD b % 8: each XCD takes an eighth of the positions, and with it of the tables.
  const int64_t per_xcd = (a.chunks + 7) / 8;
  const int64_t in_xcd = (int64_t)(blockIdx.x >> 3) * SS_WAVES + wave;
  const int64_t chunk = (int64_t)(blockIdx.x & 7) * per_xcd + in_xcd;
  if (in_xcd >= per_xcd || chunk >= a.chunks) return;
  int64_t p = chunk * a.rows;
  const int64_t chunk_end = p + a.rows < a.total_L ? p + a.rows : a.total_L;
  // positions [p, p + n) of one table at a time
  for (int n; p < chunk_end; p += n) {
    const int64_t idx = p + lane < chunk_end ? read_offset(a.indices, a.is64, p + lane) : -1;
    // the largest t whose first position is at or before p, 64 tables a step
    int lo = 0, hi = a.T;
    while (hi - lo > 1) {
      const int step = (hi - lo + 63) >> 6, t = lo + lane * step;
      const bool at = lane == 0 || (t < hi && read_offset(a.offsets, a.is64, (int64_t)t * a.B) <= p);
      lo += (__popcll(__ballot(at)) - 1) * step;
      hi = lo + step < hi ? lo + step : hi;
    }
    // what lies behind the last table is its own; a wave goes on even where offsets decrease
    const int64_t t_end = lo + 1 < a.T ? read_offset(a.offsets, a.is64, (int64_t)(lo + 1) * a.B) : a.total_L;
    const int64_t left = (t_end < chunk_end ? t_end : chunk_end) - p;
    n = left < 1 ? 1 : (int)left;
    const TableDesc& d = a.tables[lo];
    const bool live = lane < n;
    const bool there = live && idx >= 0 && idx < d.num_rows;
    if (live && !there && idx != -1) report_index(a.status, p + lane);
    const uint64_t ok = __ballot(there);
    const int P = (d.data_off + d.data_bytes + 15) >> 4;
    if (ok != 0) {
      // a position without a row copies one that another has
      const int64_t off = idx * d.row_stride;
      const int first = __ffsll((unsigned long long)ok) - 1;
      const uint32_t off_lo = __builtin_amdgcn_readlane((uint32_t)off, first), off_hi = __builtin_amdgcn_readlane((uint32_t)((uint64_t)off >> 32), first);
      off_lds[lane] = there ? off : (int64_t)((uint64_t)off_hi << 32 | off_lo);
      wave_lds_order();
      const uint8_t* base = (d.placement ? a.weights[1] : a.weights[0]) + d.weights_offset;
      const int last = n * P - 1;
      const int recip = (65536 + P - 1) / P; // k / P == k * recip >> 16 for k < 512, P <= 64
      Piece piece[STEPS];
#pragma unroll
      for (int k = 0; k < STEPS; ++k) {
        const int q = k * 64 + lane < last ? k * 64 + lane : last;
        const int r = (q * recip) >> 16, part = q - r * P;
        piece[k] = *reinterpret_cast<const Piece*>(base + off_lds[r] + part * 16);
      }
#pragma unroll
      for (int k = 0; k < STEPS; ++k) *reinterpret_cast<Piece*>(rows_lds + (k * 64 + lane) * 16) = piece[k];
      wave_lds_order();
    }
    uint8_t* out = reinterpret_cast<uint8_t*>(a.out) + p * (a.D * (OUT_TY == ST_FP32 ? 4 : 2));
    switch (d.ty) {
      case ST_INT4: write_rows<ST_INT4, OUT_TY>(rows_lds, P * 16, n, ok, a.D, out, lane, 0, 0.0f); break;
      case ST_INT8: write_rows<ST_INT8, OUT_TY>(rows_lds, P * 16, n, ok, a.D, out, lane, 0, 0.0f); break;
      case ST_FP16: write_rows<ST_FP16, OUT_TY>(rows_lds, P * 16, n, ok, a.D, out, lane, 0, 0.0f); break;
      case ST_INT2: write_rows<ST_INT2, OUT_TY>(rows_lds, P * 16, n, ok, a.D, out, lane, 0, 0.0f); break;
      case ST_FP32: write_rows<ST_FP32, OUT_TY>(rows_lds, P * 16, n, ok, a.D, out, lane, 0, 0.0f); break;
      case ST_BF16: write_rows<ST_BF16, OUT_TY>(rows_lds, P * 16, n, ok, a.D, out, lane, 0, 0.0f); break;
      case ST_FP8: write_rows<ST_FP8, OUT_TY>(rows_lds, P * 16, n, ok, a.D, out, lane, a.fp8_shift, a.fp8_mult); break;
      default: break;
    }
    wave_lds_order(); // read before the next rows are written
  }
}

template <int OUT_TY, int STEPS>
hipError_t launch_stream(const StreamArgs& a, hipStream_t stream) {
  const int64_t blocks = ((a.chunks + 7) / 8 + SS_WAVES - 1) / SS_WAVES * 8;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((sequence_stream_kernel<OUT_TY, STEPS>), dim3((unsigned)blocks), dim3(64 * SS_WAVES), 0, stream, a);
  return hipGetLastError();
}

template <int OUT_TY>
hipError_t launch_stream_steps(const StreamArgs& a, int steps, hipStream_t stream) {
  if (steps <= 3) return launch_stream<OUT_TY, 3>(a, stream);
  if (steps <= 5) return launch_stream<OUT_TY, 5>(a, stream);
  return launch_stream<OUT_TY, 8>(a, stream);
}

} // namespace

hipError_t launch_sequence_stream(const TableDesc* tables, const uint8_t* w0, const uint8_t* w1, const void* indices, bool idx64,
                                  const void* offsets, int32_t B, int32_t T, int64_t total_L, int32_t D, int32_t out_ty, void* out,
                                  int32_t max_pieces, int32_t fp8_shift, float fp8_mult, Status* status, hipStream_t stream) {
  if (total_L <= 0 || D <= 0) return hipSuccess;
  if (!sequence_stream_takes(D, out_ty, out, max_pieces)) return hipErrorInvalidValue;
  // Positions a wave takes. Rows in flight pay from 65 536 positions on (655 360 of 4 bits x 128 from 32 tables to fp16: 33.3 us
  // with 16 a wave, 31.6 with 32, 34.1 with 64); below, more waves do (65 536 from 16 tables to fp16 7.3 us with 32, 6.8 with 16);
  // and a wave goes through the tables of its positions one after the other (2 positions in each of 96 tables: 27.1 us with 32,
  // 7.5 with 4, and 10.3 in sequence_lookup_kernel).
  int rows = total_L / 16 < T ? 4 : (total_L < 65536 ? 16 : 32);
  int steps = (rows * max_pieces + 63) / 64;
  steps = steps <= 3 ? 3 : (steps <= 5 ? 5 : 8);
  if (rows * max_pieces > steps * 64) rows = steps * 64 / max_pieces; // 8 or more: a row has at most 64 pieces
  const StreamArgs a{tables, {w0, w1}, indices, offsets, out, status, total_L, (total_L + rows - 1) / rows, idx64 ? 1 : 0, B, T, D, rows,
                     fp8_shift, fp8_mult};
  if (out_ty == ST_FP32) return launch_stream_steps<ST_FP32>(a, steps, stream);
  if (out_ty == ST_FP16) return launch_stream_steps<ST_FP16>(a, steps, stream);
  return launch_stream_steps<ST_BF16>(a, steps, stream);
}

} // namespace fbgemm_amd
