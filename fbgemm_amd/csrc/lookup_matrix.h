// The pooled lookup on the matrix cores: unweighted bags of 4- and 8-bit rows in the tolerance-grade mode.
//
// A bag's sum is sum(scale * q) + sum(bias) per column: a product of a matrix of scales and a matrix of small integers. A
// wave owns eight consecutive bags of a table at a time, whose entries are one run of the index array, and takes 16 entries
// as the depth of v_mfma_f32_16x16x32_f16:
//  * B, the rows: lane (g, n) = (lane / 16, lane % 16) holds 4 * W bytes of the rows of entries 4 g .. 4 g + 3, which become
//    pairs of halves of one row in a register: the depth's 32 steps are (entry, half), and no element moves between rows.
//    A nibble in a byte of its own is an 8-bit float (4 exponent bits) of q * 2^-9, so one conversion with the scale 2^9
//    makes two halves of two of them; bytes are put into the mantissa of 1024.0, which is then taken off.
//  * A, the scales: row 2 * bag + half holds the scale of every entry of that bag in that half's place, zero elsewhere, so
//    the two halves of B land in rows of their own. One product more, by ones, adds the biases up.
// A scale is half precision in the row and an integer below 256 exact in half precision: the products are exact, their sums
// are kept in fp32. Against sums in 64 bits, fp32 output of 15 to 100 rows a bag is off by 0.79 to 1.0 of what the lean
// kernel's is. (The integers as half-precision denormals, as the lean kernel has them, cost no conversion but are added with
// up to ten bits less: the matrix cores align sums by the exponent field.) No value of another bag gets in: B is finite whatever the
// rows hold, and 0 * finite adds nothing; infinities and NaN in scales and biases stay in their bag.
//
// Bound by the lines it asks for and the output: 96 tables of 256 4-bit columns x 16 384 bags x 15 (23.6 M rows, 0.8 GB of
// output) take 0.52 ms, 0.45 with the arithmetic and the stores left out. Per 16 of those rows a wave issues 9 matrix
// products (16 cycles each, on a pipe of its own) and 91 vector instructions, the lean kernel 165; and bags need no order,
// since a long one has 16 rows per step and none waits for it. us a forward, lean kernels (the better of the two, with the
// scheduler where the bags are ordered) -> here:
//   104 tables x 16384 x 15, 4-bit, 256 wide (8 of them 2-bit, beside it)   695 -> 545
//   18 x 4571 x 26, fp32 output: 4-bit, 256 wide 73 -> 50, 128 wide 53 -> 32; 8-bit, 128 wide 55 -> 38, 64 wide 45 -> 27
//   46 x 3787 x 2:               4-bit, 256 wide 40 -> 29, 128 wide 29 -> 21; 8-bit, 128 wide 32 -> 25, 64 wide 22 -> 18
//   6 x 7081 x 45, uniform rows: 4-bit, 256 wide 88 -> 85, 128 wide 65 -> 61; 8-bit, 128 wide 84 -> 82, 64 wide 69 -> 60
//
// Rows are loaded with buffer instructions: an entry that adds nothing (past the end, rejected, skipped) has an offset
// past the table, for which the load returns zeros without a request, so no load is under a condition and the waits
// count loads.
#pragma once
#include "lookup_device.h"

namespace fbgemm_amd {

typedef uint32_t matrix_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t matrix_u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 matrix_f16x8 __attribute__((ext_vector_type(8)));
typedef float matrix_f32x4 __attribute__((ext_vector_type(4)));

constexpr int MATRIX_STAGE = 64;               // entries whose row numbers and headers are staged at a time
constexpr uint32_t MATRIX_NO_ROW = 0xffff8000u; // offset of an entry that adds nothing; past every table (MATRIX_TABLE_BYTES)
constexpr int MATRIX_OUT_WORDS = 1024;         // four bags' output
constexpr int MATRIX_LDS_WORDS = 2 * MATRIX_STAGE + MATRIX_OUT_WORDS; // in front of it the row offsets of two stages

// A lane's part of the four rows of its quarter of a block. W = 1: a dword of each. W = 2: rows of 128 bytes are read in
// 16-byte chunks, eight lanes a row (three 64-byte accesses to the L1 a row; in pieces of 8 bytes, whose addresses are not
// merged over more than 8 lanes, five), and lanes n and n + 8 then share chunk n out, see matrix_rows.
template <int W>
__device__ __forceinline__ void matrix_load(uint32_t (&dst)[4 * W], __amdgpu_buffer_rsrc_t rsrc, const uint32_t* off, uint32_t lane_off) {
  if constexpr (W == 1) {
    const matrix_u32x4 o = *reinterpret_cast<const matrix_u32x4*>(off);
#pragma unroll
    for (int j = 0; j < 4; ++j) dst[j] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(o[j] + lane_off), 0, 0);
  } else {
    static_assert(W == 2, "rows of 64 or 128 bytes");
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const matrix_u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(off[2 * k] + lane_off), 0, 0);
#pragma unroll
      for (int w = 0; w < 4; ++w) dst[4 * k + w] = v[w];
    }
  }
}

// What was loaded -> word w of row j of the quarter. W = 2: of two rows, lanes 0 .. 7 have loaded a chunk each of the
// first, lanes 8 .. 15 of the second; the former keep the first two words of their chunk and take those of the second row
// from lane n + 8, which takes the last two of the first.
template <int W>
__device__ __forceinline__ void matrix_rows(const uint32_t (&r)[4 * W], uint32_t (&x)[4][W]) {
  if constexpr (W == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j][0] = r[j];
  } else {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int w = 0; w < 2; ++w) { // row_ror:8 into the upper, the lower half of every 16 lanes
        const int lo = (int)r[4 * k + w], hi = (int)r[4 * k + w + 2];
        x[2 * k][w] = (uint32_t)__builtin_amdgcn_update_dpp(lo, hi, 0x128, 0xf, 0xc, false);
        x[2 * k + 1][w] = (uint32_t)__builtin_amdgcn_update_dpp(hi, lo, 0x128, 0xf, 0x3, false);
      }
  }
}

// Four registers of 16-bit pairs per lane as an operand of the matrix instruction.
__device__ __forceinline__ matrix_f32x4 matrix_fma(const matrix_u32x4& a, const matrix_u32x4& b, const matrix_f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(matrix_f16x8, a), __builtin_bit_cast(matrix_f16x8, b), c, 0, 0, 0);
}

// Two integers below 1024 in the mantissas of 1024.0 -> halves
typedef _Float16 matrix_f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t matrix_halves(uint32_t u) {
  const matrix_f16x2 k = {(_Float16)1024.0f, (_Float16)1024.0f};
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(matrix_f16x2, u) - k);
}

// Lane J of every 16 lanes, in all of them (row_newbcast).
template <int J>
__device__ __forceinline__ uint32_t matrix_bcast(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x150 + J, 0xf, 0xf, true);
}

__device__ __forceinline__ void matrix_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int64_t matrix_readlane64(int64_t v, int lane) {
  return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)v, lane) |
                   ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), lane) << 32));
}

// Bits [lo, hi) of the word that starts at entry `base`.
__device__ __forceinline__ uint32_t matrix_range(int lo, int hi, int base) {
  const int l = min(max(lo - base, 0), 32), h = min(max(hi - base, 0), 32);
  return ((uint32_t)(1ull << h) - 1u) & ~((uint32_t)(1ull << l) - 1u);
}

// ESZ: bytes per output element. The output of four bags at a time goes through LDS, so that every store instruction
// writes runs of consecutive bytes (each lane holds CPL consecutive columns of two bags).
template <int TY, int W, int ESZ>
__device__ __forceinline__ void matrix_store(const LookupArgs& a, const TableDesc& d, int first, int lane, const float (&v)[W * (TY == ST_INT4 ? 8 : 4)],
                                             int which, uint32_t* lds) {
  constexpr int CPL = W * (TY == ST_INT4 ? 8 : 4); // columns per lane
  constexpr int D = 16 * CPL;
  constexpr int PB = CPL * ESZ < 16 ? 8 : 16;      // bytes per piece
  constexpr int NP = CPL * ESZ / PB;               // pieces per lane and bag
  static_assert(4 * D * ESZ <= MATRIX_OUT_WORDS * 4, "the output of four bags");
  uint32_t w[CPL * ESZ / 4];
  if constexpr (ESZ == 4) {
#pragma unroll
    for (int e = 0; e < CPL; ++e) w[e] = float_to_bits(v[e]);
  } else if (a.out_ty == ST_BF16) {
#pragma unroll
    for (int e = 0; e < CPL; e += 2) w[e / 2] = pack_bf16x2(v[e], v[e + 1]);
  } else {
#pragma unroll
    for (int e = 0; e < CPL; e += 2) w[e / 2] = pack_half2(v[e], v[e + 1]);
  }
  // W = 2: lane n holds the first half of chunk n % 8 of the row, or (n / 8 = 1) the second
  const int at = W == 1 ? lane : (lane & 48) + 2 * (lane & 7) + ((lane >> 3) & 1);
  if constexpr (NP > 1) {
#pragma unroll
    for (int q = 0; q < NP; ++q)
      *reinterpret_cast<uint4*>(lds + (at * NP + q) * 4) = make_uint4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
    matrix_lds_sync();
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const uint4 p = *reinterpret_cast<const uint4*>(lds + (lane + 64 * q) * 4);
      w[4 * q] = p.x;
      w[4 * q + 1] = p.y;
      w[4 * q + 2] = p.z;
      w[4 * q + 3] = p.w;
    }
    matrix_lds_sync();
  }
  uint8_t* const out = reinterpret_cast<uint8_t*>(a.out) + (int64_t)d.out_col * ESZ;
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    const int piece = NP > 1 ? lane + 64 * q : at;
    const int bag = first + 2 * (piece / (16 * NP)) + which;
    if (bag < a.B) {
      uint8_t* p = out + (int64_t)bag * a.out_stride * ESZ + (piece % (16 * NP)) * PB;
      if constexpr (PB == 16) stream_store16(p, w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
      else stream_store8(p, w[0], w[1]);
    }
  }
}

// W: dwords of a row per lane. The rows hold exactly 64 * W bytes of elements.
//
// A wave pools a.wave_bags bags, eight at a time, as one pipeline over stages of 64 entries: while one stage is added up, the
// rows of the next are asked for block by block, as registers get free, and the indices of the one after it; the next eight
// bags' first stage follows the last one of these eight without a gap.
template <typename index_t, int TY, int W>
__device__ __forceinline__ void pool_matrix(const LookupArgs& a, const TableDesc& d, int table, int first, int lane, uint32_t* lds) {
  constexpr int CPW = TY == ST_INT4 ? 8 : 4; // columns per word
  constexpr int PAIRS = CPW / 2;
  constexpr int DEPTH = 2;                   // blocks of 16 rows in flight; 4 take the registers of the fourth wave (593 -> 638 us)
  const int g = lane >> 4, n = lane & 15;    // lane n is row n of A: bag n / 2 of the eight, half n % 2

  // lane l holds where bag l of the wave starts, and its length
  const int bags = a.B - first < a.wave_bags ? a.B - first : a.wave_bags;
  int64_t o0 = 0;
  int len = 0;
  bool bad = false;
  if (lane < bags) {
    const int64_t ob = (int64_t)table * a.B + first + lane;
    o0 = read_offset(a.offsets, a.off64, ob);
    const int64_t o1 = read_offset(a.offsets, a.off64, ob + 1);
    const int64_t l = o1 - o0;
    bad = l < 0 || l > MATRIX_MAX_RUN || o0 < 0 || o1 > a.index_size;
    if (bad) report(a.status, l < 0 ? ERR_NEGATIVE_LENGTH : ERR_BAG_OVERRUN);
    else len = (int)l;
  }
  const int64_t p0 = matrix_readlane64(o0, 0);
  // the entries of eight bags are one run; where an offset is not in order, each bag is one
  const bool together = __builtin_amdgcn_ballot_w64(bad) == 0ull && matrix_readlane64(o0 + len, bags - 1) - p0 <= MATRIX_MAX_RUN;
  const int per_eight = together ? 1 : 8;
  const int runs = (bags + 7) / 8 * per_eight;
  const int start = (int)(o0 - p0); // together only

  const uint8_t* const base = (d.placement ? a.weights[1] : a.weights[0]) + d.weights_offset;
  const uint32_t stride = (uint32_t)d.row_stride;
  const __amdgpu_buffer_rsrc_t table_rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, (int)(uint32_t)(d.num_rows * d.row_stride), 0x00020000);
  const uint32_t lane_off = (uint32_t)d.data_off + (W == 1 ? (uint32_t)n * 4 : (uint32_t)(n & 7) * 16);
  const uint32_t sb_off = (uint32_t)d.sb_off;

  uint32_t* const st_off = lds; // [2][64] byte offset of the entry's row
  const uint32_t* const hdr_off = st_off + 4 * g + (n & 3);
  const uint32_t scale_sel = n & 1 ? 0x05040c0cu : 0x0c0c0504u; // the scale, from the low half into the lane's half
  const uint32_t* const my_off = st_off + 4 * g + (W == 1 ? 0 : n >> 3);

  matrix_f32x4 acc[W][PAIRS], bsum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int w = 0; w < W; ++w)
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) acc[w][p] = bsum;
  matrix_u32x4 ones = {0x3c000000u, 0x3c000000u, 0x3c000000u, 0x3c000000u};
  asm("" : "+v"(ones)); // kept in registers: made again for every block otherwise
  uint32_t raw[DEPTH][4 * W], hdr[DEPTH]; // lane n of a quarter holds the header of its row n % 4
  int64_t bad_pos = INT64_MAX;

  // A stage: 64 entries of a run, wave-uniform. Every run has one at least.
  struct Stage {
    int run;      // `runs`: behind the last one, without entries
    int64_t from; // position of the stage's first entry
    int left;     // entries of the run from here on
  };
  auto begin_run = [&](int run) {
    Stage s;
    s.run = run;
    s.from = p0;
    s.left = 0;
    if (run >= runs) return s;
    const int b = together ? run * 8 : run;
    if (b >= bags) return s;
    if (together) {
      const int e = b + 8 < bags ? b + 7 : bags - 1, at = __builtin_amdgcn_readlane(start, b);
      s.from = p0 + at;
      s.left = __builtin_amdgcn_readlane(start + len, e) - at;
    } else {
      s.from = matrix_readlane64(o0, b);
      s.left = __builtin_amdgcn_readlane(len, b);
    }
    return s;
  };
  auto next_stage = [&](const Stage& s) {
    if (s.left <= MATRIX_STAGE) return begin_run(s.run < runs ? s.run + 1 : runs);
    Stage t = s;
    t.from += MATRIX_STAGE;
    t.left -= MATRIX_STAGE;
    return t;
  };

  int64_t row = 0;
  auto load_index = [&](const Stage& s) { // one entry per lane; zeros past the end
    const int cnt = min(max(s.left, 0), MATRIX_STAGE);
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<index_t*>(reinterpret_cast<const index_t*>(a.indices)) + s.from, 0, cnt * (int)sizeof(index_t), 0x00020000);
    if constexpr (sizeof(index_t) == 8) {
      const matrix_u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, lane * 8, 0, 0);
      row = (int64_t)((uint64_t)v.x | ((uint64_t)v.y << 32));
    } else {
      row = (int64_t)(int32_t)__builtin_amdgcn_raw_buffer_load_b32(r, lane * 4, 0, 0);
    }
  };
  auto stage_rows = [&](const Stage& s, int buf) { // indices that have arrived -> row offsets
    const bool here = lane < s.left, valid = (uint64_t)row < (uint64_t)d.num_rows;
    const uint32_t off = here && valid ? (uint32_t)row * stride : MATRIX_NO_ROW;
    const uint64_t rejected = __builtin_amdgcn_ballot_w64(here && !valid && !(d.skip_minus_one && row == -1));
    if (rejected != 0ull) { // remembered by the wave and reported once its loop is over: an atomic in it would make its waits waits for everything
      const int64_t pos = s.from + (int64_t)__builtin_ctzll(rejected);
      bad_pos = pos < bad_pos ? pos : bad_pos;
    }
    st_off[buf + lane] = off;
  };
  // a row's header together with the row, whose first line it shares: asked for a stage earlier, the line was often gone
  // from the L1 again (12 % more requests to L2 where rows recur, one more for two where they don't)
  auto issue = [&](uint32_t (&r)[4 * W], uint32_t& h, int buf, int blk) {
    h = __builtin_amdgcn_raw_buffer_load_b32(table_rsrc, (int)(hdr_off[buf + blk * 16] + sb_off), 0, 0);
    matrix_load<W>(r, table_rsrc, my_off + buf + blk * 16, lane_off);
  };
  // mask: bit 16 * (blk % 2) + j: entry 4 g + j of the block is the bag's
  auto add = [&](const uint32_t (&r)[4 * W], uint32_t h, int blk, uint32_t mask) {
    matrix_u32x4 as, ab;
    const uint32_t hs[4] = {matrix_bcast<0>(h), matrix_bcast<1>(h), matrix_bcast<2>(h), matrix_bcast<3>(h)};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t in = hs[j] & (uint32_t)__builtin_amdgcn_sbfe((int)mask, (blk & 1) * 16 + j, 1);
      as[j] = __builtin_amdgcn_perm(in, 0u, scale_sel);
      ab[j] = in & 0xffff0000u;
    }
    bsum = matrix_fma(ab, ones, bsum);
    uint32_t rows[4][W];
    matrix_rows<W>(r, rows);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      matrix_u32x4 b[PAIRS];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t x = rows[j][w];
        if constexpr (TY == ST_INT4) {
          const uint32_t e = x & 0x0f0f0f0fu, o = (x >> 4) & 0x0f0f0f0fu;
          b[0][j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(e, 512.0f, false)); // columns 0, 2
          b[1][j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(o, 512.0f, false)); // columns 1, 3
          b[2][j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(e, 512.0f, true));  // columns 4, 6
          b[3][j] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(o, 512.0f, true));  // columns 5, 7
        } else {
          b[0][j] = matrix_halves(__builtin_amdgcn_perm(0x64646464u, x, 0x04010400u));
          b[1][j] = matrix_halves(__builtin_amdgcn_perm(0x64646464u, x, 0x04030402u));
        }
      }
#pragma unroll
      for (int p = 0; p < PAIRS; ++p) acc[w][p] = matrix_fma(as, b[p], acc[w][p]);
      __builtin_amdgcn_sched_barrier(0); // one word's integers at a time in registers
    }
  };

  Stage cur = begin_run(0), next = next_stage(cur);
  load_index(cur);
  stage_rows(cur, 0);
  load_index(next);
  matrix_lds_sync();
#pragma unroll
  for (int k = 0; k < DEPTH; ++k) issue(raw[k], hdr[k], 0, k);
  int buf = 0;
  int lo = 0, hi = 0; // the entries of the lane's bag, counted from the stage's first
  bool fresh = true;  // `cur` is the first stage of a run
  while (cur.run < runs) {
    const Stage after = next_stage(next);
    stage_rows(next, buf ^ MATRIX_STAGE);
    load_index(after);
    matrix_lds_sync();
    if (fresh) {
      if (together) {
        const int b = cur.run * 8 + (n >> 1);
        lo = __shfl(start, b, 64) - (int)(cur.from - p0);
        hi = lo + __shfl(len, b, 64); // lanes past the wave's last bag hold no length
      } else {
        lo = 0;
        hi = (cur.run & 7) == (n >> 1) ? cur.left : 0;
      }
    }
    const uint32_t m0 = matrix_range(lo, hi, 0) >> (4 * g), m1 = matrix_range(lo, hi, 32) >> (4 * g);
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
      if (16 * blk < cur.left) add(raw[blk % DEPTH], hdr[blk % DEPTH], blk, blk < 2 ? m0 : m1);
      issue(raw[blk % DEPTH], hdr[blk % DEPTH], blk + DEPTH < 4 ? buf : buf ^ MATRIX_STAGE, (blk + DEPTH) % 4);
      __builtin_amdgcn_sched_barrier(0);
    }
    matrix_lds_sync();
    fresh = next.run != cur.run;
    lo -= MATRIX_STAGE;
    hi -= MATRIX_STAGE;
    if (fresh && next.run % per_eight == 0) { // the last stage of eight bags
      // lane (g, n) holds columns n * CPL .. of bags 2 g and 2 g + 1: sums 2 * which + half
      const int eight = cur.run / per_eight * 8;
#pragma unroll
      for (int which = 0; which < 2; ++which) {
        float v[W * CPW];
#pragma unroll
        for (int w = 0; w < W; ++w)
#pragma unroll
          for (int p = 0; p < PAIRS; ++p)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int c = TY == ST_INT4 ? 8 * w + 4 * (p >> 1) + (p & 1) + 2 * h : 4 * w + 2 * p + h;
              v[c] = acc[w][p][2 * which + h] + bsum[2 * which];
            }
        if (a.normalize) {
          const int m = __shfl(len, eight + 2 * g + which, 64);
          const float inv_len = m > 0 ? 1.0f / (float)m : 1.0f;
#pragma unroll
          for (int c = 0; c < W * CPW; ++c) v[c] *= inv_len;
        }
        if (a.out_ty == ST_FP32) matrix_store<TY, W, 4>(a, d, first + eight, lane, v, which, lds + 2 * MATRIX_STAGE);
        else matrix_store<TY, W, 2>(a, d, first + eight, lane, v, which, lds + 2 * MATRIX_STAGE);
      }
      bsum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int w = 0; w < W; ++w)
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) acc[w][p] = bsum;
    }
    buf ^= MATRIX_STAGE;
    cur = next;
    next = after;
  }
  if (bad_pos != INT64_MAX && lane == 0) report_index(a.status, bad_pos);
}

// One wave per workgroup, work list and workgroup -> XCD mapping as in the other lookup kernels. Every table of a launch has
// the same row type and width.
template <typename index_t, int TY, int W>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void lookup_matrix_kernel(const LookupArgs a) {
  __shared__ __attribute__((aligned(16))) uint32_t lds[MATRIX_LDS_WORDS];
  const int xb = blockIdx.x & 7;
  const int64_t w = (int64_t)(blockIdx.x >> 3);
  const int64_t start = a.xcd_start[xb];
  if (w >= a.xcd_start[xb + 1] - start) return;
  const WaveWork ww = a.work[start + w];
  const TableDesc d = a.tables[ww.table];
  pool_matrix<index_t, TY, W>(a, d, ww.table, ww.first_bag, (int)threadIdx.x, lds);
}

#define FBGEMM_AMD_DEFINE_MATRIX_LAUNCH(FN, INDEX_T)                                                                          \
  hipError_t FN(const LookupArgs& a, bool int4, bool wide, unsigned blocks, hipStream_t stream) {                             \
    if (int4 && wide) hipLaunchKernelGGL((lookup_matrix_kernel<INDEX_T, ST_INT4, 2>), dim3(blocks), dim3(64), 0, stream, a);  \
    else if (int4) hipLaunchKernelGGL((lookup_matrix_kernel<INDEX_T, ST_INT4, 1>), dim3(blocks), dim3(64), 0, stream, a);     \
    else if (wide) hipLaunchKernelGGL((lookup_matrix_kernel<INDEX_T, ST_INT8, 2>), dim3(blocks), dim3(64), 0, stream, a);     \
    else hipLaunchKernelGGL((lookup_matrix_kernel<INDEX_T, ST_INT8, 1>), dim3(blocks), dim3(64), 0, stream, a);               \
    return hipGetLastError();                                                                                                 \
  }

} // namespace fbgemm_amd
