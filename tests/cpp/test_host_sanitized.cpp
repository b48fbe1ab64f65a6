// The host side of the library (fbgemm_amd/csrc/c_api.cpp: plans, work-list cache, per-stream
// and per-thread scratch, the static scratch of the entry point that allocates nothing) driven
// on the CPU against the HIP stand-in of tests/cpp/hip_stub, built with
// -fsanitize=address,undefined. The sanitizers are the checker: a use after free, a double
// free, an overrun or a leak of "device" or host memory ends the program with a report. The
// scenarios are the lifetimes that have broken before: plan creation failing half-way, pruned-
// row mappings set twice, eviction from the work-list cache with entries a graph may hold,
// trimming, scratch handed from a host thread that has ended to a new one, split bags, the 8-bit
// pooled output, allocation failures at every point of a first forward.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "../../include/fbgemm_amd.h"
#include "../../fbgemm_amd/csrc/launchers.h"
#include "../../fbgemm_amd/csrc/lookup_common.h"
#include "../../include/fbgemm_amd_bench.h"

#define CHECK(cond)                                                         \
  do {                                                                      \
    if (!(cond)) {                                                          \
      printf("FAILED %s:%d: %s (%s)\n", __FILE__, __LINE__, #cond, fbgemm_amd_last_error()); \
      exit(1);                                                              \
    }                                                                       \
  } while (0)

namespace {

struct Problem {
  int32_t T;
  std::vector<int64_t> wo;
  std::vector<uint8_t> tys;
  std::vector<int32_t> D_offsets;
  int64_t bytes;
};

// int4 / int8 / fp16 / int2 tables of a few rows each (sizes only: no kernel reads them here)
Problem make_problem(int32_t T) {
  Problem p;
  p.T = T;
  const int32_t Ds[4] = {64, 128, 256, 32};
  const uint8_t tys[4] = {3, 2, 1, 4};
  int64_t off = 0;
  p.D_offsets.push_back(0);
  for (int t = 0; t < T; ++t) {
    p.wo.push_back(off);
    p.tys.push_back(tys[t % 4]);
    p.D_offsets.push_back(p.D_offsets.back() + Ds[t % 4]);
    const int64_t row = fbgemm_amd_padded_row_size_in_bytes(Ds[t % 4], tys[t % 4], 16, 4);
    off += (row * 100 + 127) / 128 * 128;
  }
  p.bytes = off;
  return p;
}

struct Buffers {
  void *weights, *indices, *offsets, *out, *status;
  Buffers(const Problem& p, int64_t B, int64_t n) {
    CHECK(hipMalloc(&weights, p.bytes) == hipSuccess);
    CHECK(hipMalloc(&indices, 8 * (n + 1)) == hipSuccess);
    CHECK(hipMalloc(&offsets, 8 * (p.T * B + 1)) == hipSuccess);
    CHECK(hipMalloc(&out, 4 * B * (p.D_offsets.back() + 8 * p.T)) == hipSuccess);
    CHECK(hipMalloc(&status, 16) == hipSuccess);
  }
  ~Buffers() {
    hipFree(weights);
    hipFree(indices);
    hipFree(offsets);
    hipFree(out);
    hipFree(status);
  }
};

int forward(fbgemm_amd_tbe_plan* plan, const Problem& p, Buffers& b, int64_t B, int64_t n, hipStream_t s, int32_t out_ty = 1) {
  return fbgemm_amd_tbe_forward(plan, b.weights, nullptr, b.indices, b.offsets, 64, n, p.T * B + 1, 0, nullptr, out_ty, b.out, b.status, s);
}

void plan_create_failures() {
  const Problem p = make_problem(5);
  fbgemm_amd_tbe_plan* plan = nullptr;
  CHECK(fbgemm_amd_tbe_plan_create(&plan, 0, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) < 0);
  CHECK(fbgemm_amd_tbe_plan_create(nullptr, 5, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) < 0);
  std::vector<uint8_t> bad_ty = p.tys;
  bad_ty[3] = 42; // rejected after the tables before it were filled in
  CHECK(fbgemm_amd_tbe_plan_create(&plan, 5, p.wo.data(), bad_ty.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) < 0);
  std::vector<int32_t> bad_D = p.D_offsets;
  bad_D[4] = bad_D[3];
  CHECK(fbgemm_amd_tbe_plan_create(&plan, 5, p.wo.data(), p.tys.data(), bad_D.data(), nullptr, p.bytes, 0, 16) < 0);
  // every allocation of a creation fails in turn: what was made before it goes back
  for (long k = 0; k < 8; ++k) {
    hip_stub_fail_malloc_after(k);
    plan = nullptr;
    const int rc = fbgemm_amd_tbe_plan_create(&plan, 5, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16);
    hip_stub_fail_malloc_after(-1);
    if (rc == 0) fbgemm_amd_tbe_plan_destroy(plan);
    else CHECK(plan == nullptr);
    CHECK(hip_stub_live_allocations() == 0);
  }
  fbgemm_amd_tbe_plan_destroy(nullptr);
}

void work_list_cache_and_graphs() {
  const Problem p = make_problem(6);
  fbgemm_amd_tbe_plan* plan = nullptr;
  CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
  const int64_t big_n = 1 << 21; // from here on the forwards order their bags (per-stream scratch)
  Buffers b(p, 64, big_n);
  hipStream_t s0 = hip_stub_stream(0), s1 = hip_stub_stream(1), s2 = hip_stub_stream(2);
  // a new batch size under capture is refused (it would allocate); nothing is left behind
  hip_stub_set_capturing(s0, true);
  CHECK(forward(plan, p, b, 7, big_n, s0) < 0);
  hip_stub_set_capturing(s0, false);
  CHECK(fbgemm_amd_tbe_plan_cached_work(plan) == 0);
  // batch sizes 1..6 on three streams, then some of them under capture (pinned)
  for (int64_t B = 1; B <= 6; ++B)
    for (hipStream_t s : {s0, s1, s2}) CHECK(forward(plan, p, b, B, big_n, s) == 0);
  hip_stub_set_capturing(s1, true);
  for (int64_t B : {2, 4}) CHECK(forward(plan, p, b, B, big_n, s1) == 0);
  hip_stub_set_capturing(s1, false);
  CHECK(fbgemm_amd_tbe_plan_pinned_work(plan) == 2);
  // many more batch sizes: the cache stays bounded, the pinned entries stay, the forwards go on working
  for (int64_t B = 7; B <= 48; ++B) CHECK(forward(plan, p, b, B, big_n, B % 2 ? s0 : s2) == 0);
  CHECK(fbgemm_amd_tbe_plan_cached_work(plan) <= 16);
  CHECK(fbgemm_amd_tbe_plan_pinned_work(plan) == 2);
  hip_stub_set_capturing(s1, true);
  CHECK(forward(plan, p, b, 2, big_n, s1) == 0); // a replayed graph's entry is still there
  hip_stub_set_capturing(s1, false);
  // small forwards (no scheduler), the three lane-shape variants, the 8-bit pooled output
  CHECK(forward(plan, p, b, 3, 100, s0) == 0);
  CHECK(fbgemm_amd_set_narrow_below_waves(0) == 0);
  CHECK(forward(plan, p, b, 3, 100, s0) == 0);
  CHECK(fbgemm_amd_set_narrow_below_waves(-1) == 0);
  CHECK(fbgemm_amd_set_lean(0) == 0);
  CHECK(forward(plan, p, b, 3, big_n, s0) == 0);
  CHECK(fbgemm_amd_set_lean(-1) == 0);
  CHECK(forward(plan, p, b, 5, big_n, s0, /*INT8 output*/ 2) == 0);
  CHECK(forward(plan, p, b, 40, big_n, s0, 2) == 0); // the scratch of the 8-bit output grows
  CHECK(forward(plan, p, b, 40, big_n, s1, 2) == 0); // another stream: waits for the event behind the last use
  hip_stub_set_capturing(s2, true);
  CHECK(forward(plan, p, b, 40, big_n, s2, 2) == 0); // under capture nothing is recorded or waited for
  hip_stub_set_capturing(s2, false);
  CHECK(fbgemm_amd_tbe_plan_reuse_order(plan, 1) == 0);
  CHECK(forward(plan, p, b, 5, big_n, s0) == 0);
  CHECK(fbgemm_amd_tbe_plan_reuse_order(plan, 0) == 0);
  // trim drops everything, also what graphs hold; the plan works afterwards
  CHECK(fbgemm_amd_tbe_plan_trim(plan) == 0);
  CHECK(fbgemm_amd_tbe_plan_cached_work(plan) == 0);
  CHECK(forward(plan, p, b, 2, big_n, s1) == 0);
  fbgemm_amd_tbe_plan_destroy(plan);
}

void remappings_twice_and_split_bags() {
  Problem p = make_problem(4);
  for (auto& ty : p.tys) ty = 3; // 4-bit tables only: the tolerance-grade plan cuts long bags into segments
  p.D_offsets = {0, 64, 192, 448, 512};
  p.wo = {0, 8192, 32768, 65536};
  p.bytes = 131072;
  fbgemm_amd_tbe_plan* plan = nullptr;
  CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
  CHECK(fbgemm_amd_tbe_plan_set_accumulate(plan, FBGEMM_AMD_ACC_FAST) == 0);
  Buffers b(p, 8, 4096);
  hipStream_t s = hip_stub_stream(3);
  const std::vector<int64_t> remap_off = {0, 1000, 1000, 3000, 3500}; // table 1 is not pruned
  void* remap = nullptr;
  CHECK(hipMalloc(&remap, 4 * 3500) == hipSuccess);
  void* d_remap_off = nullptr;
  CHECK(hipMalloc(&d_remap_off, 8 * 5) == hipSuccess);
  hipMemcpy(d_remap_off, remap_off.data(), 8 * 5, hipMemcpyHostToDevice);
  auto pruned = [&](int64_t B, int64_t n) {
    return fbgemm_amd_tbe_forward_pruned(plan, b.weights, nullptr, b.indices, b.offsets, 64, n, p.T * B + 1, 1, nullptr, 0, b.out,
                                         remap, 32, (const int64_t*)d_remap_off, 5, b.status, s);
  };
  CHECK(pruned(2, 4096) == 0); // few long bags: split into segments (plan-owned scratch), mappings read as arrays
  CHECK(fbgemm_amd_tbe_plan_set_index_remappings(plan, remap, 32, remap_off.data(), 5, s) == 0);
  CHECK(fbgemm_amd_tbe_plan_rank_tables(plan) == 3);
  CHECK(pruned(2, 4096) == 0);
  CHECK(fbgemm_amd_tbe_plan_set_index_remappings(plan, remap, 32, remap_off.data(), 5, s) == 0); // the records are made again
  CHECK(pruned(2, 4096) == 0);
  CHECK(pruned(8, 4096) == 0); // more bags: the segment scratch grows
  CHECK(fbgemm_amd_tbe_plan_set_index_remappings(plan, nullptr, 32, nullptr, 0, s) == 0);  // and dropped
  CHECK(fbgemm_amd_tbe_plan_rank_tables(plan) == 0);
  CHECK(pruned(2, 4096) == 0);
  CHECK(fbgemm_amd_tbe_plan_set_index_remappings(plan, remap, 32, remap_off.data(), 4, s) < 0); // wrong number of offsets
  fbgemm_amd_tbe_plan_destroy(plan);
  hipFree(remap);
  hipFree(d_remap_off);
}

fbgemm_amd_spmdm_config single_table(int32_t ty, int64_t D, int32_t use_offsets, int32_t accumulate) {
  fbgemm_amd_spmdm_config c;
  memset(&c, 0, sizeof(c));
  c.weight_ty = ty;
  c.output_ty = 0;
  c.index_bits = 64;
  c.offset_bits = 32;
  c.block_size = D;
  c.output_stride = -1;
  c.input_stride = -1;
  c.use_offsets = use_offsets;
  c.scale_bias_last = 1;
  c.accumulate = accumulate;
  return c;
}

void one_thread_of_single_table_calls(int id) {
  void *table, *idx, *lens, *out;
  CHECK(hipMalloc(&table, 1 << 20) == hipSuccess);
  CHECK(hipMalloc(&idx, 8 << 22) == hipSuccess);
  CHECK(hipMalloc(&lens, 4 * 70001) == hipSuccess);
  CHECK(hipMalloc(&out, 4 * 70000 * 128) == hipSuccess);
  hipStream_t s = hip_stub_stream(4 + id);
  // lengths instead of offsets (the prefix sum lives in the thread's scratch, which grows), a call
  // large enough to order its bags, few long bags in the tolerance-grade mode (segments)
  for (int64_t bags : {10, 3000, 70000}) {
    fbgemm_amd_spmdm_config c = single_table(3, 128, 0, FBGEMM_AMD_ACC_EXACT);
    CHECK(fbgemm_amd_spmdm_run(&c, bags, 1 << 22, 1000, table, idx, lens, nullptr, out, nullptr, s) >= 0);
  }
  fbgemm_amd_spmdm_config c = single_table(3, 128, 1, FBGEMM_AMD_ACC_FAST);
  CHECK(fbgemm_amd_spmdm_run(&c, 4, 4000, 1000, table, idx, lens, nullptr, out, nullptr, s) >= 0);
  CHECK(fbgemm_amd_spmdm_run(&c, 40, 40000, 1000, table, idx, lens, nullptr, out, nullptr, s) >= 0);
  hipFree(table);
  hipFree(idx);
  hipFree(lens);
  hipFree(out);
}

void thread_scratch_hand_over() {
  for (int round = 0; round < 3; ++round) { // threads that end hand their scratch to the next ones
    std::vector<std::thread> ts;
    for (int i = 0; i < 3; ++i) ts.emplace_back(one_thread_of_single_table_calls, i);
    for (auto& t : ts) t.join();
  }
  one_thread_of_single_table_calls(7); // and this thread adopts a set too
}

void entry_point_that_allocates_nothing() {
  void *table, *idx, *lens, *out, *status;
  CHECK(hipMalloc(&table, 1 << 20) == hipSuccess);
  CHECK(hipMalloc(&idx, 8 << 22) == hipSuccess);
  CHECK(hipMalloc(&lens, 4 * 65537) == hipSuccess);
  CHECK(hipMalloc(&out, 4 * 65536 * 128) == hipSuccess);
  CHECK(hipMalloc(&status, 16) == hipSuccess);
  const long before = hip_stub_total_allocations();
  fbgemm_amd_spmdm_config c = single_table(3, 128, 0, FBGEMM_AMD_ACC_EXACT);
  const int64_t most = fbgemm_amd_noalloc_max_bags();
  CHECK(fbgemm_amd_spmdm_launch_noalloc(&c, most, 1 << 22, 1000, table, idx, lens, nullptr, out, nullptr, status, nullptr) == 0);
  CHECK(fbgemm_amd_spmdm_launch_noalloc(&c, 100, 1 << 22, 1000, table, idx, lens, nullptr, out, nullptr, status, nullptr) == 0);
  CHECK(fbgemm_amd_spmdm_launch_noalloc(&c, most + 1, 1 << 22, 1000, table, idx, lens, nullptr, out, nullptr, status, nullptr) < 0);
  CHECK(hip_stub_total_allocations() == before); // it allocated nothing
  hipFree(table);
  hipFree(idx);
  hipFree(lens);
  hipFree(out);
  hipFree(status);
}

struct Check {
  const int32_t T = 8;
  const int64_t most = 1 << 20;
  int64_t *rows, *warning;
  void *idx, *off, *out_idx, *out_off;
  Check() {
    CHECK(hipMalloc((void**)&rows, 8 * T) == hipSuccess);
    CHECK(hipMalloc(&idx, 8 * 100) == hipSuccess);
    CHECK(hipMalloc(&off, 8 * (most + 1)) == hipSuccess);
    CHECK(hipMalloc(&out_idx, 8 * 100) == hipSuccess);
    CHECK(hipMalloc(&out_off, 8 * (most + 1)) == hipSuccess);
    CHECK(hipMalloc((void**)&warning, 8) == hipSuccess);
  }
  ~Check() {
    for (void* p : {(void*)rows, idx, off, out_idx, out_off, (void*)warning}) hipFree(p);
  }
  int operator()(int64_t bags, int mode, hipStream_t s) {
    return fbgemm_amd_check_remap_indices(rows, T, idx, off, 64, 100, bags + 1, mode, warning, nullptr, nullptr, 32, nullptr, out_idx, out_off, s);
  }
};

// Checks of any size, on several streams, eager and captured, keep nothing of one call that another
// could write: a thread's calls take no device memory from the library but what the first makes.
void checks_share_no_scratch() {
  Check call;
  CHECK(call(64, 1, hip_stub_stream(0)) == 0);
  hip_stub_finish_checks();
  const long before = hip_stub_total_allocations();
  for (int64_t bags : {int64_t(64), int64_t(8192), call.most})
    for (int mode : {1, 2})
      for (int s = 0; s < 3; ++s) {
        CHECK(call(bags, mode, hip_stub_stream(s)) == 0);
        hip_stub_finish_checks();
        hip_stub_set_capturing(hip_stub_stream(s), true);
        CHECK(call(bags, mode, hip_stub_stream(s)) == 0);
        hip_stub_set_capturing(hip_stub_stream(s), false);
      }
  CHECK(hip_stub_total_allocations() == before);
}

// The counter of a small check is its alone while it is in flight, on whatever stream (a new stream
// may have the handle of a destroyed one whose work is still running); there are only so many, and a
// finished check's is free again. Captured checks and those that do not count have none, and make none.
void checks_in_flight_have_a_counter_each() {
  Check call;
  std::thread([&] {
    const long before = hip_stub_total_allocations();
    hip_stub_set_capturing(hip_stub_stream(0), true);
    CHECK(call(64, 1, hip_stub_stream(0)) == 0);
    hip_stub_set_capturing(hip_stub_stream(0), false);
    CHECK(call(64, 2, hip_stub_stream(0)) == 0);
    CHECK(call(8192, 1, hip_stub_stream(0)) == 0);
    CHECK(hip_stub_total_allocations() == before && hip_stub_checks_in_flight() == 0);
    for (int round = 0; round < 3; ++round) {
      for (int n = 1; n <= 20; ++n) {
        CHECK(call(64, 1, hip_stub_stream(n % 2)) == 0);
        CHECK(hip_stub_checks_in_flight() == (n < 8 ? n : 8));
      }
      hip_stub_finish_checks();
    }
  }).join();
}

// The thread's own status block: a call that is refused, or that comes to nothing between begin and
// its launch, does not make the next one wait for the device.
void refused_calls_leave_the_own_status_alone() {
  void *table, *idx, *off, *out, *st;
  CHECK(hipMalloc(&table, 1 << 20) == hipSuccess);
  CHECK(hipMalloc(&idx, 8 * 4000) == hipSuccess);
  CHECK(hipMalloc(&off, 4 * 101) == hipSuccess);
  CHECK(hipMalloc(&out, 4 * 100 * 128) == hipSuccess);
  hipStream_t s = hip_stub_stream(3);
  fbgemm_amd_spmdm_config c = single_table(2, 128, 1, FBGEMM_AMD_ACC_EXACT);
  auto run = [&](int64_t rows) { return fbgemm_amd_spmdm_run(&c, 100, 4000, rows, table, idx, off, nullptr, out, nullptr, s); };
  CHECK(run(1000) == 1);
  const long waits = hip_stub_device_waits();
  CHECK(run(-1) < 0);
  CHECK(run(1000) == 1);
  CHECK(fbgemm_amd_status_begin(&st) == 0);
  CHECK(fbgemm_amd_spmdm_launch(&c, 100, 4000, 1000, table, nullptr, off, nullptr, out, nullptr, st, s) < 0);
  CHECK(fbgemm_amd_status_begin(&st) == 0);
  CHECK(run(1000) == 1);
  CHECK(hip_stub_device_waits() == waits);
  // one that had enqueued something does: its block may still be written
  CHECK(fbgemm_amd_status_begin(&st) == 0);
  CHECK(fbgemm_amd_spmdm_launch(&c, 100, 4000, 1000, table, idx, off, nullptr, out, nullptr, st, s) == 0);
  CHECK(run(1000) == 1);
  CHECK(hip_stub_device_waits() == waits + 1);
  // a thread's first waiting call, with a block of its own or with the one an ended thread has left
  for (int k = 0; k < 3; ++k) std::thread([&] { CHECK(run(1000) == 1); }).join();
  CHECK(hip_stub_device_waits() == waits + 1);
  // what a call finds wrong without a kernel reaches its user
  int32_t bits = 0;
  CHECK(fbgemm_amd_status_begin(&st) == 0);
  CHECK(fbgemm_amd_spmdm_launch(&c, 0, 5, 1000, table, idx, off, nullptr, out, nullptr, st, s) == 0);
  CHECK(fbgemm_amd_status_end(s, &bits, nullptr) == 0 && bits == FBGEMM_AMD_ERR_LENGTH_MISMATCH);
  // threads that end with their block in use: the blocks do not pile up
  const long blocks = hip_stub_total_allocations();
  for (int k = 0; k < 200; ++k)
    std::thread([&] {
      CHECK(fbgemm_amd_status_begin(&st) == 0);
      CHECK(fbgemm_amd_spmdm_launch(&c, 100, 4000, 1000, table, idx, off, nullptr, out, nullptr, st, s) == 0);
    }).join();
  CHECK(hip_stub_total_allocations() <= blocks + 64);
  // what a call without a block records is nobody's: the next waiting call does not care
  int32_t map[4] = {0, 1, 2, 3}, offs[2] = {0, 0};
  CHECK(fbgemm_amd_compressed_indices_remap(2, idx, 32, map, 4, offs, nullptr, out, out, nullptr, nullptr, s) == 0);
  const long now = hip_stub_device_waits();
  CHECK(run(1000) == 1);
  CHECK(hip_stub_device_waits() == now);
  hipFree(table);
  hipFree(idx);
  hipFree(off);
  hipFree(out);
}

// Every width, type, row layout, row stride and base alignment, in launches that take 16-byte lanes and
// such that take 4-byte ones: the loads of a row stay inside it (the stand-in's launches check that).
void row_reads_stay_in_the_row() {
  void *table, *idx, *off, *out;
  CHECK(hipMalloc(&table, 1 << 20) == hipSuccess);
  CHECK(hipMalloc(&idx, 64) == hipSuccess);
  CHECK(hipMalloc(&off, 64) == hipSuccess);
  CHECK(hipMalloc(&out, 64) == hipSuccess);
  fbgemm_amd_set_burst(0);
  for (int32_t lean : {0, 1}) {
    fbgemm_amd_set_lean(lean);
    for (int32_t ty : {0, 1, 2, 3, 4, 5})
      for (int32_t D = 1; D <= 1100; D += D < 300 ? 1 : 7)
        for (int32_t trailer : {0, 1})
          for (int32_t pad : {0, 1, 2, 4, 12})
            for (int32_t at : {0, 1, 2, 4}) {
              const int32_t elem = ty == 0 ? 4 : ty == 1 || ty == 5 ? 2 : 1;
              if (at % elem) continue;
              const int32_t bits = ty == 0 ? 32 : ty == 1 || ty == 5 ? 16 : ty == 2 ? 8 : ty == 3 ? 4 : 2;
              const int32_t row = elem > 1 ? D : (D * bits + 7) / 8 + (ty == 2 && trailer ? 8 : 4);
              fbgemm_amd_spmdm_config c = single_table(ty, D, 1, FBGEMM_AMD_ACC_EXACT);
              c.scale_bias_last = trailer;
              c.input_stride = pad ? row + pad : -1;
              for (int64_t bags : {100, 100000})
                CHECK(fbgemm_amd_spmdm_launch(&c, bags, 10, 10, (char*)table + at, idx, off, nullptr, out, nullptr, out, nullptr) == 0);
            }
  }
  fbgemm_amd_set_lean(0); // all tables in one launch of the general kernel
  for (int32_t align : {1, 4, 16}) {
    std::vector<int64_t> wo;
    std::vector<uint8_t> tys;
    std::vector<int32_t> Ds{0};
    int64_t bytes = 0;
    for (uint8_t ty : {0, 1, 2, 3, 4})
      for (int32_t D = 4; D <= 600; D += 4) {
        wo.push_back(bytes);
        tys.push_back(ty);
        Ds.push_back(Ds.back() + D);
        bytes += (fbgemm_amd_padded_row_size_in_bytes(D, ty, align, 4) * 10 + 127) / 128 * 128;
      }
    fbgemm_amd_tbe_plan* plan = nullptr;
    const int32_t T = (int32_t)tys.size();
    CHECK(fbgemm_amd_tbe_plan_create(&plan, T, wo.data(), tys.data(), Ds.data(), nullptr, bytes, 0, align) == 0);
    for (int64_t B : {1, 2000})
      for (int64_t n : {T * B, 40 * T * B}) // bags end to end in the wave, too
        CHECK(fbgemm_amd_tbe_forward(plan, table, nullptr, idx, off, 64, n, T * B + 1, 0, nullptr, 0, out, out, nullptr) == 0);
    fbgemm_amd_tbe_plan_destroy(plan);
  }
  fbgemm_amd_set_lean(-1);
  fbgemm_amd_set_burst(-1);
  for (void* p : {table, idx, off, out}) hipFree(p);
}

// The burst kernel goes over a bag by whole 8s of staged rows: a launch whose rows do not fit that many
// times would never end, and is refused on the host. The rule's own sizes fit, whatever it chooses.
void burst_launches_fit() {
  CHECK(fbgemm_amd::burst_pitch(256, 32) == 1024 && fbgemm_amd::burst_pitch(33, 4) == 32 && fbgemm_amd::burst_pitch(1000, 8) == 256);
  CHECK(!fbgemm_amd::burst_fits(256, 32, 1024) && !fbgemm_amd::burst_fits(300, 32, 8191) && fbgemm_amd::burst_fits(300, 32, 8192));
  void *table, *idx, *off, *out;
  CHECK(hipMalloc(&table, 1 << 20) == hipSuccess);
  CHECK(hipMalloc(&idx, 64) == hipSuccess);
  CHECK(hipMalloc(&off, 64) == hipSuccess);
  CHECK(hipMalloc(&out, 64) == hipSuccess);
  for (int waves : {-1, 1, 4}) {
    fbgemm_amd_set_burst(waves);
    for (int32_t ty : {0, 1, 2, 3, 4})
      for (int32_t D = 4; D <= 1100; D += D < 40 ? 4 : 36)
        for (int64_t bags : {1, 1500, 3000, 8000, 16000})
          for (int64_t len : {1, 20, 50, 100}) {
            fbgemm_amd_spmdm_config c = single_table(ty, D, 1, FBGEMM_AMD_ACC_EXACT);
            CHECK(fbgemm_amd_spmdm_launch(&c, bags, bags * len, 10, table, idx, off, nullptr, out, nullptr, out, nullptr) == 0);
          }
  }
  fbgemm_amd_set_burst(-1);
  for (void* p : {table, idx, off, out}) hipFree(p);
}

void allocation_failures_in_a_first_forward() {
  const Problem p = make_problem(5);
  Buffers b(p, 16, 1 << 21);
  hipStream_t s = hip_stub_stream(9);
  const long base = hip_stub_live_allocations();
  for (long k = 0; k < 24; ++k) {
    fbgemm_amd_tbe_plan* plan = nullptr;
    CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
    hip_stub_fail_malloc_after(k);
    const int rc = forward(plan, p, b, 16, 1 << 21, s);
    const int rc8 = forward(plan, p, b, 16, 1 << 21, s, 2);
    hip_stub_fail_malloc_after(-1);
    (void)rc;
    (void)rc8;
    CHECK(forward(plan, p, b, 16, 1 << 21, s) == 0); // a plan whose forward failed half-way works once memory is there
    fbgemm_amd_tbe_plan_destroy(plan);
    CHECK(hip_stub_live_allocations() == base);
  }
}

// A plan whose tables all have 4-bit rows in bags of 8 lanes: forwards that order their bags take the
// lean kernel's four-waves-per-SIMD instance, whose redo queue is made with every bag-order buffer
// (three streams, allocation failures in between) and freed with the work set.
void plan_of_wide_4bit_tables() {
  Problem p;
  p.T = 3;
  int64_t off = 0;
  p.D_offsets.push_back(0);
  for (int t = 0; t < p.T; ++t) {
    p.wo.push_back(off);
    p.tys.push_back(3);
    p.D_offsets.push_back(p.D_offsets.back() + 256);
    off += (fbgemm_amd_padded_row_size_in_bytes(256, 3, 16, 4) * 100 + 127) / 128 * 128;
  }
  p.bytes = off;
  // about 19 rows per bag: enough lookups for the bag order, bags too short for the end-to-end lane shapes
  const int64_t big_n = 1 << 21, B = 36000;
  Buffers b(p, B, big_n);
  const long base = hip_stub_live_allocations();
  CHECK(fbgemm_amd_set_wide4(2) == 0); // always that instance
  for (long k = -1; k < 12; ++k) {
    fbgemm_amd_tbe_plan* plan = nullptr;
    CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
    hip_stub_fail_malloc_after(k);
    (void)forward(plan, p, b, B, big_n, hip_stub_stream(0));
    hip_stub_fail_malloc_after(-1);
    for (int s = 0; s < 3; ++s) CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(s)) == 0);
    CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(1), /*INT8 output*/ 2) == 0);
    CHECK(forward(plan, p, b, 48, 100, hip_stub_stream(1)) == 0); // a small forward: no bag order, no queue
    fbgemm_amd_tbe_plan_destroy(plan);
    CHECK(hip_stub_live_allocations() == base);
  }
  CHECK(hip_stub_wide4_launches() >= 13 * 3); // the forwards above did take that instance
  // The default: the first forwards of a batch size time the two kernels in turn (waiting for the second event),
  // then the faster one stays. Under capture nothing is measured.
  CHECK(fbgemm_amd_set_wide4(-1) == 0);
  for (int faster = 0; faster < 2; ++faster) {
    hip_stub_set_elapsed_ms(1.0f, faster ? 0.5f : 0.995f); // the four-wave instance has to win by 1 %
    fbgemm_amd_tbe_plan* plan = nullptr;
    CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
    CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(0)) == 0);
    hip_stub_set_capturing(hip_stub_stream(1), true);
    const long before_capture = hip_stub_wide4_launches();
    CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(1)) == 0); // undecided and capturing: the general-purpose kernel
    CHECK(hip_stub_wide4_launches() == before_capture);
    hip_stub_set_capturing(hip_stub_stream(1), false);
    for (int i = 0; i < 24; ++i) CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(i % 3)) == 0);
    const long settled = hip_stub_wide4_launches();
    for (int i = 0; i < 6; ++i) CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(i % 3)) == 0);
    CHECK(hip_stub_wide4_launches() - settled == (faster ? 6 : 0));
    fbgemm_amd_tbe_plan_destroy(plan);
    CHECK(hip_stub_live_allocations() == base);
  }
}

// What a checked forward checks against; the stand-in's launches read none of it
struct Checked {
  int32_t T;
  int64_t *rows, *logical, *remap_off, *warning;
  void* remap;
  explicit Checked(int32_t tables) : T(tables) {
    for (int64_t** p : {&rows, &logical, &remap_off, &warning}) CHECK(hipMalloc((void**)p, 8 * (T + 1)) == hipSuccess);
    CHECK(hipMalloc(&remap, 64) == hipSuccess);
  }
  ~Checked() {
    for (void* p : {(void*)rows, (void*)logical, (void*)remap_off, (void*)warning, remap}) hipFree(p);
  }
  int operator()(fbgemm_amd_tbe_plan* plan, Buffers& b, int64_t B, int64_t n, bool pruned, hipStream_t s) {
    return fbgemm_amd_tbe_forward_checked(plan, b.weights, nullptr, b.indices, b.offsets, 64, n, T * B + 1, 0, nullptr, 1, b.out, rows, 1, warning,
                                          pruned ? logical : nullptr, pruned ? remap : nullptr, 32, pruned ? remap_off : nullptr,
                                          pruned ? T + 1 : 0, s);
  }
};

// In a checked forward an index outside its table reads row 0: a plan with a table that has no rows
// (the last one's row 0 would lie behind the weights) is not for the kernels, whatever the forward's size.
void checked_forwards_need_rows_everywhere() {
  const Problem whole = make_problem(4);
  Checked call(whole.T);
  Buffers b(whole, 3000, 16);
  for (int rowless : {-1, 1, 3}) {
    Problem p = whole;
    if (rowless == 1) p.wo[1] = p.wo[2] - 16; // no room for a row
    if (rowless == 3) p.bytes = p.wo[3];
    fbgemm_amd_tbe_plan* plan = nullptr;
    CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
    for (int t = 0; t < 4; ++t) CHECK((fbgemm_amd_tbe_plan_num_rows(plan, t) == 0) == (t == rowless));
    for (int64_t B : {2, 3000}) {
      const long before = hip_stub_launches();
      CHECK(call(plan, b, B, 16, false, hip_stub_stream(0)) == (rowless >= 0 ? 1 : 0));
      CHECK((hip_stub_launches() == before) == (rowless >= 0));
    }
    fbgemm_amd_tbe_plan_destroy(plan);
  }
}

// A checked forward that the kernels do not take keeps nothing of the work set: the plain forwards
// behind it go on measuring the two lean kernels, and settle on the faster one.
void refused_checked_forwards_keep_no_turn() {
  Problem p;
  p.T = 3; // two wide 4-bit tables and a 2-bit one
  p.tys = {3, 3, 4};
  p.D_offsets = {0, 256, 512, 544};
  p.wo = {0, 16384, 32768};
  p.bytes = 40960;
  const int64_t big_n = 1 << 21, B = 36000;
  Checked call(p.T);
  Buffers b(p, B, big_n);
  CHECK(fbgemm_amd_set_matrix(0) == 0);
  hip_stub_set_elapsed_ms(1.0f, 0.5f);
  for (int fast : {0, 1}) {
    fbgemm_amd_tbe_plan* plan = nullptr;
    CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
    CHECK(fbgemm_amd_tbe_plan_set_accumulate(plan, fast ? FBGEMM_AMD_ACC_FAST : FBGEMM_AMD_ACC_EXACT) == 0);
    for (int i = 0; i < 20; ++i) { // refused: a mapping beside a general table, the tolerance-grade mode
      CHECK(call(plan, b, B, big_n, !fast, hip_stub_stream(i % 2)) == 1);
      CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(i % 2)) == 0);
    }
    const long settled = hip_stub_wide4_launches();
    for (int i = 0; i < 6; ++i) CHECK(forward(plan, p, b, B, big_n, hip_stub_stream(i % 2)) == 0);
    CHECK(hip_stub_wide4_launches() - settled == 6);
    fbgemm_amd_tbe_plan_destroy(plan);
  }
  CHECK(fbgemm_amd_set_matrix(-1) == 0);
}

// The matrix kernel counts the entries of a run in 31 bits: forwards whose bags could be longer are not its
void forwards_beyond_the_matrix_kernels_runs() {
  Problem p;
  p.T = 2;
  p.tys = {3, 3};
  p.D_offsets = {0, 256, 512};
  p.wo = {0, 16384};
  p.bytes = 32768;
  const int64_t B = 9000;
  Buffers b(p, B, 16); // no kernel reads the indices here
  fbgemm_amd_tbe_plan* plan = nullptr;
  CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
  CHECK(fbgemm_amd_tbe_plan_set_accumulate(plan, FBGEMM_AMD_ACC_FAST) == 0);
  long before = hip_stub_matrix_launches();
  for (int64_t n : {int64_t(1) << 20, fbgemm_amd::MATRIX_MAX_RUN}) {
    CHECK(forward(plan, p, b, B, n, hip_stub_stream(0)) == 0);
    CHECK(hip_stub_matrix_launches() == ++before);
  }
  for (int64_t n : {fbgemm_amd::MATRIX_MAX_RUN + 1, int64_t(0x7fffffff), int64_t(1) << 33}) CHECK(forward(plan, p, b, B, n, hip_stub_stream(0)) == 0);
  CHECK(hip_stub_matrix_launches() == before);
  fbgemm_amd_tbe_plan_destroy(plan);
}

// Records of mappings, a plan's and a caller's, where an allocation fails: the call says so, leaves nothing behind, no
// error for the next launch to find either, and works once memory is there
void records_without_memory() {
  const std::vector<int64_t> offs = {0, 1000, 1000, 3000};
  void* remap = nullptr;
  CHECK(hipMalloc(&remap, 4 * 3000) == hipSuccess);
  Problem p = make_problem(3);
  fbgemm_amd_tbe_plan* plan = nullptr;
  CHECK(fbgemm_amd_tbe_plan_create(&plan, p.T, p.wo.data(), p.tys.data(), p.D_offsets.data(), nullptr, p.bytes, 0, 16) == 0);
  const long base = hip_stub_live_allocations();
  hipStream_t s = hip_stub_stream(2);
  for (long k = 0; k < 5; ++k) {
    fbgemm_amd_rank_records* ranks = nullptr;
    hip_stub_fail_malloc_after(k);
    CHECK(fbgemm_amd_rank_records_create(&ranks, remap, 32, offs.data(), 4, s) < 0 && !ranks);
    CHECK(hipGetLastError() == hipSuccess);
    hip_stub_fail_malloc_after(k);
    CHECK(fbgemm_amd_tbe_plan_set_index_remappings(plan, remap, 32, offs.data(), 4, s) < 0);
    hip_stub_fail_malloc_after(-1);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(fbgemm_amd_tbe_plan_rank_tables(plan) == 0 && hip_stub_live_allocations() == base);
  }
  fbgemm_amd_rank_records* ranks = nullptr;
  CHECK(fbgemm_amd_rank_records_create(&ranks, remap, 32, offs.data(), 4, s) == 2 && ranks);
  CHECK(fbgemm_amd_tbe_plan_set_index_remappings(plan, remap, 32, offs.data(), 4, s) == 0);
  fbgemm_amd_rank_records_destroy(ranks);
  fbgemm_amd_tbe_plan_destroy(plan);
  hipFree(remap);
}

// Both pooled-lookup kernels in one launch: lists that fit a grid each, and only apart
void lists_that_one_grid_cannot_hold() {
  const int64_t most = 0x7fffffffLL / 8; // waves of the longest run that a grid holds
  CHECK(fbgemm_amd::lookup_both_fits(most, 0) && fbgemm_amd::lookup_both_fits(0, most) && fbgemm_amd::lookup_both_fits(most - 1, 1) && fbgemm_amd::lookup_both_fits(1000, 1000));
  CHECK(!fbgemm_amd::lookup_both_fits(most, 1) && !fbgemm_amd::lookup_both_fits(1, most) && !fbgemm_amd::lookup_both_fits(most, most));
}

} // namespace

int main() {
  lists_that_one_grid_cannot_hold();
  forwards_beyond_the_matrix_kernels_runs();
  records_without_memory();
  plan_of_wide_4bit_tables();
  plan_create_failures();
  work_list_cache_and_graphs();
  remappings_twice_and_split_bags();
  thread_scratch_hand_over();
  entry_point_that_allocates_nothing();
  checks_in_flight_have_a_counter_each();
  refused_calls_leave_the_own_status_alone();
  burst_launches_fit();
  row_reads_stay_in_the_row();
  checks_share_no_scratch();
  checked_forwards_need_rows_everywhere();
  refused_checked_forwards_keep_no_turn();
  allocation_failures_in_a_first_forward();
  printf("launches %ld, device allocations %ld\n", hip_stub_launches(), hip_stub_total_allocations());
  printf("PASSED\n");
  return 0;
}
