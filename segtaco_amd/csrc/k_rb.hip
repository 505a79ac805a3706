// k_rb.hip — standalone launches of the row-balanced schedules (bodies in
// sched_rb.h): one workgroup per (row block, column panel).
#include "engine.h"
#include "sched_rb.h"

namespace segtaco {

template <int DT, int V>
__global__ __launch_bounds__(kBlockThreads) void k_rb_sr(const KArgs a) {
  int32_t blk, panel;
  if (!decode_block(a.panels, a.nblocks, blk, panel)) return;
  rb_sr_body<DT, V>(a, blk, panel);
}

template <int DT, int V>
__global__ __launch_bounds__(kBlockThreads) void k_rb_pr(const KArgs a) {
  int32_t blk, panel;
  if (!decode_block(a.panels, a.nblocks, blk, panel)) return;
  rb_pr_body<DT, V>(a, blk, panel);
}

template <int DT, int V>
__global__ __launch_bounds__(kBlockThreads) void k_rb_pr_all(const KArgs a) {
  int32_t blk, panel;
  if (!decode_block(a.panels, a.nblocks, blk, panel)) return;
  rb_pr_body<DT, V, 1, true>(a, blk, panel);
}

template <int DT, int V>
__global__ __launch_bounds__(kBlockThreads) void k_rb_pr4(const KArgs a) {
  int32_t blk, panel;
  if (!decode_block(a.panels, a.nblocks, blk, panel)) return;
  rb_pr_body<DT, V, 4, true>(a, blk, panel);
}

#define SEGTACO_CASE(KERNEL, DT, V, grid, args, stream)                        \
  case DT * 16 + V:                                                           \
    hipLaunchKernelGGL((KERNEL<DT, V>), dim3((unsigned)(grid)), dim3(kBlockThreads), 0, stream, \
                       args);                                                 \
    break
// slices of up to 4 columns
#define SEGTACO_CASES_V4(...)          \
  SEGTACO_CASE_DT(0, __VA_ARGS__);     \
  SEGTACO_CASE_DT(1, __VA_ARGS__);     \
  SEGTACO_CASE_DT(2, __VA_ARGS__)
#define SEGTACO_CASE_DT(DT, KERNEL, ...)     \
  SEGTACO_CASE(KERNEL, DT, 1, __VA_ARGS__);  \
  SEGTACO_CASE(KERNEL, DT, 2, __VA_ARGS__);  \
  SEGTACO_CASE(KERNEL, DT, 4, __VA_ARGS__)
#define SEGTACO_DISPATCH(KERNEL, dt, vec, ...) \
  switch ((dt) * 16 + (vec)) {                 \
    SEGTACO_CASES_V4(KERNEL, __VA_ARGS__);     \
    SEGTACO_CASE(KERNEL, 1, 8, __VA_ARGS__);   \
    SEGTACO_CASE(KERNEL, 2, 8, __VA_ARGS__);   \
    default: return hipErrorInvalidValue;      \
  }
#define SEGTACO_DISPATCH_V4(KERNEL, dt, vec, ...) \
  switch ((dt) * 16 + (vec)) {                    \
    SEGTACO_CASES_V4(KERNEL, __VA_ARGS__);        \
    default: return hipErrorInvalidValue;         \
  }

hipError_t launch_rb_sr(int dt, int vec, const KArgs &a, hipStream_t s) {
  const int64_t grid = grid_for(a.panels, a.nblocks);
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffff) return hipErrorInvalidConfiguration;
  SEGTACO_DISPATCH(k_rb_sr, dt, vec, grid, a, s);
  return hipGetLastError();
}

hipError_t launch_rb_pr(int dt, int vec, const KArgs &a, hipStream_t s) {
  const int64_t grid = grid_for(a.panels, a.nblocks);
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffff) return hipErrorInvalidConfiguration;
  // Four row sets per wave where most rows are one step (mean length up to P)
  // and a quarter of the workgroups still fills the chip. Power-law, us per
  // call, one set / four: 60013^2 (24 entries per row) N = 4 23.0 / 21.7, N = 1
  // 20.7 / 16.1; 262144^2 N = 1 64 / 41; but even rows of 20 entries at N = 16
  // (P = 16) 33 / 44, and 16-byte slices of 16-bit B lose to their registers
  // (262144^2 BF16 N = 16 128 / 147).
  if (grid <= 4 * (int64_t)device_cus()) {
    SEGTACO_DISPATCH(k_rb_pr_all, dt, vec, grid, a, s);
    return hipGetLastError();
  }
  if (grid < 8192 || vec == 8 || a.nnz > (int64_t)a.M << a.lg) {
    SEGTACO_DISPATCH(k_rb_pr, dt, vec, grid, a, s);
    return hipGetLastError();
  }
  KArgs f = a;
  f.nblocks = (a.nblocks + 3) / 4;
  SEGTACO_DISPATCH_V4(k_rb_pr4, dt, vec, grid_for(f.panels, f.nblocks), f, s);
  return hipGetLastError();
}

}  // namespace segtaco
