// k_batch.hip — host dispatch of the persistent batched launch
// (k_batch_main, batch_main.h / k_batch_inst.hip), its counter reset and the
// batched carry fix-up.
#include "batch_main.h"
#include "sched_eb.h"
#include "sched_rb.h"

namespace segtaco {

__global__ void k_batch_reset(char *counters, size_t stride) {
  *reinterpret_cast<unsigned long long *>(counters + threadIdx.x * stride) = 0ull;
}

template <int V>
__device__ __forceinline__ void fixup_unit(const KArgs &a, int32_t blk, int32_t panel) {
  if (a.nnz == 0)
    zero_rows<V>(a, blk, panel);
  else
    fixup_body<V>(a, blk, panel);
}

__global__ __launch_bounds__(kBlockThreads) void k_batch_fixup(
    const BatchDesc *__restrict__ d, int32_t n,
    const int64_t *__restrict__ prefix, int64_t total) {
  for (int64_t u = blockIdx.x; u < total; u += gridDim.x) {
    const int32_t m = find_product(prefix, n, u);
    const BatchDesc &D = d[m];
    KArgs a = D.a;
    const int64_t local = u - D.fix_begin;
    const int32_t panel = (int32_t)(local % a.panels);
    const int32_t blk = (int32_t)(local / a.panels);
    switch (D.vec) {
      case 1: fixup_unit<1>(a, blk, panel); break;
      case 2: fixup_unit<2>(a, blk, panel); break;
      case 4: fixup_unit<4>(a, blk, panel); break;
      default: fixup_unit<8>(a, blk, panel); break;
    }
  }
}

// RUN(DT, kForm) for the pair (dt, form)
#define SEGTACO_BATCH_FORMS(DT, RUN)       \
  switch (form) {                          \
    case kBatchEbSr: RUN(DT, kBatchEbSr);  \
    case kBatchAny: RUN(DT, kBatchAny);    \
    case kBatchSv: RUN(DT, kBatchSv);      \
    default: return hipErrorInvalidValue;  \
  }
#define SEGTACO_BATCH_DISPATCH(RUN)        \
  switch (dt) {                            \
    case 0: SEGTACO_BATCH_FORMS(0, RUN)    \
    case 1: SEGTACO_BATCH_FORMS(1, RUN)    \
    case 2: SEGTACO_BATCH_FORMS(2, RUN)    \
    default: return hipErrorInvalidValue;  \
  }

hipError_t batch_main_grid(int dt, size_t lds, int32_t *grid, BatchForm form) {
#define RUN(DT, F) return batch_main_grid_t<DT, F>(lds, grid)
  SEGTACO_BATCH_DISPATCH(RUN)
#undef RUN
}

hipError_t launch_batch_reset(char *counters, size_t stride, int32_t count, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_reset, dim3(1), dim3((unsigned)count), 0, s, counters, stride);
  return hipGetLastError();
}

hipError_t launch_batch_main(int dt, const BatchDesc *d, int32_t n,
                             const int64_t *prefix, int64_t total,
                             unsigned long long *counter, int32_t grid,
                             size_t lds, hipStream_t s, BatchForm form) {
  if (total <= 0) return hipSuccess;
  // workgroups without a unit would only queue at the counter (5 ns each)
  if (grid > total) grid = (int32_t)total;
#define RUN(DT, F) return launch_batch_main_t<DT, F>(d, n, prefix, total, counter, grid, lds, s)
  SEGTACO_BATCH_DISPATCH(RUN)
#undef RUN
}

hipError_t launch_batch_fixup(const BatchDesc *d, int32_t n,
                              const int64_t *fix_prefix, int64_t total,
                              hipStream_t s) {
  if (total <= 0) return hipSuccess;
  const int64_t grid = total < (1 << 20) ? total : (1 << 20);
  hipLaunchKernelGGL(k_batch_fixup, dim3((unsigned)grid), dim3(kBlockThreads),
                     0, s, d, n, fix_prefix, total);
  return hipGetLastError();
}

}  // namespace segtaco
