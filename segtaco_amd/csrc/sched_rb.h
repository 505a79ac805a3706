// sched_rb.h — row-balanced schedule bodies for gfx950 (wave64), shared by
// the standalone kernels (k_rb.hip) and the batched kernel (k_batch.hip).
//
// rb_sr (reference: spmm_rb_sr.h:187-243, K1): each lane group of Q lanes
// owns one output row and one column tile of Q*V columns; it walks the row's
// stored entries in CSR order, gathering V-wide slices of B rows (one
// coalesced Q*V-element request per entry) and accumulating sequentially, so
// every C element is a sequential sum in entry order (Eigen's order, with
// FMA).
//
// rb_pr (reference: spmm_rb_pr.h:223-375, K2): P = group slots of Q lanes
// share one row; slot s takes entries s, s+P, s+2P, ... and the P partial
// sums are combined with a butterfly over lane distances Q..Q*P/2, a fixed
// tree order, so results are deterministic. The reference's 32-lane,
// 4-column warps become 64-lane waves with Q*P*R = 64.
//
// Both walk in batches whose gathers are in flight together. A batch's
// columns and values are loaded during the batch before it, so a batch costs
// one memory latency, not two, and a row's last, partial batch one too.
//
// Neither schedule needs C cleared first: every row (empty ones included) is
// written exactly once.
#pragma once

#include "device_common.h"

namespace segtaco {

// acc += v * x for this lane's V columns; compensated with kComp.
template <int DT, int V, bool kComp>
__device__ __forceinline__ void rb_add(const typename RawT<DT, V>::type &x, float v,
                                       float (&acc)[V], float (&cmp)[V]) {
  float f[V];
  unpack<DT, V>(x, f);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    if constexpr (kComp)
      neumaier_add(acc[j], cmp[j], v, f[j]);
    else
      acc[j] = fmaf(v, f[j], acc[j]);
  }
}
// The same where `on`, without a branch.
template <int DT, int V, bool kComp>
__device__ __forceinline__ void rb_add_if(bool on, const typename RawT<DT, V>::type &x, float v,
                                          float (&acc)[V], float (&cmp)[V]) {
  float s[V], t[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    s[j] = acc[j];
    t[j] = cmp[j];
  }
  rb_add<DT, V, kComp>(x, v, s, t);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    acc[j] = on ? s[j] : acc[j];
    if constexpr (kComp) cmp[j] = on ? t[j] : cmp[j];
  }
}


// Columns and values of a batch of U consecutive entries, as 16-byte loads
// at element alignment (kRun: entries i .. i + U - 1 exist), or one load
// per entry at min(i + u, last). Without values the value loads read crd (in
// bounds: at most 4 bytes per entry) and are replaced by 1.0.
template <int DT, bool kRun, int U>
struct RbEntries {
  int32_t c[U];
  typename RawT<DT, 1>::type v[U];
  __device__ __forceinline__ void load(const KArgs &a, int32_t i, int32_t last) {
    constexpr int kEb = sizeof(v[0]);
    const char *vsrc = static_cast<const char *>(a.vals ? a.vals : a.crd);
    if constexpr (kRun) {
      __builtin_memcpy(c, __builtin_assume_aligned(a.crd + i, 4), sizeof(c));
      __builtin_memcpy(v, __builtin_assume_aligned(vsrc + (int64_t)i * kEb, kEb), sizeof(v));
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t j = i + min(u, last - i);
        c[u] = a.crd[j];
        __builtin_memcpy(&v[u], __builtin_assume_aligned(vsrc + (int64_t)j * kEb, kEb), kEb);
      }
    }
  }
  __device__ __forceinline__ float val(const KArgs &a, int u) const {
    if (!a.vals) return 1.0f;
    if constexpr (DT == 0)
      return v[u];
    else
      return half_to_f32<DT>(v[u]);
  }
};

// The sum of entries p .. e - 1 (p < e) for this lane's V columns. Whole
// batches run without a predicate on their entries. The wave's last batch loads
// no entries after it and a partial one gathers only rows that are there (short
// rows: two in three empty, the others of 8, FP32, us per call without / with these:
// N = 32 24 / 21, N = 50 69 / 54; banded, 33 entries per row: N = 64 88 / 78, N = 128 172 /
// 151; uniform 20 entries N = 32 31 / 31); a compensated row is long, and the test
// in its loop would cost more than the loads (lengths in rising order, BF16
// N = 3 173 / 224). kLean: without these, for the batched kernel, where their
// registers would spill (BF16 88 bytes).
// kRun: entries up to e + 2 * U - 2 exist.
template <int DT, int V, bool kOff32, int U, bool kRun, bool kComp, bool kLean>
__device__ __forceinline__ void rb_sr_sum(const KArgs &a, int32_t p, int32_t e, int32_t col,
                                          float (&acc)[V]) {
  using R = typename RawT<DT, V>::type;
  float cmp[V];
  zero_vec(cmp);
  RbEntries<DT, kRun, U> m;
  m.load(a, p, e - 1);
  R x[U];
  for (; e - p >= U; p += U) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      x[u] = load_row_raw<DT, V, kOff32>(a.B, m.c[u], a.ldb, col);
    if (!kComp && !kLean && __ballot(e - p > U) == 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) rb_add<DT, V, kComp>(x[u], m.val(a, u), acc, cmp);
      p = e;
      break;
    }
    const RbEntries<DT, kRun, U> w = m;
    m.load(a, kRun ? p + U : min(p + U, e - 1), e - 1);
#pragma unroll
    for (int u = 0; u < U; ++u) rb_add<DT, V, kComp>(x[u], w.val(a, u), acc, cmp);
  }
  if (p < e) {
    R y[U] = {};
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (kComp || kLean || u < e - p)
        y[u] = load_row_raw<DT, V, kOff32>(a.B, u < e - p ? m.c[u] : m.c[0], a.ldb, col);
#pragma unroll
    for (int u = 0; u < U; ++u)
      rb_add_if<DT, V, kComp>(u < e - p, y[u], m.val(a, u), acc, cmp);
  }
  if constexpr (kComp) {
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] += cmp[j];
  }
}

// One output row of rb_sr (entries p .. e - 1) for this lane's V columns.
template <int DT, int V, bool kOff32, int U, bool kRun, bool kLean>
__device__ __forceinline__ void rb_sr_row(const KArgs &a, int32_t row, int32_t p, int32_t e,
                                          int32_t col) {
  float acc[V];
  zero_vec(acc);
  if (e - p > a.comp_threshold)
    rb_sr_sum<DT, V, kOff32, U, kRun, true, kLean>(a, p, e, col, acc);
  else if (p < e)
    rb_sr_sum<DT, V, kOff32, U, kRun, false, kLean>(a, p, e, col, acc);
  store_row<V>(a.C + (int64_t)row * a.ldc + col, acc);
}

// The sum of the n > 0 entries p, p + 2^lg, ... of a slot of rb_pr. A batch loads
// no entries that are not there: where B stays in the caches the loads themselves
// are the time (banded, 33 entries per row, 8 slots, us per call, all four loads /
// those needed: FP32 N = 4 21 / 16, N = 64 176 / 159, BF16 N = 1 18 / 14). kAll: all
// four all the same, for launches whose time is their longest row's chain of
// batches, which the tests would lengthen: the four-set form (power-law 60013 x
// 50021, FP32 N = 4: 21.7 us, 23.3 with the tests) and launches of up to four
// workgroups per CU (power-law 20000^2, FP32 N = 4, 8 slots: 23 and 26 us). Chosen per
// wave, the two loops' registers cost the banded calls their gain.
template <int DT, int V, bool kOff32, bool kComp, bool kAll>
__device__ __forceinline__ void rb_pr_sum(const KArgs &a, int32_t p, int32_t n, int lg,
                                          int32_t col, float (&acc)[V]) {
  using R = typename RawT<DT, V>::type;
  constexpr int U = 4;
  float cmp[V], v[U];
  zero_vec(cmp);
  int32_t c[U];
  const int32_t last = p + ((n - 1) << lg);
  auto entries = [&](int32_t b) {
    if (kAll || b + U <= n) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t i = !kAll || b + u < n ? p + ((b + u) << lg) : last;
        c[u] = a.crd[i];
        v[u] = load_val<DT>(a.vals, i);
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (b + u < n) {
          const int32_t i = p + ((b + u) << lg);
          c[u] = a.crd[i];
          v[u] = load_val<DT>(a.vals, i);
        }
      }
    }
  };
  entries(0);
  R x[U];
  int32_t b = 0;
  for (; b + U <= n; b += U) {
    float w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      x[u] = load_row_raw<DT, V, kOff32>(a.B, c[u], a.ldb, col);
      w[u] = v[u];
    }
    entries(b + U);
#pragma unroll
    for (int u = 0; u < U; ++u) rb_add<DT, V, kComp>(x[u], w[u], acc, cmp);
  }
  if (b < n) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (kAll || b + u < n) x[u] = load_row_raw<DT, V, kOff32>(a.B, c[u], a.ldb, col);
#pragma unroll
    for (int u = 0; u < U; ++u) rb_add_if<DT, V, kComp>(b + u < n, x[u], v[u], acc, cmp);
  }
  if constexpr (kComp) {
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] += cmp[j];
  }
}

// Zeros to the rows of rb_sr's row block `blk`, column panel `panel`.
template <int V>
__device__ __forceinline__ void zero_rows(const KArgs &a, int32_t blk, int32_t panel) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t row =
      ((int64_t)(blk * kWavesPerBlock + wave) << (6 - a.lq)) + (lane >> a.lq);
  const int32_t nominal = ((panel << a.lq) + (lane & ((1 << a.lq) - 1))) * V;
  float z[V];
  zero_vec(z);
  if (row < a.M && nominal < a.N)
    store_row<V>(a.C + row * a.ldc + lane_col<V>(nominal, a.N), z);
}

// rb_sr over row block `blk`, column panel `panel`: lane group gi owns row gi.
template <int DT, int V, bool kLean, bool kOff32>
__device__ __forceinline__ void rb_sr_walk(const KArgs &a, int32_t blk,
                                           int32_t panel) {
  constexpr int U = 8;  // entries per batch
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int lq = a.lq;
  const int64_t row =
      ((int64_t)(blk * kWavesPerBlock + wave) << (6 - lq)) + (lane >> lq);
  const int32_t nominal = ((panel << lq) + (lane & ((1 << lq) - 1))) * V;
  const int32_t col = lane_col<V>(nominal, a.N);
  const bool live = row < a.M && nominal < a.N;
  const int32_t p = live ? a.pos[row] : 0, e = live ? a.pos[row + 1] : 0;
  // the wave's loads stay inside crd and vals, but for the last entries
  const bool run = __ballot(live && a.nnz - e < 2 * U) == 0;
  if (!live) return;
  if (run)
    rb_sr_row<DT, V, kOff32, U, true, kLean>(a, (int32_t)row, p, e, col);
  else
    rb_sr_row<DT, V, kOff32, U, false, kLean>(a, (int32_t)row, p, e, col);
}

template <int DT, int V, bool kLean = false>
__device__ __forceinline__ void rb_sr_body(const KArgs &a, int32_t blk,
                                           int32_t panel) {
  if (a.b_off32)
    rb_sr_walk<DT, V, kLean, true>(a, blk, panel);
  else
    rb_sr_walk<DT, V, kLean, false>(a, blk, panel);
}

// rb_pr over row block `blk`, column panel `panel`: R sets of 64/(P*Q) rows per
// wave. A row of up to P entries is one step (row pointer, column, gather) of
// three dependent loads, so a wave with several sets has them in flight
// together. The block's waves take its sets in turn: a wave sums the rest of its
// longer rows one set after another, and adjacent rows are often alike (lengths
// in rising order, 100000^2, us per call, a wave's sets adjacent / so: FP32 N = 3
// 65 / 57, N = 8 69 / 63, BF16 N = 12 163 / 135; one set per wave 47, 44, 131).
template <int DT, int V, bool kOff32, int R, bool kAll>
__device__ __forceinline__ void rb_pr_walk(const KArgs &a, int32_t blk,
                                           int32_t panel) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lq = a.lq, lg = a.lg;
  const int lr = 6 - lq - lg;  // log2(rows per set)
  const int64_t row0 = ((int64_t)blk * kWavesPerBlock * R + wave) << lr;
  const int64_t set = (int64_t)kWavesPerBlock << lr;  // rows to the wave's next set
  if (row0 >= a.M) return;  // uniform over the wave
  const int32_t slot = (lane >> lq) & ((1 << lg) - 1);
  const int32_t P = 1 << lg;
  const int32_t nominal = ((panel << lq) + (lane & ((1 << lq) - 1))) * V;
  const int32_t col = lane_col<V>(nominal, a.N);
  const bool colok = nominal < a.N;

  // this slot's entries of set k's row: p, p + P, ... (n of them)
  int32_t p[R], n[R];
  bool comp[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int64_t row = row0 + k * set + (lane >> (lq + lg));
    const bool live = row < a.M && colok;
    const int32_t s = live ? a.pos[row] : 0;
    const int32_t len = live ? a.pos[row + 1] - s : 0;
    p[k] = s + slot;
    n[k] = len > slot ? ((len - slot - 1) >> lg) + 1 : 0;
    comp[k] = len > a.comp_threshold;
  }
  float acc[R][V];
#pragma unroll
  for (int k = 0; k < R; ++k) zero_vec(acc[k]);
  if (R > 1 || __ballot(n[0] > 1) == 0) {
    // each slot's first entry, all sets' loads in flight together (a slot
    // without one reads entry 0; a wave of empty rows loads nothing: two rows in
    // three empty, BF16 N = 128 110 / 90 us per call)
    bool some = false;
#pragma unroll
    for (int k = 0; k < R; ++k) some = some || n[k] > 0;
    if (__ballot(some) != 0) {
      int32_t c[R];
      float v[R];
      typename RawT<DT, V>::type x[R];
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int32_t i = n[k] > 0 ? p[k] : 0;
        c[k] = a.crd[i];
        v[k] = load_val<DT>(a.vals, i);
      }
#pragma unroll
      for (int k = 0; k < R; ++k) x[k] = load_row_raw<DT, V, kOff32>(a.B, c[k], a.ldb, col);
#pragma unroll
      for (int k = 0; k < R; ++k) {
        float cmp[V];
        rb_add_if<DT, V, false>(n[k] > 0, x[k], v[k], acc[k], cmp);
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
      if (n[k] > 0 && comp[k]) {
        zero_vec(acc[k]);
        rb_pr_sum<DT, V, kOff32, true, kAll>(a, p[k], n[k], lg, col, acc[k]);
      } else if (n[k] > 1) {
        rb_pr_sum<DT, V, kOff32, false, kAll>(a, p[k] + P, n[k] - 1, lg, col, acc[k]);
      }
    }
  } else if (n[0] > 0) {
    if (comp[0])
      rb_pr_sum<DT, V, kOff32, true, kAll>(a, p[0], n[0], lg, col, acc[0]);
    else
      rb_pr_sum<DT, V, kOff32, false, kAll>(a, p[0], n[0], lg, col, acc[0]);
  }
  // butterfly over the P slots of each row (lane distances Q*P/2 .. Q)
#pragma unroll
  for (int k = 0; k < R; ++k) butterfly<V>(acc[k], P << lq >> 1, 1 << lq);
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int64_t row = row0 + k * set + (lane >> (lq + lg));
    if (row < a.M && colok && slot == 0) store_row<V>(a.C + row * a.ldc + col, acc[k]);
  }
}

template <int DT, int V, int R = 1, bool kAll = false>
__device__ __forceinline__ void rb_pr_body(const KArgs &a, int32_t blk,
                                           int32_t panel) {
  if (a.b_off32)
    rb_pr_walk<DT, V, true, R, kAll>(a, blk, panel);
  else
    rb_pr_walk<DT, V, false, R, kAll>(a, blk, panel);
}

}  // namespace segtaco
