// device_common.h — shared device helpers for the gfx950 SpMM kernels.
//
// Storage types: DT 0 = FP32, 1 = BF16, 2 = FP16 (vals and B share the
// storage type; accumulation is always FP32). V is the number of B elements
// one lane loads per gather (one 32/64/128-bit load), so a lane group of Q
// lanes covers a column tile of Q*V columns of one B row with a single
// coalesced request of Q*V*sizeof(elem) bytes.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch.h"

namespace segtaco {

#define SEGTACO_WAVE 64

__device__ __forceinline__ float bf16_to_f32(uint32_t h16) {
  return __uint_as_float(h16 << 16);
}
__device__ __forceinline__ float f16_to_f32(uint32_t h16) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h16);
}

template <int DT>
__device__ __forceinline__ float half_to_f32(uint32_t h16) {
  if constexpr (DT == 1)
    return bf16_to_f32(h16 & 0xffffu);
  else
    return f16_to_f32(h16 & 0xffffu);
}

// One stored A value (index p); vals == nullptr reads as 1.0
// (the reference's __guard_load_default_one, gpu_library.h:154-161).
template <int DT>
__device__ __forceinline__ float load_val(const void *__restrict__ vals,
                                          int64_t p) {
  if (vals == nullptr) return 1.0f;
  if constexpr (DT == 0) {
    return static_cast<const float *>(vals)[p];
  } else {
    return half_to_f32<DT>(static_cast<const uint16_t *>(vals)[p]);
  }
}


// load_val for an entry stream read once (non-temporal: not kept in L2, which
// the gathers of B can use instead).
template <int DT>
__device__ __forceinline__ float load_val_stream(const void *__restrict__ vals, int64_t p) {
  if (vals == nullptr) return 1.0f;
  if constexpr (DT == 0) {
    return __builtin_nontemporal_load(static_cast<const float *>(vals) + p);
  } else {
    return half_to_f32<DT>(__builtin_nontemporal_load(static_cast<const uint16_t *>(vals) + p));
  }
}

// V consecutive elements starting at element index i (i aligned to V).
template <int DT, int V>
__device__ __forceinline__ void load_vec(const void *__restrict__ base,
                                         int64_t i, float (&out)[V]) {
  if constexpr (DT == 0) {
    const float *p = static_cast<const float *>(base) + i;
    if constexpr (V == 4) {
      float4 x = *reinterpret_cast<const float4 *>(p);
      out[0] = x.x; out[1] = x.y; out[2] = x.z; out[3] = x.w;
    } else if constexpr (V == 2) {
      float2 x = *reinterpret_cast<const float2 *>(p);
      out[0] = x.x; out[1] = x.y;
    } else {
      static_assert(V == 1, "fp32 vector width");
      out[0] = *p;
    }
  } else {
    const uint16_t *p = static_cast<const uint16_t *>(base) + i;
    if constexpr (V == 8) {
      uint4 x = *reinterpret_cast<const uint4 *>(p);
      uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        out[2 * k] = half_to_f32<DT>(w[k]);
        out[2 * k + 1] = half_to_f32<DT>(w[k] >> 16);
      }
    } else if constexpr (V == 4) {
      uint2 x = *reinterpret_cast<const uint2 *>(p);
      out[0] = half_to_f32<DT>(x.x);
      out[1] = half_to_f32<DT>(x.x >> 16);
      out[2] = half_to_f32<DT>(x.y);
      out[3] = half_to_f32<DT>(x.y >> 16);
    } else if constexpr (V == 2) {
      uint32_t x = *reinterpret_cast<const uint32_t *>(p);
      out[0] = half_to_f32<DT>(x);
      out[1] = half_to_f32<DT>(x >> 16);
    } else {
      static_assert(V == 1, "16-bit vector width");
      out[0] = half_to_f32<DT>(*p);
    }
  }
}

// Packed (not yet widened) V-element slice of a B row: what a gather leaves
// in registers while in flight. unpack() widens it to FP32 at use.
template <int DT, int V>
struct RawT;
template <>
struct RawT<0, 4> { using type = float4; };
template <>
struct RawT<0, 2> { using type = float2; };
template <>
struct RawT<0, 1> { using type = float; };
template <int DT>
struct RawT<DT, 8> { using type = uint4; };
template <int DT>
struct RawT<DT, 4> { using type = uint2; };
template <int DT>
struct RawT<DT, 2> { using type = uint32_t; };
template <int DT>
struct RawT<DT, 1> { using type = uint16_t; };

// A slice starts at any element: the last lane's columns end at N (lane_col)
// and rows of odd leading dimensions start anywhere. gfx950 reads 8- and
// 16-byte vectors from memory at any element alignment.
template <int DT, int V>
__device__ __forceinline__ typename RawT<DT, V>::type load_raw(
    const void *__restrict__ base, int64_t i) {
  constexpr int kEb = DT == 0 ? 4 : 2;
  typename RawT<DT, V>::type x;
  __builtin_memcpy(&x, __builtin_assume_aligned(static_cast<const char *>(base) + i * kEb, kEb),
                   sizeof(x));
  return x;
}

// First column of the slice of lane `lane` of a panel row whose nominal slice
// is [nominal, nominal + V): moved back to end at N, so that no lane reads or
// writes past the row (V <= N). The columns it shares with its left neighbour
// get the same value from both.
template <int V>
__device__ __forceinline__ int32_t lane_col(int32_t nominal, int32_t N) {
  return min(nominal, N - V);
}

template <int DT, int V>
__device__ __forceinline__ void unpack(const typename RawT<DT, V>::type &x,
                                       float (&out)[V]) {
  if constexpr (DT == 0) {
    if constexpr (V == 4) {
      out[0] = x.x; out[1] = x.y; out[2] = x.z; out[3] = x.w;
    } else if constexpr (V == 2) {
      out[0] = x.x; out[1] = x.y;
    } else {
      out[0] = x;
    }
  } else {
    if constexpr (V == 8) {
      const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        out[2 * k] = half_to_f32<DT>(w[k]);
        out[2 * k + 1] = half_to_f32<DT>(w[k] >> 16);
      }
    } else if constexpr (V == 4) {
      out[0] = half_to_f32<DT>(x.x);
      out[1] = half_to_f32<DT>(x.x >> 16);
      out[2] = half_to_f32<DT>(x.y);
      out[3] = half_to_f32<DT>(x.y >> 16);
    } else if constexpr (V == 2) {
      out[0] = half_to_f32<DT>(x);
      out[1] = half_to_f32<DT>(x >> 16);
    } else {
      out[0] = half_to_f32<DT>(x);
    }
  }
}

// V elements of row `row` of a row-major matrix (leading dimension ld,
// elements) from column c. kOff32: row, ld < 2^24 and every byte offset of
// the matrix fits 32 bits, so the offset is one 24-bit multiply added to the
// uniform base as a 32-bit byte offset (global_load with a scalar base)
// instead of 64-bit integer arithmetic with quarter-rate multiplies.
template <int DT, int V, bool kOff32>
__device__ __forceinline__ typename RawT<DT, V>::type load_row_raw(
    const void *__restrict__ base, int32_t row, int64_t ld, int32_t c) {
  if constexpr (kOff32) {
    constexpr uint32_t kEb = DT == 0 ? 4 : 2;
    const uint32_t off = (__umul24((uint32_t)row, (uint32_t)ld) + (uint32_t)c) * kEb;
    typename RawT<DT, V>::type x;
    __builtin_memcpy(&x, __builtin_assume_aligned(static_cast<const char *>(base) + off, kEb),
                     sizeof(x));
    return x;
  } else {
    return load_raw<DT, V>(base, (int64_t)row * ld + c);
  }
}

// The byte offset of row `row`, and V elements from column c of the row at
// such an offset: load_row_raw<DT, V, true> in two halves, for offsets that
// several lanes use.
template <int DT>
__device__ __forceinline__ uint32_t row_offset(int32_t row, int64_t ld) {
  return __umul24((uint32_t)row, (uint32_t)ld) * (DT == 0 ? 4 : 2);
}
template <int DT, int V>
__device__ __forceinline__ typename RawT<DT, V>::type load_off_raw(
    const void *__restrict__ base, uint32_t off, int32_t c) {
  constexpr uint32_t kEb = DT == 0 ? 4 : 2;
  typename RawT<DT, V>::type x;
  __builtin_memcpy(&x, __builtin_assume_aligned(
                           static_cast<const char *>(base) + (off + (uint32_t)c * kEb), kEb),
                   sizeof(x));
  return x;
}

// n elements of LDS from p (16-byte aligned), in 16-byte reads.
template <int n, typename T>
__device__ __forceinline__ void load_lds(const T *p, T (&x)[n]) {
  static_assert(sizeof(T) == 4 && n % 4 == 0, "16-byte reads");
  __builtin_memcpy(x, __builtin_assume_aligned(p, 16), sizeof(x));
}

// Makes this wave's LDS writes visible to all of its lanes: a release/acquire
// fence at wavefront scope around a wave barrier (no block-wide s_barrier).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x of the lane a DPP row shift (CTRL) names; 0 where that lane lies outside
// the row of 16 lanes.
template <int CTRL>
__device__ __forceinline__ int32_t dpp_or_zero(int32_t x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, false);
}

// Inclusive scan over the wave's 64 lanes, sum (kMax false) or maximum
// (kMax true), of values >= 0 (0 is the identity of both): shifts by 1, 2,
// 4 and 8 lanes inside each row of 16 (DPP, no LDS), then each row adds the
// totals of the rows below it (lanes 15, 31 and 47).
template <bool kMax>
__device__ __forceinline__ int32_t wave_scan(int32_t x) {
  auto op = [](int32_t u, int32_t v) { return kMax ? max(u, v) : u + v; };
  x = op(x, dpp_or_zero<0x111>(x));  // row_shr:1
  x = op(x, dpp_or_zero<0x112>(x));  // row_shr:2
  x = op(x, dpp_or_zero<0x114>(x));  // row_shr:4
  x = op(x, dpp_or_zero<0x118>(x));  // row_shr:8
  const int32_t b1 = __builtin_amdgcn_readlane(x, 15);
  const int32_t b2 = op(b1, __builtin_amdgcn_readlane(x, 31));
  const int32_t b3 = op(b2, __builtin_amdgcn_readlane(x, 47));
  const int row = (threadIdx.x & 63) >> 4;
  return row == 0 ? x : op(x, row == 1 ? b1 : row == 2 ? b2 : b3);
}

// x + (x of lane ^ D) for a power of two D < 64: row shifts and quad permutes
// below 16 (DPP) and gfx950's half-row swaps above, no LDS shuffle
// (ds_bpermute: an LDS access and a wait per value). Both lanes of a pair get
// the same bits.
template <int D>
__device__ __forceinline__ float add_xor_lane(float x) {
  const int32_t i = __float_as_int(x);
  if constexpr (D >= 16) {
    // swap(x, x): {even rows / lower half twice, odd rows / upper half twice}
    const auto p = D == 32
                       ? __builtin_amdgcn_permlane32_swap((uint32_t)i, (uint32_t)i, false, false)
                       : __builtin_amdgcn_permlane16_swap((uint32_t)i, (uint32_t)i, false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
  } else {
    int32_t o;
    if constexpr (D == 8) {
      o = __builtin_amdgcn_update_dpp(i, i, 0x128, 0xF, 0xF, false);  // row_ror:8
    } else if constexpr (D == 4) {
      o = __builtin_amdgcn_update_dpp(i, i, 0x104, 0xF, 0x5, false);  // row_shl:4, banks 0, 2
      o = __builtin_amdgcn_update_dpp(o, i, 0x114, 0xF, 0xA, false);  // row_shr:4, banks 1, 3
    } else if constexpr (D == 2) {
      o = __builtin_amdgcn_update_dpp(i, i, 0x4E, 0xF, 0xF, false);  // quad_perm 2,3,0,1
    } else {
      o = __builtin_amdgcn_update_dpp(i, i, 0xB1, 0xF, 0xF, false);  // quad_perm 1,0,3,2
    }
    return x + __int_as_float(o);
  }
}

// Butterfly sums of n values over lane distances `from`, from/2, .. `to`
// (uniform powers of two): one uniform branch per distance.
template <int n>
__device__ __forceinline__ void butterfly(float (&x)[n], int32_t from, int32_t to) {
#define SEGTACO_BUTTERFLY(D_)                                    \
  if (from >= D_ && to <= D_) {                                  \
    _Pragma("unroll") for (int j = 0; j < n; ++j) x[j] = add_xor_lane<D_>(x[j]); \
  }
  SEGTACO_BUTTERFLY(32)
  SEGTACO_BUTTERFLY(16)
  SEGTACO_BUTTERFLY(8)
  SEGTACO_BUTTERFLY(4)
  SEGTACO_BUTTERFLY(2)
  SEGTACO_BUTTERFLY(1)
#undef SEGTACO_BUTTERFLY
}

// V consecutive FP32 values to memory, at any float alignment.
template <int V>
__device__ __forceinline__ void store_row(float *p, const float (&v)[V]) {
  __builtin_memcpy(__builtin_assume_aligned(p, 4), v, sizeof(v));
}
template <int V>
__device__ __forceinline__ void load_row_f32(const float *p, float (&v)[V]) {
  __builtin_memcpy(v, __builtin_assume_aligned(p, 4), sizeof(v));
}

// V consecutive FP32 values (aligned to V floats; V == 8 is two float4).
template <int V>
__device__ __forceinline__ void store_vec(float *__restrict__ p,
                                          const float (&v)[V]) {
  if constexpr (V == 8) {
    reinterpret_cast<float4 *>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4 *>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
  } else if constexpr (V == 4) {
    *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else if constexpr (V == 2) {
    *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
  } else {
    p[0] = v[0];
  }
}

// store_row for data nothing reads back soon (non-temporal: not kept in L2),
// as whole 16- / 8-byte vector stores.
template <int V>
__device__ __forceinline__ void store_row_nt(float *__restrict__ p, const float (&v)[V]) {
  typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
  typedef float f2 __attribute__((ext_vector_type(2), aligned(4)));
  if constexpr (V == 8) {
    __builtin_nontemporal_store(f4{v[0], v[1], v[2], v[3]}, reinterpret_cast<f4 *>(p));
    __builtin_nontemporal_store(f4{v[4], v[5], v[6], v[7]}, reinterpret_cast<f4 *>(p) + 1);
  } else if constexpr (V == 4) {
    __builtin_nontemporal_store(f4{v[0], v[1], v[2], v[3]}, reinterpret_cast<f4 *>(p));
  } else if constexpr (V == 2) {
    __builtin_nontemporal_store(f2{v[0], v[1]}, reinterpret_cast<f2 *>(p));
  } else {
    __builtin_nontemporal_store(v[0], p);
  }
}

template <int V>
__device__ __forceinline__ void load_f32vec(const float *__restrict__ p,
                                            float (&v)[V]) {
  if constexpr (V == 8) {
    float4 a = reinterpret_cast<const float4 *>(p)[0];
    float4 b = reinterpret_cast<const float4 *>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else if constexpr (V == 4) {
    float4 a = *reinterpret_cast<const float4 *>(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  } else if constexpr (V == 2) {
    float2 a = *reinterpret_cast<const float2 *>(p);
    v[0] = a.x; v[1] = a.y;
  } else {
    v[0] = p[0];
  }
}

template <int V>
__device__ __forceinline__ void zero_vec(float (&v)[V]) {
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = 0.0f;
}

// Neumaier (compensated) accumulation of the exact-or-rounded product v*b.
// Contraction is disabled so that t is the rounded sum of s and x.
__device__ __forceinline__ void neumaier_add(float &s, float &c, float v,
                                             float b) {
#pragma clang fp contract(off)
  const float x = v * b;
  const float t = s + x;
  if (fabsf(s) >= fabsf(x))
    c += (s - t) + x;
  else
    c += (x - t) + s;
  s = t;
}

// XCD-aware decode of a 1-D grid into (row/tile block, column panel).
// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD
// b % 8), so the column panels of one row block are given consecutive
// per-XCD slots: they then share that XCD's L2 for the block's pos/crd/vals.
// Returns false for the padding blocks of the last round.
__device__ __forceinline__ bool decode_block(int32_t panels, int32_t nblocks,
                                             int32_t &blk, int32_t &panel) {
  const int32_t b = (int32_t)blockIdx.x;
  if (panels == 1) {
    blk = b;
    panel = 0;
    return blk < nblocks;
  }
  const int32_t xcd = b & 7;
  const int32_t k = b >> 3;
  panel = k % panels;
  blk = xcd + 8 * (k / panels);
  return blk < nblocks;
}

// Grid size that decode_block expects for `nblocks` row blocks.
__host__ __device__ inline int64_t grid_for(int32_t panels, int64_t nblocks) {
  if (panels == 1) return nblocks;
  return 8 * ((nblocks + 7) / 8) * panels;
}

// The reference's taco_binarySearchBefore (gpu_library.h:185-205) — see the
// oracle restatement for the exact tie-break it keeps.
__device__ __forceinline__ int32_t search_before(const int32_t *__restrict__ a,
                                                 int32_t start, int32_t end,
                                                 int64_t target) {
  if ((int64_t)a[end] <= target) return end;
  int32_t lo = start, hi = end;
  while (hi - lo > 1) {
    const int32_t mid = (hi + lo) >> 1;
    const int64_t v = a[mid];
    if (v < target)
      lo = mid;
    else if (v > target)
      hi = mid;
    else
      return mid;
  }
  return lo;
}

// Last row r in [lo, hi] with pos[r] <= p (the non-empty row holding entry p
// when pos[lo] <= p < pos[hi + 1]).
__device__ __forceinline__ int32_t row_of(const int32_t *__restrict__ pos,
                                          int32_t lo, int32_t hi, int32_t p) {
  while (lo < hi) {
    const int32_t mid = (lo + hi + 1) >> 1;
    if (pos[mid] <= p)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Last row r in [lo, hi) with pos[r] <= target, given pos[lo] <= target <
// pos[hi]: 64 probes per step. The whole wave calls it; the result is uniform.
__device__ __forceinline__ int32_t wave_row_of(const int32_t *__restrict__ pos, int32_t lo,
                                               int32_t hi, int32_t target) {
  const int32_t lane = threadIdx.x & 63;
  while (hi - lo > 1) {
    const int32_t step = ((hi - lo - 1) >> 6) + 1;
    const int64_t at = (int64_t)lo + (int64_t)(lane + 1) * step;
    const bool le = at < hi && pos[at] <= target;
    const int32_t c = __popcll(__ballot(le));  // probes are ascending
    lo += c * step;
    hi = (int32_t)min((int64_t)hi, (int64_t)lo + step);
  }
  return lo;
}

// Two wave_row_of searches in [0, M) at once (their probe loads overlap):
// the rows of entries e0 and e1 (e1 >= nnz: M).
__device__ __forceinline__ void wave_rows_of(const int32_t *__restrict__ pos, int32_t M,
                                             int32_t e0, int32_t e1, int32_t &r0, int32_t &r1) {
  const int32_t lane = threadIdx.x & 63;
  int32_t l0 = 0, l1 = 0, h0 = M, h1 = M;
  while (h0 - l0 > 1 || h1 - l1 > 1) {
    const int32_t st0 = ((h0 - l0 - 1) >> 6) + 1, st1 = ((h1 - l1 - 1) >> 6) + 1;
    const int64_t a0 = (int64_t)l0 + (int64_t)(lane + 1) * st0;
    const int64_t a1 = (int64_t)l1 + (int64_t)(lane + 1) * st1;
    // clamped probes load pos[M] (= nnz, above e0); no branch around the loads
    const int32_t p0 = pos[a0 < h0 ? a0 : M], p1 = pos[a1 < h1 ? a1 : M];
    const int32_t c0 = __popcll(__ballot(a0 < h0 && p0 <= e0));
    const int32_t c1 = __popcll(__ballot(a1 < h1 && p1 <= e1));
    l0 += c0 * st0;
    l1 += c1 * st1;
    h0 = (int32_t)min((int64_t)h0, (int64_t)l0 + st0);
    h1 = (int32_t)min((int64_t)h1, (int64_t)l1 + st1);
  }
  r0 = l0;
  r1 = l1;
}

}  // namespace segtaco
