// seg.h — the segment form of the eb_sr schedule (k_seg.hip): its arguments,
// launchers, and the rule for taking it.
#pragma once

#include <algorithm>

#include "launch.h"

namespace segtaco {

constexpr int32_t kSegMaxRange = 1024;  // entries per wave at most
constexpr int kSegStep = 8;             // entries per step of the sums

struct SegArgs {
  KArgs a;          // lq: log2 of the gather's lanes per entry
  int32_t ls;       // log2 of the lanes of a sum
  int32_t range;    // entries per wave, a multiple of a.tile
  int32_t nranges;  // ceil(nnz / range)
  int32_t tpr;      // tiles per range
  int32_t slice;    // rows per wave for the zero fill of empty rows
};

// LDS entries of a range: whole steps of the sums.
__host__ __device__ inline int32_t seg_pad(int32_t range) {
  return (range + kSegStep - 1) & ~(kSegStep - 1);
}
// Floats between the columns of the gathered B slices: 4 more than a
// multiple of the 64 banks, so that the lanes of a sum (one column each) read
// their 16 bytes from different banks.
__host__ __device__ inline int32_t seg_stride(int32_t range) {
  return ((seg_pad(range) - 4 + 63) & ~63) + 4;
}

// LDS of one wave: the gathered B slices (vec << lq columns, FP32), per entry
// the value and 12 bytes of segment and piece lists; with several tiles per
// range two sums (1 << ls floats) per tile and a list entry.
__host__ __device__ inline size_t seg_lds_wave(int32_t range, int32_t lq, int vec, int32_t tpr,
                                               int32_t ls) {
  const size_t b = ((size_t)vec << lq) * seg_stride(range) * 4 + (size_t)seg_pad(range) * 16 +
                   (tpr > 1 ? (size_t)tpr * (8 * ((size_t)1 << ls) + 4) : 0);
  return (b + 15) & ~(size_t)15;
}

// Fills g for an eb_sr call with arguments a (tile, ntiles, nnz, N, ... set),
// storage type dt and walk_blocks workgroups that k_eb_sr would launch, and
// returns the vector width to launch with; 0 when k_eb_sr takes the call.
int32_t seg_plan(int32_t dt, const KArgs &a, int64_t walk_blocks, SegArgs *g);

hipError_t launch_seg(int dt, int vec, const SegArgs &g, hipStream_t s);
hipError_t launch_seg_fixup(const SegArgs &g, hipStream_t s);
template <int DT>
hipError_t launch_seg_t(int vec, const SegArgs &g, hipStream_t s);

}  // namespace segtaco
