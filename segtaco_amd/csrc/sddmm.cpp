// sddmm.cpp — host side of the SDDMM entry point (include/segtaco/sddmm.h):
// operand checks, vector width, lane count and tile selection, and the kernel
// launch. The kernel finds its rows itself; the workspace that the entry point
// asks for is left untouched.
#include <algorithm>

#include "engine.h"
#include "launch.h"
#include "sddmm.h"
#include "segtaco/sddmm.h"

namespace segtaco {
namespace {

// Entries per wave: as few as give 4096 waves (four per SIMD), but 16 and about
// a batch of the wave's slots at least. From 9 K entries per CU on, where an entry
// is work enough, short tiles again: 256 entries, 128 for rows of 256 bytes. Us per
// call at the tiles 512 / 256 / 128 / 64 / 32 / 16 (before, with a partition launch and
// tiles of 512):
//   power-law 1000^2 (16 K entries) J = 128 FP32 57 / 29 / 16 / 9.3 / 6.4 / 5.0 (58),
//     J = 8 13 / 7.7 / 5.0 / 4.4 / 4.4 / 4.4 (15)
//   8000^2 (125 K) J = 128 FP32 71 / 37 / 21 / 13 / 11 / 14 (72), J = 8 14 / 8.3 / 5.6 /
//     5.1 / 5.7 / 8.9 (16)
//   60013^2 (960 K) J = 16 FP32 23 / 17 / 18 (24), J = 128 BF16 49 / 38 / 38 (51)
//   uniform 100000^2 (2 M) J = 128 FP32 146 / 155 / 149 (147), BF16 76 / 77 / 79 (78)
//   uniform 150000^2 (3 M) J = 128 FP32 232 / 228 / 219 (233), BF16 134 / 116 / 115
//     (134), J = 64 76 / 66 / 65 (76), J = 32 FP32 60 / 60 / 59 (61), J = 8 37 / 38 / 42 (37)
//   power-law 262144^2 (4.2 M) J = 128 FP32 340 / 326 / 318 (341), J = 32 94 / 86 / 86
//     (94), J = 8 BF16 54 / 57 / 62 (53)
//   banded 200000^2 (6.6 M) J = 128 FP32 338 / 257 / 249 (338), J = 32 74 / 77 / 83 (74),
//     J = 64 BF16 96 / 99 / 105 (95)
int32_t sddmm_tile(int64_t nnz, int64_t row_bytes, int32_t lq) {
  if (nnz >= (int64_t)device_cus() * 9 * 1024 && row_bytes >= 128)
    return row_bytes >= 256 ? 128 : 256;
  int32_t tile = std::max(16, std::min(64, 256 >> lq));
  while (tile < kSdTile && nnz > (int64_t)4096 * tile) tile <<= 1;
  return tile;
}

// Elements per lane and load: the widest that J holds, whatever the alignment;
// but slices of four that take a 16-bit row in four lanes with nothing twice
// (J = 12, us per call, slices of 8 / so: uniform 3 M entries 46 / 34, banded 61 / 53).
int32_t sddmm_vec(int32_t dtype, int32_t J) {
  int32_t V = dtype == SEGTACO_DT_F32 ? 4 : 8;
  while (V > J) V >>= 1;
  if (V == 8 && J < 16 && J % 8 && J % 4 == 0) V = 4;
  return V;
}

}  // namespace
}  // namespace segtaco

using namespace segtaco;

extern "C" {

size_t segtaco_sddmm_workspace_bytes(const segtaco_csr_t *S) {
  if (!S || S->nnz <= 0) return 0;
  return align_up(sizeof(int32_t) * (size_t)(ceil_div(S->nnz, kSdTile) + 1), 256);
}

int32_t segtaco_sddmm(const segtaco_csr_t *S, const void *X, int64_t ldx,
                      const void *Y, int64_t ldy, int32_t J, int32_t dtype,
                      float *out, void *workspace, size_t workspace_bytes,
                      void *stream_v) {
  if (!S || S->M < 0 || S->K < 0 || S->nnz < 0 || J < 0)
    return set_error(SEGTACO_ERR_INVALID, "segtaco_sddmm: bad operand shape");
  if (S->nnz > kMaxNnz)
    return set_error(SEGTACO_ERR_UNSUPPORTED, "segtaco_sddmm: nnz %d above the supported %d",
                     S->nnz, kMaxNnz);
  if (dtype < SEGTACO_DT_F32 || dtype > SEGTACO_DT_F16)
    return set_error(SEGTACO_ERR_INVALID, "segtaco_sddmm: unknown dtype %d", dtype);
  if (S->vals && S->vals_dtype != dtype)
    return set_error(SEGTACO_ERR_INVALID,
                     "segtaco_sddmm: values stored as %d but X/Y as %d", S->vals_dtype,
                     dtype);
  if (S->nnz == 0) return SEGTACO_OK;
  if (S->M == 0 || !S->pos || !S->crd || !out)
    return set_error(SEGTACO_ERR_INVALID, "segtaco_sddmm: null operand");
  hipStream_t stream = static_cast<hipStream_t>(stream_v);
  if (J == 0) {
    SEGTACO_HIP(launch_fill_zero(out, 1, S->nnz, S->nnz, stream));
    return SEGTACO_OK;
  }
  if (!X || !Y || ldx < J || ldy < J)
    return set_error(SEGTACO_ERR_INVALID, "segtaco_sddmm: X/Y missing or leading dimension < J");
  const size_t need = segtaco_sddmm_workspace_bytes(S);
  if (!workspace || workspace_bytes < need)
    return set_error(SEGTACO_ERR_INVALID, "segtaco_sddmm: workspace of %zu bytes needed",
                     need);
  const int32_t eb = elem_bytes(dtype);
  const int32_t V = sddmm_vec(dtype, J);
  int32_t lq = 0;
  while ((1 << lq) < 64 && (int64_t)(1 << lq) * V < J) ++lq;

  SddmmArgs a{};
  a.M = S->M;
  a.K = S->K;
  a.J = J;
  a.nnz = S->nnz;
  a.pos = S->pos;
  a.crd = S->crd;
  a.vals = S->vals;
  a.X = X;
  a.ldx = ldx;
  a.Y = Y;
  a.ldy = ldy;
  a.out = out;
  a.lq = lq;
  a.off32 = b_off32_ok(S->M, ldx, eb) && b_off32_ok(S->K, ldy, eb);
  a.tile = sddmm_tile(S->nnz, (int64_t)J * eb, lq);
  a.ntiles = (int32_t)ceil_div(S->nnz, a.tile);
  SEGTACO_HIP(launch_sddmm(dtype, V, a, stream));
  return SEGTACO_OK;
}

}  // extern "C"
