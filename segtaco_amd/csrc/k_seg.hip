// k_seg.hip — the segment form of eb_sr for one storage type, chosen by
// SEGTACO_SEG_DT at compile time (0 FP32, 1 BF16, 2 FP16; the build compiles
// this file once per type).
//
// eb_sr cuts the entries into tiles of T and sums each row's entries inside
// a tile sequentially; rows over several tiles are the left fold of their
// tile sums. k_eb_sr gives each tile to one lane group of Q lanes, one per V
// columns. A narrow product has few lanes per group, so a wave holds up to 64
// groups that read crd and vals at 64 distant places and end their rows at
// different steps; a small one leaves most of the chip without a tile; and
// both pay three launches (partition, walk, fix-up).
//
// Here a wave takes a range of whole tiles, one at least: up to 384 entries (128 at
// N = 16), less where that would leave fewer than 2048 waves, a longer tile alone:
//   * it finds the range's rows itself (a 64-way search of pos, three
//     dependent loads for 262144 rows), so there is no partition launch;
//   * all lanes gather the range's B slices, entry after entry, whatever row
//     they belong to, into LDS (column-major, FP32);
//   * the range's pieces (row x tile) are listed in LDS, and lane groups of
//     one lane per column sum them from there, each taking the next piece as
//     it finishes its last. A piece's sum is a serial chain of up to T steps,
//     but of LDS reads instead of gathers.
// The sums and folds are those of eb_sr for the same T, bit for bit: a
// piece is summed sequentially, the pieces of a row that begins and ends in
// the range are folded in order; a row that began before the range stores
// each tile's part to carry_head, one that continues past it its fold so far
// to the range's carry_tail, and k_seg_fixup folds those.
//
// Measured, us per call (k_eb_sr's three launches -> this): power-law
// 1000^2, N = 16, tile 128: 53 -> 12.5; 60000^2, N = 4: 166 -> 24 (tile 128),
// 66 -> 35 (tile 8); 262144^2, N = 4: 298 -> 72 (tile 128), 129 -> 77 (tile
// 32); N = 1: 255 -> 74. What bounds it now is instruction issue in the sums:
// at N = 4 and tile 128 a range's longest piece takes 16 steps and most
// groups idle through its last ones (1485 VALU instructions per wave of 384
// entries, 26 of the 66 us); the 4.2 M gathers, one 128-byte line each, need
// about 12 us. Ranges of 128 to 1024 entries measured within 30 % of the best
// at each width: longer ones balance the groups, shorter ones let more waves
// share a CU's LDS. Tiles shorter than a range cost its piece lists and the later
// pieces' sums (60000^2, N = 4: 24 at tile 128, 35 at tile 8), and the 16 gathers per
// lane are more than a short range fills: at N <= 4, where a wave's 64 groups cover
// 1024 entries, ten of them re-load the last of 384.
#include "device_common.h"
#include "seg.h"

#ifndef SEGTACO_SEG_DT
#error "SEGTACO_SEG_DT must be defined (0, 1 or 2)"
#endif

namespace segtaco {
namespace {

constexpr int kSegG = 16;  // gathers per lane in flight before they go to LDS

// Flags of a segment or piece beside its start (ranges are at most 1024 long).
constexpr uint32_t kSegStart = 0x3ff;
constexpr uint32_t kSegComp = 0x8000;   // of a compensated row
constexpr uint32_t kSegMany = 0x4000;   // of a segment over several tiles
constexpr uint32_t kSegFirst = 0x2000;  // the segment's first piece

template <int DT, int V, bool kOff32, bool kComp>
__global__ __launch_bounds__(64) void k_eb_seg(const SegArgs g) {
  extern __shared__ __align__(16) char smem[];
  using R = typename RawT<DT, V>::type;
  const KArgs &a = g.a;
  const int lane = threadIdx.x;
  const int32_t w = blockIdx.x;
  // gather: Q lanes of V columns per entry
  const int lq = a.lq;
  const int32_t Q = 1 << lq, G = 64 >> lq;
  const int32_t q = lane & (Q - 1);
  const int32_t grp = lane >> lq;
  const bool colok = q * V < a.N;
  const int32_t col = lane_col<V>(q * V, a.N);
  const int32_t P = seg_pad(g.range), sx = seg_stride(g.range);
  float *s_x = reinterpret_cast<float *>(smem);  // [Q * V][sx]: column-major
  float *s_val = s_x + ((size_t)(V * sx) << lq);
  int32_t *s_row = reinterpret_cast<int32_t *>(s_val + P);
  uint16_t *s_seg = reinterpret_cast<uint16_t *>(s_row + P);  // segment starts
  // pieces (segment x tile): start and flags, and segment
  uint16_t *s_pc = g.tpr > 1 ? s_seg + P : s_seg;
  uint16_t *s_pk = s_pc + P;
  // several tiles per range: sums of the pieces of segments over several
  // tiles, [first piece, tile], then [later piece, tile]; and those segments
  float *s_sum = reinterpret_cast<float *>(s_seg + 4 * P);  // [2 * tpr][1 << ls]
  uint16_t *s_many = reinterpret_cast<uint16_t *>(s_sum + ((size_t)(2 * g.tpr) << g.ls));

  const int32_t *__restrict__ pos = a.pos;
  const int32_t T = a.tile;
  const int32_t s0 = w * g.range;
  const int32_t cn = min(a.nnz - s0, g.range);
  const int32_t s1 = s0 + cn;
  const bool last_range = s1 >= a.nnz;

  // 1. gather: group grp takes entries grp, grp + G, ... of the range; a batch
  // issues all its loads with no branch around them (entries past the range
  // re-load its last one), and the first is in flight during the search for
  // the range's rows.
  int32_t c[kSegG];
  R x[kSegG];
  auto columns = [&](int32_t i0) {
#pragma unroll
    for (int u = 0; u < kSegG; ++u) c[u] = a.crd[s0 + min(i0 + u * G + grp, cn - 1)];
  };
  auto gather = [&]() {
#pragma unroll
    for (int u = 0; u < kSegG; ++u) x[u] = load_row_raw<DT, V, kOff32>(a.B, c[u], a.ldb, col);
  };
  auto stage = [&](int32_t i0) {
#pragma unroll
    for (int u = 0; u < kSegG; ++u) {
      const int32_t i = i0 + u * G + grp;
      if (i < cn) {
        float f[V];
        unpack<DT, V>(x[u], f);
#pragma unroll
        for (int j = 0; j < V; ++j) s_x[(q * V + j) * sx + i] = f[j];
      }
    }
  };
  columns(0);
  gather();
  int32_t r0, rn;
  wave_rows_of(pos, a.M, s0, s1, r0, rn);
  rn = min(rn, a.M - 1);
  const bool head = pos[r0] < s0;  // the first segment began before the range
  stage(0);
  for (int32_t i0 = kSegG * G; i0 < cn; i0 += kSegG * G) {
    columns(i0);
    gather();
    stage(i0);
  }
  for (int32_t i = lane; i < cn; i += 64) s_val[i] = load_val<DT>(a.vals, s0 + i);

  // 2. empty rows of this wave's slice of the rows, as zeros: 64 rows at a
  // time, each lane group a row (nobody else writes them).
  {
    const int64_t z0 = (int64_t)w * g.slice;
    const int32_t z1 = (int32_t)min((int64_t)a.M, z0 + g.slice);
    float z[V];
    zero_vec(z);
    for (int64_t r = z0; r < z1; r += 64) {
      const int64_t mine = r + lane;
      const uint64_t m = __ballot(mine < z1 && pos[mine] == pos[mine + 1]);
      if (m == 0) continue;
      for (int32_t i = 0; i < Q; ++i) {
        const int32_t b = i * G + grp;
        if (((m >> b) & 1) && colok) store_row<V>(a.C + (r + b) * a.ldc + col, z);
      }
    }
  }

  // 3. the range's segments, 64 rows per step; and for this range's tiles the
  // row each starts in and the fix-up record (the tile where the row that ends
  // in it began, if an earlier one), which the workspace holds after a call.
  int32_t nseg = 0;
  int32_t row_end = 0;  // end of the last listed row
  {
    const int32_t t0 = w * g.tpr;
    const int32_t t_end = min(t0 + g.tpr, a.ntiles);
    int32_t *rows = const_cast<int32_t *>(a.tile_row);
    int32_t *fix = const_cast<int32_t *>(a.fix_t0);
    int64_t rb = r0;
    while (rb <= rn) {
      const int64_t r = rb + lane;
      int32_t p0 = s1, p1 = s1;
      if (r <= rn) {
        p0 = pos[r];
        p1 = pos[r + 1];
      }
      const bool in = p0 < p1 && p0 < s1;
      const uint64_t m = __ballot(in);
      if (in) {
        const int32_t k = nseg + (int32_t)__builtin_amdgcn_mbcnt_hi(
                                     (uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        s_row[k] = (int32_t)r;
        s_seg[k] = (uint16_t)((max(p0, s0) - s0) |
                              (kComp && p1 - p0 > a.comp_threshold ? kSegComp : 0u));
        {
          const int32_t b1 = (p1 - 1) / T;
          int32_t b = p0 > s0 ? (int32_t)(((int64_t)p0 + T - 1) / T) : t0;
          for (; b <= b1 && b < t_end; ++b) {
            rows[b] = (int32_t)r;
            fix[b] = (b == b1 && (int64_t)p0 < (int64_t)b * T) ? p0 / T : -1;
          }
        }
      }
      nseg += __popcll(m);
      if (m) {
        row_end = __builtin_amdgcn_readlane(p1, 63 - __clzll((long long)m));
        if (row_end >= s1) break;
        rb += 64;
      } else {
        // 64 empty rows: on to the row of the next entry
        rb = wave_row_of(pos, (int32_t)min(rb + 63, (int64_t)rn), a.M, row_end);
      }
    }
    if (last_range && lane == 0) rows[a.ntiles] = a.M;
  }
  const bool cross = row_end > s1;  // the last segment continues past the range
  wave_sync();

  // 4. the pieces of the segments, when the range holds several tiles.
  int32_t np = nseg, nmany = 0;
  if (g.tpr > 1) {
    np = 0;
    for (int32_t kb = 0; kb < nseg; kb += 64) {
      const int32_t k = kb + lane;
      int32_t cnt = 0, st = 0, b0 = 0;
      uint32_t f = 0;
      if (k < nseg) {
        const uint32_t s = s_seg[k];
        const int32_t en = k + 1 < nseg ? (int32_t)(s_seg[k + 1] & kSegStart) : cn;
        st = (int32_t)(s & kSegStart);
        f = s & kSegComp;
        b0 = st / T;
        cnt = (en - 1) / T - b0 + 1;
      }
      const int32_t inc = wave_scan<false>(cnt);
      const uint64_t mm = __ballot(cnt > 1);
      if (cnt > 1) {
        f |= kSegMany;
        s_many[nmany + __popcll(mm & (((uint64_t)1 << lane) - 1))] = (uint16_t)k;
      }
      nmany += __popcll(mm);
      const int32_t at = np + inc - cnt;
      for (int32_t j = 0; j < cnt; ++j) {
        s_pc[at + j] = (uint16_t)((j == 0 ? st | kSegFirst : (b0 + j) * T) | f);
        s_pk[at + j] = (uint16_t)k;
      }
      np += __builtin_amdgcn_readlane(inc, 63);
    }
    wave_sync();
  }

  // 5. sums: lane groups of one lane per column take the pieces in order, each
  // the next one as it finishes its last; a step reads an aligned block of
  // eight entries (two 16-byte reads of the column and two of the values).
  const int ls = g.ls;
  const int32_t L = 1 << ls;
  const int32_t l = lane & (L - 1);
  const int32_t sg = lane >> ls;
  const bool ok = l < a.N;
  const int32_t scol = min(l, a.N - 1);
  // where the gather put column scol (its last lane's slice ends at N)
  const int32_t whole = a.N / V * V;
  const float *xc = s_x + (scol < whole ? scol : scol - a.N + V + whole) * sx;
  float acc = 0.0f, cmp = 0.0f;
  const uint64_t leaders = __ballot(l == 0);
  const uint64_t below = ((uint64_t)1 << (lane & ~(L - 1))) - 1;
  int32_t nxt = 0;
  int32_t gi = 0, ge = 0, gp = 0;  // next entry, end of the piece, the piece
  uint32_t gf = 0;
  for (;;) {
    const bool need = gi >= ge;
    const uint64_t m = __ballot(need) & leaders;
    if (m) {
      const int32_t p = nxt + __popcll(m & below);
      nxt += __popcll(m);
      if (need) {
        gi = ge = 0;
        if (p < np) {
          gp = p;
          gf = s_pc[p];
          gi = (int32_t)(gf & kSegStart);
          ge = p + 1 < np ? (int32_t)(s_pc[p + 1] & kSegStart) : cn;
          acc = cmp = 0.0f;
        }
      }
      if (!__ballot(gi < ge)) break;
    }
    if (gi < ge) {
      const int32_t i0 = gi & ~(kSegStep - 1);
      const uint32_t lo = (uint32_t)(gi - i0), n = (uint32_t)min(ge - i0, kSegStep) - lo;
      float v[kSegStep], x[kSegStep];
      load_f32vec<kSegStep>(s_val + i0, v);
      load_f32vec<kSegStep>(xc + i0, x);
      if (kComp && (gf & kSegComp)) {
#pragma unroll
        for (int u = 0; u < kSegStep; ++u)
          if (u - lo < n) neumaier_add(acc, cmp, v[u], x[u]);
      } else {
#pragma unroll
        for (int u = 0; u < kSegStep; ++u) {
          const float t = fmaf(v[u], x[u], acc);
          acc = u - lo < n ? t : acc;
        }
      }
      gi = i0 + kSegStep;
      if (gi >= ge) {
        if (kComp && (gf & kSegComp)) acc += cmp;
        const int32_t k = g.tpr > 1 ? (int32_t)s_pk[gp] : gp;
        if (head && k == 0) {
          if (ok) a.carry_head[(int64_t)((s0 + ge - 1) / T) * a.N + scol] = acc;
        } else if (g.tpr > 1 && (gf & kSegMany)) {
          const int32_t b = (ge - 1) / T + (gf & kSegFirst ? 0 : g.tpr);
          s_sum[(b << ls) + l] = acc;
        } else if (ok) {
          *(cross && k == nseg - 1 ? a.carry_tail + (int64_t)w * g.tpr * a.N + scol
                                   : a.C + (int64_t)s_row[k] * a.ldc + scol) = acc;
        }
      }
    }
  }
  if (nmany == 0) return;

  // 6. rows over several tiles of the range: their pieces' sums, in order.
  wave_sync();
  for (int32_t i = sg; i < nmany; i += 64 >> ls) {
    const int32_t k = s_many[i];
    if (head && k == 0) continue;
    const int32_t st = (int32_t)(s_seg[k] & kSegStart);
    const int32_t en = k + 1 < nseg ? (int32_t)(s_seg[k + 1] & kSegStart) : cn;
    const int32_t b1 = (en - 1) / T;
    int32_t b = st / T;
    acc = s_sum[(b << ls) + l];
    while (++b <= b1) acc += s_sum[((g.tpr + b) << ls) + l];
    if (ok)
      *(cross && k == nseg - 1 ? a.carry_tail + (int64_t)w * g.tpr * a.N + scol
                               : a.C + (int64_t)s_row[k] * a.ldc + scol) = acc;
  }
}

// The rows that cross ranges: per range, one lane group (a lane per column)
// writes the row that began in an earlier range and ends in this one as the
// fold of the tail of the range it began in and every tile's part after that
// range, in order. A long row of short tiles has hundreds of parts, so 64
// loads are in flight at a time.
__global__ __launch_bounds__(kBlockThreads) void k_seg_fixup(const SegArgs g) {
  const KArgs &a = g.a;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int32_t w = ((blockIdx.x * kWavesPerBlock + wave) << (6 - g.ls)) + (lane >> g.ls);
  if (w < 1 || w >= g.nranges) return;
  const int32_t s0 = w * g.range;
  const int32_t s1 = (int32_t)min((int64_t)a.nnz, (int64_t)s0 + g.range);
  const int32_t r = a.tile_row[w * g.tpr];
  const int32_t p0 = a.pos[r], p1 = a.pos[r + 1];
  if (p0 >= s0 || p1 > s1) return;
  const int32_t w0 = p0 / g.range;
  const int32_t t_last = (p1 - 1) / a.tile;
  for (int32_t col = lane & ((1 << g.ls) - 1); col < a.N; col += 1 << g.ls) {
    float acc = a.carry_tail[(int64_t)w0 * g.tpr * a.N + col];
    constexpr int kH = 64;
    for (int32_t t = (w0 + 1) * g.tpr; t <= t_last; t += kH) {
      float h[kH];
#pragma unroll
      for (int k = 0; k < kH; ++k)
        h[k] = a.carry_head[(int64_t)min(t + k, t_last) * a.N + col];
#pragma unroll
      for (int k = 0; k < kH; ++k)
        if (t + k <= t_last) acc += h[k];
    }
    a.C[(int64_t)r * a.ldc + col] = acc;
  }
}

template <int DT, int V>
hipError_t launch_seg_v(const SegArgs &g, hipStream_t s) {
  if (g.nranges <= 0) return hipSuccess;
  const size_t lds = seg_lds_wave(g.range, g.a.lq, V, g.tpr, g.ls);
  const dim3 gr((unsigned)g.nranges), b(64);
  const bool comp = g.a.comp_threshold < g.a.nnz;  // some row may be compensated
  if (g.a.b_off32) {
    if (comp)
      hipLaunchKernelGGL((k_eb_seg<DT, V, true, true>), gr, b, lds, s, g);
    else
      hipLaunchKernelGGL((k_eb_seg<DT, V, true, false>), gr, b, lds, s, g);
  } else {
    if (comp)
      hipLaunchKernelGGL((k_eb_seg<DT, V, false, true>), gr, b, lds, s, g);
    else
      hipLaunchKernelGGL((k_eb_seg<DT, V, false, false>), gr, b, lds, s, g);
  }
  return hipGetLastError();
}

}  // namespace

template <int DT>
hipError_t launch_seg_t(int vec, const SegArgs &g, hipStream_t s) {
  switch (vec) {
    case 1: return launch_seg_v<DT, 1>(g, s);
    case 2: return launch_seg_v<DT, 2>(g, s);
    case 4: return launch_seg_v<DT, 4>(g, s);
    case 8:
      if constexpr (DT != 0) return launch_seg_v<DT, 8>(g, s);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}
template hipError_t launch_seg_t<SEGTACO_SEG_DT>(int, const SegArgs &, hipStream_t);

#if SEGTACO_SEG_DT == 0
namespace {
int64_t ceil_div64(int64_t a, int64_t b) { return (a + b - 1) / b; }
}  // namespace

hipError_t launch_seg(int dt, int vec, const SegArgs &g, hipStream_t s) {
  switch (dt) {
    case 0: return launch_seg_t<0>(vec, g, s);
    case 1: return launch_seg_t<1>(vec, g, s);
    case 2: return launch_seg_t<2>(vec, g, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_seg_fixup(const SegArgs &g, hipStream_t s) {
  if (g.nranges < 2) return hipSuccess;
  const int64_t per_block = (int64_t)kWavesPerBlock << (6 - g.ls);
  const int64_t grid = (g.nranges + per_block - 1) / per_block;
  hipLaunchKernelGGL(k_seg_fixup, dim3((unsigned)grid), dim3(kBlockThreads), 0, s, g);
  return hipGetLastError();
}

int32_t seg_plan(int32_t dt, const KArgs &a, int64_t walk_blocks, SegArgs *g) {
  // Which calls. Measured at tile 128 and at the default (shorter) tiles, FP32
  // and BF16, us per call, walk / segments:
  //   up to 8 columns: segments at every size (above, and 262144^2 N = 8:
  //     144 / 95 and 129 / 95);
  //   9 to 16 (N = 16, tile 128): 500 K entries 40 / 25 and 39 / 27, 960 K 43 /
  //     35 and 40 / 46, 1.2 M 41 / 42 and 38 / 54: up to 2^20 entries in FP32, 2^19
  //     in 16 bits, whose slices of 8 gather more columns than N has. Short
  //     tiles cut more pieces, and uniform rows, which the walk takes best, lose
  //     (FP32, tile 16, power-law and uniform: 500 K 47 / 35 and 22 / 26, 1 M 50 / 46
  //     and 32 / 40; BF16 1 M 65 / 62 and 33 / 50): up to 2^19 entries;
  //   17 to 64: small products (1000^2, 15.6 K entries, N = 64: 36 / 22 at
  //     tile 128, 21 / 13 at tile 8), and where the walk leaves half of the
  //     chip without a workgroup: 8000^2 N = 64 (63 workgroups) 43 / 28, but
  //     20000^2 N = 50 (156 workgroups) 40 / 46, 60000^2 N = 64 53 / 131.
  // A range has to fit the wave's LDS, and the zero fill walks M / ranges
  // rows per wave, so mostly empty matrices keep the row-parallel partition.
  if (a.tile > kSegMaxRange || a.N > 64 || (int64_t)a.M > 2 * (int64_t)a.nnz) return 0;
  const int64_t products = (int64_t)a.nnz * a.N;
  const int32_t most = dt == 0 && a.tile >= 64 ? 1 << 20 : 1 << 19;  // entries, N 9 to 16
  const bool take = a.N <= 8    ? true
                    : a.N <= 16 ? a.nnz <= most
                                : products <= 2000000 ||
                                      (products <= 12000000 && walk_blocks < 128);
  if (!take) return 0;
  SegArgs &s = *g;
  s.a = a;
  int32_t v = dt == 0 ? 4 : 8;
  while (v > a.N) v >>= 1;
  s.a.lq = 0;
  while ((v << s.a.lq) < a.N) ++s.a.lq;
  s.ls = 0;
  while ((1 << s.ls) < a.N) ++s.ls;
  // about 2048 entries per lane of a group, but at least 2048 waves
  int64_t want = std::min(std::max(2048 >> s.ls, 128), 384);
  want = std::min(want, ceil_div64(a.nnz, 2048));
  s.tpr = (int32_t)std::max<int64_t>(1, want / a.tile);
  s.range = s.tpr * a.tile;
  s.nranges = (int32_t)ceil_div64(a.nnz, s.range);
  s.slice = (int32_t)ceil_div64(a.M, s.nranges);
  if (seg_lds_wave(s.range, s.a.lq, v, s.tpr, s.ls) > 65536) return 0;
  return v;
}
#endif

}  // namespace segtaco
