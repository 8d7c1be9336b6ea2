// The wave-systolic EDR sweep shared by the batched kernels (edr_batched.hip)
// and the plain handler (edr.hip): one trajectory pair per segment of SEG
// lanes, K consecutive DP rows per lane.
//
// Values are kept as E[r][c] = D[r][c] - r, which makes two of the three
// candidates of a cell free of arithmetic (Grid.cpp:1288-1300; s = 0 on a
// match, 1 otherwise):
//   U = D[r-1][c] + 1   -> E[r-1][c]
//   M = D[r-1][c-1] + s -> E[r-1][c-1] + s - 1
//   L = D[r][c-1] + 1   -> E[r][c-1] + 1
// and the rule (M strictly smallest -> M, L strictly smallest -> L, else U)
// reduces exactly to E = (M == L) ? U : min(M, L, U).  The boundary is
// E[0][c] = c, E[r][0] = 0.
//
// What bounds it: VALU issue (4 cycles per wave64 instruction on one SIMD).
// A step of a lane is K cells of its K rows in one column: one DPP shift for
// the row above (the left lane's bottom row), then per cell an add, a min3, a
// compare and a select.  One row per lane paid the shift, a row store and a
// feed read per cell; with K = 4 they are paid once per four cells.  The match
// test (two subtractions, two compares, a borrow) is left out of a block of 16
// columns when the box of the strip's rows and the box of the columns the
// block touches lie at least u apart: then no pair of their points matches
// (see may_touch), s = 1 throughout, and M needs no arithmetic either.
#pragma once

#include <type_traits>

#include "gat_common.hpp"

namespace edr {

constexpr int kBlk = 16;    // steps per feed block
constexpr int kPad = 16;    // NaN points before every trajectory of a padded store
constexpr int kLaneRows = 4;  // most rows per lane
// Where column 0 lies in a strip's row: columns back to 2 - SEG are stored, and
// a 64-lane pair's blocks read from a multiple of four values on (column 1).
constexpr int kOff64 = 67;
template <int SEG>
constexpr int kRowOff = SEG == 64 ? kOff64 : SEG;

// Lane l of a segment takes src from lane l - 1; lane 0 keeps old.  Segments
// of 16 lanes are DPP rows (row_shr:1); a 64-lane segment is the wave
// (wave_shr:1).
template <int SEG>
__device__ __forceinline__ int shift_in(int old, int src) {
  static_assert(SEG == 16 || SEG == 64, "segments of 16 or 64 lanes");
  return __builtin_amdgcn_update_dpp(old, src, SEG == 16 ? 0x111 : 0x138, 0xf, 0xf, false);
}

__device__ __forceinline__ float2 nan_point() { return make_float2(__builtin_nanf(""), __builtin_nanf("")); }

// Point i of the n >= 1 points at P, one that matches nothing when i lies
// outside them.  The load is unconditional (clamped): behind a branch its value
// would be waited for at the branch's end, one memory latency per point.
__device__ __forceinline__ float2 point_or_nan(const float2* P, int i, int n) {
  // (The byte offset fits 32 bits, so a scalar P needs no 64-bit address.)
  const uint32_t at = uint32_t(min(max(i, 0), n - 1)) * uint32_t(sizeof(float2));
  const float2 v = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(P) + at);
  return make_float2(uint32_t(i) < uint32_t(n) ? v.x : __builtin_nanf(""), v.y);
}

// The same; in a padded store (!kGuard) point n is a NaN point, and one
// unsigned minimum takes every i outside 0 .. n - 1 to it.
template <bool kGuard>
__device__ __forceinline__ float2 point_in(const float2* P, int i, int n) {
  if constexpr (kGuard) {
    return point_or_nan(P, i, n);
  } else {
    const uint32_t at = min(uint32_t(i) * uint32_t(sizeof(float2)), uint32_t(n) * uint32_t(sizeof(float2)));
    return *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(P) + at);
  }
}

// Box tests of point sets by (xmin, ymin, xmax, ymax).  Float subtraction is
// monotone, so for points a in box q and b in box c, fl(b.x - a.x) >=
// fl(c.xmin - q.xmax): when the latter is >= u no pair of their points matches
// on x, and likewise for the other three sides.  NaN points match nothing and
// are left out of the boxes; an empty box (inf, inf, -inf, -inf) touches none.
__device__ __forceinline__ bool may_touch(const float4& q, const float4& c, float u) {
  return !((c.x - q.z) >= u || (q.x - c.z) >= u || (c.y - q.w) >= u || (q.y - c.w) >= u);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// The union of the boxes of a segment's lanes, in every lane (row_ror within
// the 16-lane rows, then across rows for a 64-lane segment).
template <int SEG>
__device__ __forceinline__ float4 segment_box(float4 b) {
#define GAT_EDR_BOX_STEP(CTRL)                                                                              \
  b = make_float4(fminf(b.x, dpp_f<CTRL>(b.x)), fminf(b.y, dpp_f<CTRL>(b.y)), fmaxf(b.z, dpp_f<CTRL>(b.z)), \
                  fmaxf(b.w, dpp_f<CTRL>(b.w)))
  GAT_EDR_BOX_STEP(0x128);
  GAT_EDR_BOX_STEP(0x124);
  GAT_EDR_BOX_STEP(0x122);
  GAT_EDR_BOX_STEP(0x121);
#undef GAT_EDR_BOX_STEP
  if constexpr (SEG == 64) {
    for (int d = 16; d < 64; d <<= 1)
      b = make_float4(fminf(b.x, __shfl_xor(b.x, d)), fminf(b.y, __shfl_xor(b.y, d)), fmaxf(b.z, __shfl_xor(b.z, d)),
                      fmaxf(b.w, __shfl_xor(b.w, d)));
  }
  return b;
}

__device__ __forceinline__ float4 empty_box() { return make_float4(INFINITY, INFINITY, -INFINITY, -INFINITY); }

// (A point of NaN x and finite y may widen the box in y only, which tests more
// and skips nothing that matches.)
__device__ __forceinline__ float4 grow(const float4& b, const float2& p) {
  return make_float4(fminf(b.x, p.x), fminf(b.y, p.y), fmaxf(b.z, p.x), fmaxf(b.w, p.y));
}

// K rows of a lane: their points, E of the row's last column, and the row
// above's E at that column.
template <int K>
struct LaneRows {
  float rx[K], ry[K];
  int e[K], next[K];  // E of the last column, and L = E + 1 of the next
  int up;
  __device__ __forceinline__ void start() {
#pragma unroll
    for (int i = 0; i < K; ++i) {
      e[i] = 0;
      next[i] = 1;
    }
    up = 0;
  }
  // Rows first .. first + K - 1 (0-based points) of the trajectory R of n points.
  template <bool kGuard>
  __device__ __forceinline__ float4 load(const float2* R, int n, int first) {
    float4 b = empty_box();
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const float2 p = point_in<kGuard>(R, first + i, n);
      rx[i] = p.x;
      ry[i] = p.y;
      b = grow(b, p);
    }
    return b;
  }
  // One column: the K cells below u0 = E of the row above.  kNear tests the
  // rows against the column's point; otherwise nothing matches.
  template <bool kNear>
  __device__ __forceinline__ void step(int u0, const float2& p, float u) {
    // The compares first: they depend on the previous column only, and a select
    // may read its mask two wait states after the compare.
    int mm[K];
    bool same[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      mm[i] = i == 0 ? up : e[i - 1];
      if constexpr (kNear) {
        const bool match = fabsf(rx[i] - p.x) < u && fabsf(ry[i] - p.y) < u;
        mm[i] -= match ? 1 : 0;
      }
      same[i] = mm[i] == next[i];
    }
    int uu = u0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const int mn = min(min(uu, next[i]), mm[i]);
      uu = same[i] ? uu : mn;
      e[i] = uu;
    }
    up = u0;
    // Last: the next column's shift reads e[K - 1] two wait states after its write.
#pragma unroll
    for (int i = 0; i < K; ++i) next[i] = e[i] + 1;
  }
};

// The type of a strip's row in LDS: 16 bits where four pairs share a wave; a
// 64-lane pair's row is read in 16-byte pieces, and 32-bit values need no
// unpacking (an instruction per step).
template <int SEG>
using RowValue = std::conditional_t<SEG == 64, int32_t, int16_t>;

// One strip: rows row0 + 1 .. row0 + SEG * K of every segment's pair across
// all its columns.  `above` holds E of the row above the strip by column
// (interleaved across the wave's segments, [column + kRowOff][segment]); it is
// read once per step as a broadcast, lane 0 of a segment taking it as the
// `old` operand of the shift, and every lane stores its bottom row's value
// into it at its own column.  The last lane stores each column last, so the
// strip leaves its bottom row behind, and each column is read (step c - 1) no
// later than its first store (lane 0, same step, after the read).
//
// Lane l computes column t - l + 1 at step t.  Before its first column a
// lane's values stay E[r][0] = 0 (its inputs are 0 and NaN points match
// nothing); past a pair's last column it computes values nobody reads.  D[n][m]
// is taken by the lane that owns row n at the step it reaches column m; the
// block it falls into is the only one that tests for it.
//
// kGuard: the store holds no padding, so every load is checked against
// 0 .. m - 1 (NaN outside).  Otherwise a NaN point follows every trajectory, and
// the padding before it covers a 16-lane segment's look-behind.
template <int SEG, int K, bool kGuard>
__device__ __forceinline__ void sweep_strip(const float2* R, int n, const float2* C, int m, int row0, int mmax,
                                            const int (&ns)[64 / SEG], const int (&ms)[64 / SEG], const float4& colbox,
                                            float u, RowValue<SEG> (*above)[64 / SEG], int seg, int l, int& res,
                                            bool& mine) {
  constexpr int kSegs = 64 / SEG;
  constexpr int kOff = kRowOff<SEG>;
  // hist: kSpread bits per block, the newest lowest; row r of a 64-lane segment
  // is at the chunks of r and r + 1 blocks ago, a 16-lane segment at the last two.
  constexpr int kSpread = SEG == 16 ? 1 : 4;
  constexpr uint32_t kWindow =
      SEG == 16 ? 0x3u : (1u << 0 | 1u << 4) | (1u << 5 | 1u << 9) | (1u << 10 | 1u << 14) | (1u << 15 | 1u << 19);
  LaneRows<K> rows;
  rows.start();
  // The box of each 16-lane row's rows.  (A 64-lane segment's rows of lanes lie
  // 16 columns apart: each is tested against the columns it is at.  One box of
  // all 256 rows against the five chunks they cover called 0.30 of a top-k
  // batch's blocks near, this 0.22.)
  const float4 rowbox = segment_box<16>(rows.template load<kGuard>(R, n, row0 + l * K));
  // Row n inside this strip: its lane, its row of the lane and the step its
  // last column comes at; the same per segment, wave-uniform.
  const int loc = n - 1 - row0;
  const bool ends = loc >= 0 && loc < SEG * K;
  const int lc = ends ? loc / K : -1, ic = ends ? loc % K : 0;
  const int tcap = l == lc ? m + l - 1 : -1;
  mine = mine || l == lc;
  int tend[kSegs];
#pragma unroll
  for (int j = 0; j < kSegs; ++j) {
    const int at = ns[j] - 1 - row0;
    tend[j] = (at >= 0 && at < SEG * K) ? ms[j] + at / K - 1 : -1;
  }
  const int steps = mmax + SEG - 1;
  const float2* cp = C - l;  // column point of step t is cp[t]
  auto column = [&](int t) __attribute__((always_inline)) -> float2 {
    if constexpr (kGuard || SEG == 64) {
      return point_in<kGuard>(C, t - l, m);
    } else {
      return cp[t];
    }
  };
  float2 src[kBlk];
  auto block = [&](auto near_c, auto cap_c, int t0) __attribute__((always_inline)) {
    constexpr bool kNear = decltype(near_c)::value, kCap = decltype(cap_c)::value;
    const RowValue<SEG>(*feed)[kSegs] = &above[kOff + t0 + 1];
    int fv[kBlk];
#pragma unroll
    for (int j = 0; j < kBlk; ++j) fv[j] = feed[j][seg];
    RowValue<SEG>(*own)[kSegs] = &above[kOff + t0 - l + 1];
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      const int u0 = shift_in<SEG>(fv[j], rows.e[K - 1]);
      rows.template step<kNear>(u0, src[j], u);
      // The same step of the next block, in flight behind the rest of this
      // one (unused when that block tests nothing).
      if constexpr (kNear) src[j] = column(t0 + kBlk + j);
      if constexpr (kCap) {
#pragma unroll
        for (int i = 0; i < K; ++i) res = (t0 + j == tcap && i == ic) ? rows.e[i] : res;
      }
      own[j][seg] = RowValue<SEG>(rows.e[K - 1]);
      // The stores of different lanes to one column come from different steps,
      // and the last lane's must stay last; per lane their addresses differ, so
      // without this the scheduler could reorder them.
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // A block of a near strip that takes a result: rolled, since it runs once
  // per pair and unrolled its masks would crowd the registers of the others.
  auto block_near_cap = [&](int t0) __attribute__((always_inline)) {
#pragma unroll 1
    for (int t = t0; t < t0 + kBlk; ++t) {
      const int fv = above[kOff + t + 1][seg];
      const float2 p = column(t);
      const int u0 = shift_in<SEG>(fv, rows.e[K - 1]);
      rows.template step<true>(u0, p, u);
#pragma unroll
      for (int i = 0; i < K; ++i) res = (t == tcap && i == ic) ? rows.e[i] : res;
      above[kOff + t - l + 1][seg] = RowValue<SEG>(rows.e[K - 1]);
    }
  };
  auto captures = [&](int t0) __attribute__((always_inline)) -> bool {
    bool c = false;
#pragma unroll
    for (int j = 0; j < kSegs; ++j) c = c || (tend[j] >= t0 && tend[j] < t0 + kBlk);
    return c;
  };
  using Yes = std::true_type;
  using No = std::false_type;
#pragma unroll
  for (int j = 0; j < kBlk; ++j) src[j] = make_float2(0.0f, 0.0f);
  if (__ballot(may_touch(rowbox, colbox, u)) == 0) {
    // No pair of the wave can match in this strip.
    for (int t0 = 0; t0 < steps; t0 += kBlk) {
      if (captures(t0)) block(No{}, Yes{}, t0);
      else block(No{}, No{}, t0);
    }
    return;
  }
  // Chunk b: columns 16 b .. 16 b + 15 of each segment, one per lane of a row.
  auto chunk = [&](int b) __attribute__((always_inline)) -> float2 {
    return point_in<kGuard>(C, b * kBlk + (l & 15), m);
  };
  auto touches = [&](const float2& p) __attribute__((always_inline)) -> uint32_t {
    const float4 cb = segment_box<16>(grow(empty_box(), p));
    const uint64_t t = __ballot(may_touch(rowbox, cb, u));
    if constexpr (SEG == 16) return t != 0 ? 1u : 0u;
    // (The same in all lanes of a row.)
    return uint32_t(t & 1u) | uint32_t(t >> 15 & 2u) | uint32_t(t >> 30 & 4u) | uint32_t(t >> 45 & 8u);
  };
  uint32_t hist = touches(chunk(0));
  float2 ahead = chunk(1);
  bool loaded = false;  // src holds this block's points
  for (int t0 = 0, b = 0; t0 < steps; t0 += kBlk, ++b) {
    const bool near = (hist & kWindow) != 0;
    const float2 pn = ahead;
    ahead = chunk(b + 2);
    const bool cap = captures(t0);
    if (near && !cap && !loaded) {
#pragma unroll
      for (int j = 0; j < kBlk; ++j) src[j] = column(t0 + j);
    }
    loaded = near && !cap;
    if (near) {
      if (cap) block_near_cap(t0);
      else block(Yes{}, No{}, t0);
    } else {
      if (cap) block(No{}, Yes{}, t0);
      else block(No{}, No{}, t0);
    }
    hist = (hist << kSpread) | touches(pn);
  }
}

// The box of a segment's columns (0 .. m - 1).
template <int SEG>
__device__ __forceinline__ float4 columns_box(const float2* C, int m, int l) {
  float4 b = empty_box();
#pragma unroll 4
  for (int i = l; i < m; i += SEG) b = grow(b, C[i]);
  return segment_box<SEG>(b);
}

// The whole sweep of the wave's pairs (rows R of n points, columns C of m >= n
// points, n = m = 0 for an idle segment): strips of SEG * kLaneRows rows, the
// last of as many rows per lane as it needs.  `above` holds E of row 0 on
// entry.  *mine: this lane holds its segment's E[n][m] in the return value.
template <int SEG, bool kGuard>
__device__ __forceinline__ int sweep_pairs(const float2* R, int n, const float2* C, int m, int nmax, int mmax,
                                           const int (&ns)[64 / SEG], const int (&ms)[64 / SEG], float u,
                                           RowValue<SEG> (*above)[64 / SEG], int seg, int l, bool* mine) {
  const float4 colbox = columns_box<SEG>(C, m, l);
  int res = 0;
  bool got = false;
  for (int row0 = 0; row0 < nmax;) {
    // Orders the previous strip's (or the initial) writes of `above` before
    // this strip's reads of them by other lanes.
    __syncthreads();
    // Four rows per lane while that many are left, then two (three lane rows
    // take a strip of two and one of one: 14 VALU per step against 13 for a
    // variant of their own), then one.
    const int left = (nmax - row0 + SEG - 1) / SEG;
    if (left >= 4) {
      sweep_strip<SEG, 4, kGuard>(R, n, C, m, row0, mmax, ns, ms, colbox, u, above, seg, l, res, got);
      row0 += 4 * SEG;
    } else if (left >= 2) {
      sweep_strip<SEG, 2, kGuard>(R, n, C, m, row0, mmax, ns, ms, colbox, u, above, seg, l, res, got);
      row0 += 2 * SEG;
    } else {
      sweep_strip<SEG, 1, kGuard>(R, n, C, m, row0, mmax, ns, ms, colbox, u, above, seg, l, res, got);
      row0 += SEG;
    }
  }
  *mine = got;
  return res;
}

}  // namespace edr
