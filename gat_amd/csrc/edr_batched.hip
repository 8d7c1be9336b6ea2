// Batched EDR for gfx950: many (query, candidate) pairs in one persistent
// launch.  Same recurrence as Grid::SimilarityExecuter (Grid.cpp:1222-1318);
// no reference counterpart for the batching itself.
//
// Wave-systolic layout (edr_dp.hpp).  A wave64 runs four independent pairs, one
// per 16-lane DPP row ("segment"), or one long pair over all 64 lanes.  Inside
// a segment of S lanes, lane l owns K consecutive DP rows of a strip of S * K
// rows and computes them for column t - l + 1 at step t, so a strip sweeps its
// rows across all columns in m + S - 1 steps: the row above comes from the left
// lane's bottom row of the step before (a DPP shift), everything else from the
// lane's own registers.  The first lane's row above the strip is kept in LDS
// as 16-bit values, into which every lane stores its bottom row, the strip's
// last lane last.
//
// Work: jobs of up to four pairs (one for 64-lane segments) with the same
// strip count, ordered longest first, handed out by one atomic counter per
// launch, so the batch's tail is short and no host round trip separates length
// buckets.
#include <cmath>

#include "edr_dp.hpp"
#include "gat_common.hpp"

namespace {

using edr::kBlk;
using edr::kPad;

struct Job {
  int32_t first, count;
};
static_assert(sizeof(Job) == sizeof(gat_edr_job), "job layout");

// A launch over a window of the job array: jobs [window[0], window[0] +
// window[1]) of the njobs the array holds, the window written on the device
// (by edr_jobs_kernel) after the launch was queued.
__device__ __forceinline__ int32_t take_window(const int32_t* window, int32_t& njobs) {
  if (!window) return 0;
  const int32_t first = min(max(window[0], 0), njobs);
  njobs = min(njobs - first, max(window[1], 0));
  return first;
}


__device__ __forceinline__ int64_t uniform64(int64_t v) {
  const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))));
  const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(uint64_t(v) >> 32))));
  return int64_t(uint64_t(lo) | (uint64_t(hi) << 32));
}

// Issue priority of a wave by the length of its job's schedule in steps:
// the longest pairs of a batch set its end, so their waves go first.
__device__ __forceinline__ void job_priority(int64_t steps) {
  if (steps >= 16384) __builtin_amdgcn_s_setprio(3);
  else if (steps >= 8192) __builtin_amdgcn_s_setprio(2);
  else if (steps >= 4096) __builtin_amdgcn_s_setprio(1);
  else __builtin_amdgcn_s_setprio(0);
}

// Without a job list (jobs null) a launch runs pairs 0 .. *live - 1 one per job,
// in the order given, or none when *live exceeds the npairs the array holds;
// *cells gets their cell count and *stamp the time the launch began.
struct RawPairs {
  const unsigned long long* live;
  unsigned long long* cells;
  uint32_t* stamp;
};

__device__ __forceinline__ int32_t raw_jobs(const RawPairs& raw, int64_t npairs) {
  const unsigned long long n = *raw.live;
  return n > (unsigned long long)npairs ? 0 : int32_t(n);
}

__device__ __forceinline__ void store_clock(uint32_t* p) {
  const uint64_t t = wall_clock64();
  p[0] = uint32_t(t);
  p[1] = uint32_t(t >> 32);
}

// SEG lanes per pair: 16 (four pairs per wave) or 64 (one pair per wave, a
// quarter of the strips, for the longest pairs, whose strips would otherwise
// run one after another for milliseconds).  Waves per SIMD each class can hold:
// four 16-lane pairs' rows of 2048 columns (16.8 KB of LDS per wave) cap that
// class at two; the others are held to 128 VGPRs so four fit.
template <int MAXM, int SEG>
__global__ __launch_bounds__(64, (MAXM >= 2048 && SEG == 16) ? 2 : 4) void edr_wave_kernel(const int2* __restrict__ pairs, int64_t npairs,
                                                      const Job* __restrict__ jobs, int32_t njobs,
                                                      const int32_t* __restrict__ window,
                                                      int32_t* __restrict__ counter, int32_t nqueries, int32_t ncands,
                                                      const float2* __restrict__ qxy, const int64_t* __restrict__ qoff,
                                                      const int32_t* __restrict__ qlen, const float2* __restrict__ cxy,
                                                      const int64_t* __restrict__ coff,
                                                      const int32_t* __restrict__ clen, float u,
                                                      int32_t* __restrict__ out, RawPairs raw) {
  constexpr int kSeg = SEG;        // lanes per pair
  constexpr int kSegs = 64 / SEG;  // pairs per wave
  // Row above the current strip, E[r0][c] = D[r0][c] - r0, at [c + kOff][segment]
  // for columns 2 - SEG .. MAXM + SEG + kBlk - 1 (the lanes' look-behind, the
  // columns, and the last blocks' overrun).  Segments interleave, so one
  // segment's consecutive columns are 2 * kSegs bytes apart and each step's
  // feed is a load of its own; a 64-lane pair's are 32 bits each, read four at
  // a time.
  constexpr int kOff = edr::kRowOff<SEG>;
  constexpr int kRows = kOff + MAXM + SEG + kBlk;
  __shared__ __align__(16) edr::RowValue<SEG> above[kRows][kSegs];
  const int lane = threadIdx.x;
  const int seg = lane / kSeg;
  const int l = lane & (kSeg - 1);
  if (jobs) jobs += take_window(window, njobs);
  else njobs = raw_jobs(raw, npairs);
  if (raw.stamp && blockIdx.x == 0 && lane == 0) store_clock(raw.stamp);
  for (;;) {
    int ji = 0;
    if (lane == 0) ji = atomicAdd(counter, 1);
    ji = __builtin_amdgcn_readfirstlane(ji);
    if (ji < 0 || ji >= njobs) break;  // a counter that was not cleared hands out nothing
    const Job job = jobs ? jobs[ji] : Job{ji, 1};
    // Jobs and pairs that point outside their arrays are skipped.
    const bool live = seg < job.count && job.first >= 0 && int64_t(job.first) + seg < npairs;
    int n = 0, m = 0;
    // Dead segments read rows nowhere (n = 0) and columns from the store's
    // first trajectory, whose leading padding covers the lanes' look-behind
    // (loads further back than the padding are replaced by NaN, below).
    const float2* R = cxy;
    const float2* C = cxy + kPad;
    int64_t row_off = 0, col_off = kPad;
    bool valid = false, query_rows = false;
    if (live) {
      const int2 pr = pairs[job.first + seg];
      const bool ids_ok = pr.x >= 0 && pr.x < nqueries && pr.y >= 0 && pr.y < ncands;
      const int nq = ids_ok ? qlen[pr.x] : 0, nc = ids_ok ? clen[pr.y] : 0;
      // Lengths outside 1..MAXM (and bad ids) are reported as -1 and never indexed.
      valid = nq >= 1 && nc >= 1 && nq <= MAXM && nc <= MAXM;
      if (valid) {
        // Rows are the shorter trajectory; on equal lengths the query
        // (Grid.cpp:1234-1247).
        query_rows = nc >= nq;
        row_off = query_rows ? qoff[pr.x] : coff[pr.y];
        col_off = query_rows ? coff[pr.y] : qoff[pr.x];
        R = (query_rows ? qxy : cxy) + row_off;
        C = (query_rows ? cxy : qxy) + col_off;
        n = query_rows ? nq : nc;
        m = query_rows ? nc : nq;
      }
    }
    if constexpr (kSegs == 1) {
      // One pair for the whole wave: its pointers and lengths are scalars.
      n = __builtin_amdgcn_readfirstlane(n);
      m = __builtin_amdgcn_readfirstlane(m);
      const bool q_rows = __builtin_amdgcn_readfirstlane(query_rows ? 1 : 0) != 0;
      R = (q_rows ? qxy : cxy) + uniform64(row_off);
      C = (q_rows || !valid ? cxy : qxy) + uniform64(col_off);
    }
    // Wave-uniform extents: the largest column count and strip count of the job.
    const int m0 = __builtin_amdgcn_readlane(m, 0), m1 = __builtin_amdgcn_readlane(m, 16);
    const int m2 = __builtin_amdgcn_readlane(m, 32), m3 = __builtin_amdgcn_readlane(m, 48);
    const int mmax = max(max(m0, m1), max(m2, m3));
    if (raw.cells && l == 0 && valid) atomicAdd(raw.cells, (unsigned long long)n * (unsigned long long)m);
    const int n0 = __builtin_amdgcn_readlane(n, 0), n1 = __builtin_amdgcn_readlane(n, 16);
    const int n2 = __builtin_amdgcn_readlane(n, 32), n3 = __builtin_amdgcn_readlane(n, 48);
    const int nmax = max(max(n0, n1), max(n2, n3));
    const int strips = (nmax + kSeg * edr::kLaneRows - 1) / (kSeg * edr::kLaneRows);
    job_priority(int64_t(strips) * (mmax + kSeg - 1) * 2);
    // Row 0: E[0][c] = c, as far as the job's last block reads.  (Kept rolled:
    // unrolled, its length grows with MAXM and so does the register count.)
    const int used = min(kRows, kOff + mmax + SEG + kBlk);
#pragma unroll 2
    for (int i = l; i < used; i += kSeg) above[i][seg] = edr::RowValue<SEG>(i - kOff);
    int ns[kSegs], ms[kSegs];
    if constexpr (kSegs == 4) {
      ns[0] = n0; ns[1] = n1; ns[2] = n2; ns[3] = n3;
      ms[0] = m0; ms[1] = m1; ms[2] = m2; ms[3] = m3;
    } else {
      ns[0] = n0;
      ms[0] = m0;
    }
    bool mine = false;
    const int res = edr::sweep_pairs<SEG, false>(R, n, C, m, nmax, mmax, ns, ms, u, above, seg, l, &mine);
    __syncthreads();  // the next job re-initialises `above`
    if (live && !valid && l == 0) out[job.first + seg] = -1;
    if (valid && mine) out[job.first + seg] = res + n;  // D = E + n
  }
}

// One pair over W waves of a workgroup (no reference counterpart): wave w
// runs the pair's strips w, w + W, ... of 64 * K rows in lockstep with the
// others, one block of 16 steps per iteration and a workgroup barrier between
// iterations, so a pair's strips overlap instead of running one after another.
// A strip reads the row above it from the previous strip's wave: that wave's
// last lane writes its bottom row, E per column, into the wave's own LDS row
// buffer at step c + 62 for column c, and the consumer reads column c at step
// c - 1 of its own strip; a block's feed is read one block ahead of its use.
// So a strip starts kLag = 6 blocks after the previous one (column 16b + 32,
// the last read during a consumer's block b, is written in the producer's
// block b + 5), and no sooner than its wave has finished its previous strip —
// which also keeps a wave's writes to its buffer behind the next wave's reads
// of the previous contents (those reads start kLag blocks earlier on every
// column).  Every wave runs the same number of iterations, so the barriers
// always match.  The cell rule, the row/column orientation, the far-block test
// and the capture of D[n][m] are sweep_strip's (edr_dp.hpp) with 64-lane
// segments; K (1, 2 or 4) is the least that gives every wave at most one strip,
// up to 4: a wave is alone on its SIMD here, so a step costs its instructions
// (17 VALU at K = 4, 5 at K = 1) and fewer rows per lane end a pair sooner.
constexpr int kLag = 6;

template <int MAXM, int W>
struct PipeShared {
  // Columns -62 .. 0 sit before column 0 (lane 63's look-behind); a block's
  // feed, read a block ahead, goes up to column 16 * nblocks + 16 <= m + 94.
  static constexpr int kOff = 64;
  static constexpr int kLen = kOff + MAXM + 112;
  int16_t rows[W + 1][kLen];  // [W]: row 0, E[0][c] = c
  // The column trajectory, columns -63 .. 16 * nblocks + 15 (<= m + 93) at
  // [kColOff + column], NaN outside 0 .. m - 1: too few waves run here to hide
  // a global load's latency behind a block's 16 steps.
  static constexpr int kColOff = 64;
  static constexpr int kColLen = kColOff + MAXM + 96;
  float2 cols[kColLen];
  static constexpr int kChunks = MAXM / kBlk;
  float4 chunk[kChunks];  // boxes of columns 16 b .. 16 b + 15
  int32_t job_slot;
};

template <int K, int MAXM, int W>
__device__ __forceinline__ void pipe_pair(PipeShared<MAXM, W>& sh, const float2* R, int n, int m, float u, int wv,
                                          int l, int32_t* out) {
  using S = PipeShared<MAXM, W>;
  constexpr int kRows = 64 * K;
  const int strips = (n + kRows - 1) / kRows;
  const int steps = m + 63;
  const int nblocks = (steps + kBlk - 1) / kBlk;
  const int nchunks = (m + kBlk - 1) / kBlk;
  // Strip s starts at block (s / W) * P + (s % W) * kLag, P = max(nblocks,
  // W * kLag): kLag after strip s - 1 and P >= nblocks after the same wave's
  // previous strip.
  const int P = max(nblocks, W * kLag);
  const int kend = ((strips - 1) / W) * P + ((strips - 1) % W) * kLag + nblocks;
  __builtin_amdgcn_s_setprio(3);  // these pairs set the batch's end
  edr::LaneRows<K> rows;
  rows.start();
  int s = wv, start = wv * kLag;
  int tcap = -1, ic = 0, tend = -1, res = 0;
  bool mine = false;
  uint64_t near0 = 0, near1 = 0, near2 = 0;  // blocks of the strip that may match
  bool loaded = false;
  float2 src[kBlk];
  int fv[kBlk];
#pragma unroll
  for (int j = 0; j < kBlk; ++j) {
    src[j] = make_float2(0.0f, 0.0f);
    fv[j] = 0;
  }
  const int16_t* above = sh.rows[W];
  int16_t* own = sh.rows[wv];
  auto begin_strip = [&]() __attribute__((always_inline)) {
    rows.start();
    // Each 16-lane row of lanes against the columns it is at: row r, block b,
    // the chunks b - r and b - r - 1 (as in sweep_strip).
    const float4 own_box = edr::segment_box<16>(rows.template load<true>(R, n, s * kRows + l * K));
    float4 cb[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int c = l + 64 * i;
      cb[i] = c < nchunks ? sh.chunk[min(c, S::kChunks - 1)] : edr::empty_box();
    }
    near0 = near1 = near2 = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const auto row = [&](float v) __attribute__((always_inline)) {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16 * r));
      };
      const float4 box = make_float4(row(own_box.x), row(own_box.y), row(own_box.z), row(own_box.w));
      const uint64_t t0 = __ballot(edr::may_touch(box, cb[0], u)), t1 = __ballot(edr::may_touch(box, cb[1], u)),
                     t2 = __ballot(edr::may_touch(box, cb[2], u));
#pragma unroll
      for (int d = r; d < r + 2; ++d) {
        near0 |= t0 << d;
        near1 |= t1 << d | (d ? t0 >> (64 - d) : 0);
        near2 |= t2 << d | (d ? t1 >> (64 - d) : 0);
      }
    }
    loaded = false;
    const int loc = n - 1 - s * kRows;  // < kRows in the last strip only
    const bool ends = loc < kRows;
    ic = ends ? loc % K : 0;
    tend = ends ? m + loc / K - 1 : -1;
    const bool here = ends && l == loc / K;
    tcap = here ? tend : -1;
    mine = mine || here;
    above = sh.rows[s == 0 ? W : (s - 1) % W] + S::kOff + 1;
#pragma unroll
    for (int j = 0; j < kBlk; ++j) fv[j] = above[j];
  };
  auto column = [&](int t) __attribute__((always_inline)) { return sh.cols[S::kColOff + t - l]; };
  auto block = [&](auto near_c, auto cap_c, int t0) __attribute__((always_inline)) {
    constexpr bool kNear = decltype(near_c)::value, kCap = decltype(cap_c)::value;
    int bottom[kBlk];
    const int16_t* feed = above + t0 + kBlk;
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      const int u0 = edr::shift_in<64>(fv[j], rows.e[K - 1]);
      rows.template step<kNear>(u0, src[j], u);
      if constexpr (kCap) {
#pragma unroll
        for (int i = 0; i < K; ++i) res = (t0 + j == tcap && i == ic) ? rows.e[i] : res;
      }
      bottom[j] = rows.e[K - 1];
      fv[j] = feed[j];
      if constexpr (kNear) src[j] = column(t0 + kBlk + j);
      __builtin_amdgcn_sched_barrier(0);
    }
    // The last lane's cells after the chain of steps: a branch per step would
    // sit in its way.
    if (l == 63) {
      int16_t* dst = own + S::kOff + t0 - 62;
#pragma unroll
      for (int j = 0; j < kBlk; ++j) dst[j] = int16_t(bottom[j]);
    }
  };
  auto block_near_cap = [&](int t0) __attribute__((always_inline)) {
#pragma unroll 1
    for (int t = t0; t < t0 + kBlk; ++t) {
      const int u0 = edr::shift_in<64>(above[t], rows.e[K - 1]);
      rows.template step<true>(u0, column(t), u);
#pragma unroll
      for (int i = 0; i < K; ++i) res = (t == tcap && i == ic) ? rows.e[i] : res;
      if (l == 63) own[S::kOff + t - 62] = int16_t(rows.e[K - 1]);
    }
  };
  for (int k = 0; k < kend; ++k) {
    const int b = k - start;
    if (b >= 0 && s < strips) {
      if (b == 0) begin_strip();
      const int t0 = b * kBlk;
      const uint64_t word = b < 64 ? near0 : b < 128 ? near1 : near2;
      const bool near = (word >> (b & 63)) & 1u;
      const bool cap = tend >= t0 && tend < t0 + kBlk;
      if (near) {
        if (cap) {
          block_near_cap(t0);
#pragma unroll
          for (int j = 0; j < kBlk; ++j) fv[j] = above[t0 + kBlk + j];
          loaded = false;
        } else {
          if (!loaded) {
#pragma unroll
            for (int j = 0; j < kBlk; ++j) src[j] = column(t0 + j);
          }
          block(std::true_type{}, std::false_type{}, t0);
          loaded = true;
        }
      } else {
        if (cap) block(std::false_type{}, std::true_type{}, t0);
        else block(std::false_type{}, std::false_type{}, t0);
        loaded = false;
      }
      if (b == nblocks - 1) {
        s += W;
        start += P;
      }
    }
    __syncthreads();
  }
  if (mine) *out = res + n;  // D = E + n
}

template <int MAXM, int W>
__global__ __launch_bounds__(64 * W) void edr_pipe_kernel(const int2* __restrict__ pairs, int64_t npairs,
                                                          const Job* __restrict__ jobs, int32_t njobs,
                                                          const int32_t* __restrict__ window,
                                                          int32_t* __restrict__ counter, int32_t nqueries,
                                                          int32_t ncands, const float2* __restrict__ qxy,
                                                          const int64_t* __restrict__ qoff,
                                                          const int32_t* __restrict__ qlen,
                                                          const float2* __restrict__ cxy,
                                                          const int64_t* __restrict__ coff,
                                                          const int32_t* __restrict__ clen, float u,
                                                          int32_t* __restrict__ out, RawPairs raw) {
  using S = PipeShared<MAXM, W>;
  __shared__ S sh;
  const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / 64);
  const int l = threadIdx.x & 63;
  if (jobs) jobs += take_window(window, njobs);
  else njobs = raw_jobs(raw, npairs);
  if (raw.stamp && blockIdx.x == 0 && threadIdx.x == 0) store_clock(raw.stamp);
  for (int i = threadIdx.x; i < S::kLen; i += 64 * W) sh.rows[W][i] = int16_t(i - S::kOff);
  for (;;) {
    if (threadIdx.x == 0) sh.job_slot = atomicAdd(counter, 1);
    __syncthreads();
    const int ji = __builtin_amdgcn_readfirstlane(sh.job_slot);
    __syncthreads();  // every wave has read the slot before the next job overwrites it
    if (ji < 0 || ji >= njobs) break;  // a counter that was not cleared hands out nothing
    const Job job = jobs ? jobs[ji] : Job{ji, 1};
    // One pair per job; everything below is uniform across the workgroup.
    const bool live = job.count >= 1 && job.first >= 0 && int64_t(job.first) < npairs;
    int n = 0, m = 0;
    int64_t row_off = 0, col_off = 0;
    bool valid = false, query_rows = false;
    if (live) {
      const int2 pr = pairs[job.first];
      const bool ids_ok = pr.x >= 0 && pr.x < nqueries && pr.y >= 0 && pr.y < ncands;
      const int nq = ids_ok ? qlen[pr.x] : 0, nc = ids_ok ? clen[pr.y] : 0;
      valid = nq >= 1 && nc >= 1 && nq <= MAXM && nc <= MAXM;
      if (valid) {
        query_rows = nc >= nq;
        row_off = query_rows ? qoff[pr.x] : coff[pr.y];
        col_off = query_rows ? coff[pr.y] : qoff[pr.x];
        n = query_rows ? nq : nc;
        m = query_rows ? nc : nq;
      }
    }
    if (!valid) {
      if (live && threadIdx.x == 0) out[job.first] = -1;
      continue;
    }
    // One pair for the whole workgroup: its pointers and lengths are scalars.
    n = __builtin_amdgcn_readfirstlane(n);
    m = __builtin_amdgcn_readfirstlane(m);
    const bool q_rows = __builtin_amdgcn_readfirstlane(query_rows ? 1 : 0) != 0;
    const float2* R = (q_rows ? qxy : cxy) + uniform64(row_off);
    const float2* C = (q_rows ? cxy : qxy) + uniform64(col_off);
    if (raw.cells && threadIdx.x == 0) atomicAdd(raw.cells, (unsigned long long)n * (unsigned long long)m);
    // Stage the columns the blocks read, a box per chunk of 16.
    for (int i = int(threadIdx.x) - 64; i < m + 96; i += 64 * W) {
      const float2 p = edr::point_or_nan(C, i, m);
      sh.cols[S::kColOff + i] = p;
      // 64 divides the stride and the start: a row of 16 lanes holds one chunk.
      const float4 box = edr::segment_box<16>(edr::grow(edr::empty_box(), p));
      if ((threadIdx.x & 15) == 0 && i >= 0 && i < m) sh.chunk[i / kBlk] = box;
    }
    __syncthreads();
    const int per = (n + 64 * W - 1) / (64 * W);
    if (per <= 1) pipe_pair<1>(sh, R, n, m, u, wv, l, out + job.first);
    else if (per == 2) pipe_pair<2>(sh, R, n, m, u, wv, l, out + job.first);
    else pipe_pair<4>(sh, R, n, m, u, wv, l, out + job.first);
    // (pipe_pair ends at a barrier: the next job may reuse the buffers.)
  }
}

// Candidate filter: a (query, candidate) pair can contain a matching point
// pair only if neither box lies a float-difference of u or more beyond the
// other on either axis.  Float subtraction is monotone, so for points a (query)
// and b (candidate) with b.x >= cand.xmin and a.x <= query.xmax,
// fl(b.x - a.x) >= fl(cand.xmin - query.xmax): when the latter is >= u no point
// pair matches on x, and likewise for the other three sides.  Pairs the filter
// drops have no match at all, so their distance is the all-mismatch value.
__device__ __forceinline__ bool may_match(const float4& q, const float4& c, float u) {
  return !((c.x - q.z) >= u || (q.x - c.z) >= u || (c.y - q.w) >= u || (q.y - c.w) >= u);
}

// A workgroup tests kFilterQ queries against its candidates: each lane keeps
// its candidate's box in registers across the queries, so the candidate boxes
// are read once per kFilterQ queries instead of once per query.  The order of
// the output pairs is not defined.
constexpr int kFilterQ = 16;

__global__ __launch_bounds__(256) void edr_filter_kernel(const float4* __restrict__ qbox, int32_t nq,
                                                         const float4* __restrict__ cbox, int32_t nc, float u,
                                                         int2* __restrict__ out, uint64_t capacity,
                                                         unsigned long long* __restrict__ count) {
  __shared__ float4 qs[kFilterQ];
  const int q0 = int(blockIdx.y) * kFilterQ;
  if (threadIdx.x < kFilterQ && q0 + int(threadIdx.x) < nq) qs[threadIdx.x] = qbox[q0 + int(threadIdx.x)];
  __syncthreads();
  const int nqb = min(kFilterQ, nq - q0);
  const int lane = threadIdx.x & 63;
  for (int c = blockIdx.x * 256 + threadIdx.x; c - lane < nc; c += gridDim.x * 256) {
    const float4 cb = c < nc ? cbox[c] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int j = 0; j < nqb; ++j) {
      const bool keep = c < nc && may_match(qs[j], cb, u);
      const uint64_t mask = __ballot(keep);
      if (mask == 0) continue;
      unsigned long long base = 0;
      if (lane == 0) base = atomicAdd(count, (unsigned long long)__popcll(mask));
      base = __builtin_amdgcn_readfirstlane(uint32_t(base)) |
             (uint64_t(__builtin_amdgcn_readfirstlane(uint32_t(base >> 32))) << 32);
      const uint64_t at = base + __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
      if (keep && at < capacity) out[at] = make_int2(q0 + j, c);
    }
  }
}

// The same filter through a grid over the candidates' boxes (no reference
// counterpart): every candidate whose box spans at most kGridMaxCells cells
// is listed in each cell it touches (gat_edr_cand_grid, built by the host);
// a query tests the candidates of the cells its box, widened by u and one
// cell on every side, touches, so it sees every candidate that could pass
// may_match (keep implies c.xmin < q.xmax + u and c.xmax > q.xmin - u in
// exact arithmetic, and the widening covers the rounding of the cell of
// q.xmax + u).  A pair is reported by one cell only: the one at (max(cell of
// c.xmin, first column), max(cell of c.ymin, first row)), which both the
// candidate's cells and the query's hold.  Candidates the grid does not list
// (boxes not finite, inverted or too wide) are tested by every query, and a
// query whose box is not finite or inverted tests every candidate.  One wave
// per query; the output set equals edr_filter_kernel's.
struct CandGrid {
  int32_t g;
  float x0, y0, inv_x, inv_y;
  const uint32_t* start;  // g * g + 1 entry offsets, cells row by row
  const int32_t* id;
  const float4* box;
  const int32_t* always;
  int32_t nalways;
};

// Cell column (or row) of v: floor((v - o) * inv) clamped to 0 .. g - 1 (the
// host lists candidates with the same float operations).
__device__ __forceinline__ int grid_cell(float v, float o, float inv, int g) {
  const float t = floorf((v - o) * inv);
  return int(fminf(fmaxf(t, 0.0f), float(g - 1)));
}

constexpr int kGridFilterWaves = 4;

__global__ __launch_bounds__(64 * kGridFilterWaves) void edr_filter_grid_kernel(
    const float4* __restrict__ qbox, int32_t nq, const float4* __restrict__ cbox, int32_t nc, CandGrid gr, float u,
    int2* __restrict__ out, uint64_t capacity, unsigned long long* __restrict__ count,
    uint32_t* __restrict__ stamp) {
  if (stamp && blockIdx.x == 0 && threadIdx.x == 0) store_clock(stamp);
  const int lane = threadIdx.x & 63;
  const int q = int(blockIdx.x) * kGridFilterWaves + int(threadIdx.x >> 6);
  if (q >= nq) return;  // the whole wave
  const float4 qb = qbox[q];
  auto emit = [&](bool keep, int c) __attribute__((always_inline)) {
    const uint64_t mask = __ballot(keep);
    if (mask == 0) return;
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(count, (unsigned long long)__popcll(mask));
    base = __builtin_amdgcn_readfirstlane(uint32_t(base)) |
           (uint64_t(__builtin_amdgcn_readfirstlane(uint32_t(base >> 32))) << 32);
    const uint64_t at = base + __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
    if (keep && at < capacity) out[at] = make_int2(q, c);
  };
  const bool boxed = isfinite(qb.x) && isfinite(qb.y) && isfinite(qb.z) && isfinite(qb.w) && qb.x <= qb.z &&
                     qb.y <= qb.w;
  if (!boxed) {
    for (int c0 = 0; c0 < nc; c0 += 64) {
      const int c = c0 + lane;
      emit(c < nc && may_match(qb, cbox[c], u), c);
    }
    return;
  }
  for (int a0 = 0; a0 < gr.nalways; a0 += 64) {
    const int a = a0 + lane;
    const int c = a < gr.nalways ? gr.always[a] : 0;
    emit(a < gr.nalways && c >= 0 && c < nc && may_match(qb, cbox[c], u), c);
  }
  const int cx0 = max(grid_cell(qb.x - u, gr.x0, gr.inv_x, gr.g) - 1, 0);
  const int cx1 = min(grid_cell(qb.z + u, gr.x0, gr.inv_x, gr.g) + 1, gr.g - 1);
  const int cy0 = max(grid_cell(qb.y - u, gr.y0, gr.inv_y, gr.g) - 1, 0);
  const int cy1 = min(grid_cell(qb.w + u, gr.y0, gr.inv_y, gr.g) + 1, gr.g - 1);
  const int wx = cx1 - cx0 + 1, ncells = wx * (cy1 - cy0 + 1);
  for (int k0 = 0; k0 < ncells; k0 += 64) {
    // Lane k takes cell k0 + k; its entries are numbered after the lower lanes'.
    const int k = k0 + lane;
    int cellx = 0, celly = 0;
    uint32_t s = 0, cnt = 0;
    if (k < ncells) {
      cellx = cx0 + k % wx;
      celly = cy0 + k / wx;
      const int cell = celly * gr.g + cellx;
      s = gr.start[cell];
      cnt = gr.start[cell + 1] - s;
    }
    uint32_t incl = cnt;
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = uint32_t(__shfl_up(int(incl), d, 64));
      if (lane >= d) incl += y;
    }
    const uint32_t total = uint32_t(__builtin_amdgcn_readlane(int(incl), 63));
    for (uint32_t i0 = 0; i0 < total; i0 += 64) {
      const uint32_t i = i0 + uint32_t(lane);
      // The lane whose cell holds entry i: the first with incl > i.
      int j = 0;
      for (int step = 32; step >= 1; step >>= 1)
        if (uint32_t(__shfl(int(incl), j + step - 1, 64)) <= i) j += step;
      j = min(j, 63);
      const uint32_t sj = uint32_t(__shfl(int(s), j, 64));
      const uint32_t before = uint32_t(__shfl(int(incl), j, 64)) - uint32_t(__shfl(int(cnt), j, 64));
      const int jx = __shfl(cellx, j, 64), jy = __shfl(celly, j, 64);
      bool keep = false;
      int c = 0;
      if (i < total) {
        const uint32_t e = sj + (i - before);
        const float4 b = gr.box[e];
        c = gr.id[e];
        const int rx = max(grid_cell(b.x, gr.x0, gr.inv_x, gr.g), cx0);
        const int ry = max(grid_cell(b.y, gr.y0, gr.inv_y, gr.g), cy0);
        keep = rx == jx && ry == jy && c >= 0 && c < nc && may_match(qb, b, u);
      }
      emit(keep, c);
    }
  }
}

// The all-mismatch table: out[r * (maxlen + 1) + c] = D[r][c] of the recurrence
// with every substitution costing 1, for 0 <= r, c <= maxlen.  A pair of
// lengths n <= m with no matching point has distance out[n][m].  A serial chain
// of 2 * maxlen anti-diagonals: one workgroup with a barrier after each took
// 2.32 ms, which an index's first top-k waited for.  In two launches: a
// workgroup sweeps strips of 256 rows as the EDR kernels do (edr_dp.hpp), a
// barrier per 16 columns, and keeps every 64th row; then a wave per 64 rows
// sweeps them again from the row above and stores them all, 64 bytes per lane
// (4.2M values stored by the one workgroup would take its CU 0.45 ms alone): 0.36
// and 0.09 ms.
constexpr int kTabWaves = 8, kTabRows = 256, kTabLag = 5;  // lane 63 is 62 columns behind: blocks b .. b + 4
constexpr int kTabRing = 128;                             // a reader is at most 79 columns behind

__global__ __launch_bounds__(64 * kTabWaves) void edr_mismatch_rows_kernel(int32_t maxlen, int32_t* __restrict__ out) {
  __shared__ int32_t ring[kTabWaves][kTabRing];
  static_assert(kTabWaves * kTabRows >= GAT_MAX_TRAJ_LEN, "the waves cover every row");
  const int64_t w = maxlen + 1;
  for (int64_t c = threadIdx.x; c < w; c += blockDim.x) {
    out[c] = int32_t(c);
    out[c * w] = int32_t(c);
  }
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int nblocks = (maxlen + 63 + kBlk - 1) / kBlk;
  const int kend = nblocks + (kTabWaves - 1) * kTabLag;
  const int row = wv * kTabRows + (l + 1) * 4;  // the lane's last row
  edr::LaneRows<4> rows;
  rows.start();
  for (int k = 0; k < kend; ++k) {
    const int b = k - wv * kTabLag;
    if (b >= 0 && b < nblocks && wv * kTabRows < maxlen) {
      const int t0 = b * kBlk;
      int bottom[kBlk];
#pragma unroll
      for (int j = 0; j < kBlk; ++j)
        bottom[j] = wv == 0 ? t0 + j + 1 : ring[wv == 0 ? 0 : wv - 1][(t0 + j + 1) & (kTabRing - 1)];
#pragma unroll
      for (int j = 0; j < kBlk; ++j) {
        const int u0 = edr::shift_in<64>(bottom[j], rows.e[3]);
        rows.step<false>(u0, make_float2(0.0f, 0.0f), 0.0f);
        bottom[j] = rows.e[3];
      }
      if ((l & 15) == 15) {
#pragma unroll
        for (int j = 0; j < kBlk; ++j) {
          const int c = t0 + j - l + 1;
          if (l == 63) ring[wv][c & (kTabRing - 1)] = bottom[j];
          if (c >= 1 && c <= maxlen && row <= maxlen) out[row * w + c] = bottom[j] + row;
        }
      }
    }
    __syncthreads();
  }
}

struct alignas(4) FourInts {
  int32_t v[4];
};

__global__ __launch_bounds__(64) void edr_mismatch_fill_kernel(int32_t maxlen, int32_t* __restrict__ out) {
  const int64_t w = maxlen + 1;
  const int l = threadIdx.x;
  const int r0 = int(blockIdx.x) * 64, row = r0 + l + 1;
  const int steps = maxlen + 63;
  const bool mine = row <= maxlen && l < 63;  // every 64th row is there already
  edr::LaneRows<1> rows;
  rows.start();
  auto feed = [&](int t0) { return out[r0 * w + min(t0 + 1 + (l & 15), maxlen)] - r0; };
  int ahead = feed(0);
  for (int t0 = 0; t0 < steps; t0 += kBlk) {
    const int above = ahead;
    ahead = feed(t0 + kBlk);
    int32_t v[kBlk];
#pragma unroll
    for (int j = 0; j < kBlk; ++j) {
      const int u0 = edr::shift_in<64>(__builtin_amdgcn_readlane(above, j), rows.e[0]);
      rows.step<false>(u0, make_float2(0.0f, 0.0f), 0.0f);
      v[j] = rows.e[0] + row;
    }
    const int c0 = t0 - l + 1;
    int32_t* dst = out + row * w + c0;
    if (mine && c0 >= 1 && c0 + kBlk - 1 <= maxlen) {
#pragma unroll
      for (int j = 0; j < kBlk; j += 4)
        *reinterpret_cast<FourInts*>(dst + j) = FourInts{{v[j], v[j + 1], v[j + 2], v[j + 3]}};
    } else if (mine) {
#pragma unroll
      for (int j = 0; j < kBlk; ++j)
        if (c0 + j >= 1 && c0 + j <= maxlen) dst[j] = v[j];
    }
  }
}

// Exact top-k merge of one query per workgroup (no reference counterpart: the
// reference keeps a k-entry priority queue per query on the host,
// Grid.cpp:1600-1729).  A candidate's distance is its DP distance when it
// survived the filter, else the all-mismatch value of its length pair.  (The
// reference's cell rule is not a minimum, so a DP distance can exceed that
// value: survivors are never assumed to lie below it.)  The distances are
// histogrammed per trajectory length (at most GAT_MAX_TRAJ_LEN lengths,
// whatever the database size), each survivor moved from its length's value to
// its DP distance, and the cut T is the smallest distance whose running count
// reaches kk.  Every candidate below T is taken (fewer than kk: the
// non-survivors of the lengths whose value is below T, the survivors whose DP
// distance is), then the r smallest ids at distance T, found among the first ids
// where T is common, else among the first r + (number of survivors) ids of the
// lists of the lengths whose value is T (their survivors left out) and the
// survivors at T.  The kk results are ranked by (distance, id).
constexpr int kTopkMax = 1024;
constexpr int kLenBins = GAT_MAX_TRAJ_LEN + 1;     // lengths 0..GAT_MAX_TRAJ_LEN
constexpr int kDistBins = 2 * GAT_MAX_TRAJ_LEN + 1;  // distances 0..n + m
constexpr int kTopkBlock = 256;
constexpr int kScanAhead = 8;                               // ids per thread in flight
constexpr int kScanRound = kScanAhead * kTopkBlock;
constexpr int kScanRounds = 16;

// Index of c among the survivors s0 .. s1 - 1, or -1.
template <class Survivors>
__device__ __forceinline__ int32_t survivor_index(const Survivors& sv, int32_t s0, int32_t s1, int32_t c) {
  int32_t lo = s0, hi = s1;
  while (lo < hi) {
    const int32_t mid = lo + ((hi - lo) >> 1);
    if (sv.id(mid) < c) lo = mid + 1;
    else hi = mid;
  }
  return (lo < s1 && sv.id(lo) == c) ? lo : -1;
}

// Number of entries <= x in the ascending ids[0, n).
__device__ __forceinline__ int32_t count_le(const int32_t* __restrict__ ids, int32_t n, int32_t x) {
  int32_t lo = 0, hi = n;
  while (lo < hi) {
    const int32_t mid = lo + ((hi - lo) >> 1);
    if (ids[mid] <= x) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Sum over the workgroup, returned to every thread.
__device__ __forceinline__ int32_t topk_block_sum(int32_t v, int32_t* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();  // every thread has read red from the previous call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

// Survivors s0 .. s1 - 1 of a query, ascending by id: lists in global memory
// (edr_lists_kernel), or gathered into LDS by edr_merge_kernel.
struct GlobalSurvivors {
  const int32_t* __restrict__ sid;
  const int32_t* __restrict__ sdist;
  static constexpr bool kInLds = false;
  __device__ int32_t id(int32_t i) const { return sid[i]; }
  __device__ int32_t dist(int32_t i) const { return sdist[i]; }
};
struct LdsSurvivors {
  const unsigned long long* v;  // id << 32 | distance
  static constexpr bool kInLds = true;
  __device__ int32_t id(int32_t i) const { return int32_t(v[i] >> 32); }
  __device__ int32_t dist(int32_t i) const { return int32_t(uint32_t(v[i])); }
};

// kByLength: ftable rows are indexed by the two lengths in either order
// (gat_edr_length_table), so a query's values are one contiguous row.
template <bool kByLength, class Survivors>
__device__ __forceinline__ void topk_query(int q, const Survivors& sv, int32_t s0, int32_t s1,
                                           const int32_t* __restrict__ ftable, int32_t w,
                                           const int32_t* __restrict__ qlen, const int32_t* __restrict__ clen,
                                           int32_t nc, const int32_t* __restrict__ len_ids,
                                           const int32_t* __restrict__ len_off, int32_t k, int32_t kk,
                                           int32_t* __restrict__ out_ids, int32_t* __restrict__ out_dist,
                                           int32_t* __restrict__ status) {
  // The query's all-mismatch value per candidate length (16 bits: four
  // workgroups of the merge fit a CU); kNoValue for one outside 0..kDistBins - 1.
  constexpr uint16_t kNoValue = 0xFFFF;
  static_assert(kDistBins < kNoValue, "distances fit 16 bits");
  __shared__ uint16_t val[kLenBins];
  __shared__ int32_t hist[kDistBins];  // candidates per distance
  __shared__ int32_t out_d[kTopkMax], out_i[kTopkMax];
  __shared__ int32_t red[kTopkBlock / 64];
  __shared__ int32_t n_out, sh_T, sh_below, sh_at, sh_nt, sh_ng;
  __shared__ int32_t part_at[kScanAhead][kTopkBlock / 64];
  const int tid = threadIdx.x;
  const int a = qlen[q];
  if (a < 1 || a > GAT_MAX_TRAJ_LEN) {
    if (tid == 0) atomicOr(status, 4);
    return;
  }
#pragma unroll 9
  for (int L = tid; L < kLenBins; L += kTopkBlock) {
    const int32_t v = kByLength ? ftable[int64_t(a) * w + L] : ftable[int64_t(min(a, L)) * w + max(a, L)];
    val[L] = L < 1 ? 0 : v < 0 || v >= kDistBins ? kNoValue : uint16_t(v);
  }
  for (int b = tid; b < kDistBins; b += kTopkBlock) hist[b] = 0;
  if (tid == 0) {
    n_out = 0;
    sh_T = -1;
    sh_below = 0;
  }
  __syncthreads();
#pragma unroll 8
  for (int L = 1 + tid; L < kLenBins; L += kTopkBlock) {
    const int32_t cnt = len_off[L + 1] - len_off[L];
    const int32_t v = val[L];
    if (cnt > 0) {
      if (v >= kDistBins) atomicOr(status, 1);
      else atomicAdd(&hist[v], cnt);
    }
  }
  for (int32_t i = s0 + tid; i < s1; i += kTopkBlock) {
    const int32_t c = sv.id(i);
    const int32_t L = (c >= 0 && c < nc) ? clen[c] : 0;
    const int32_t d = sv.dist(i);
    if (L < 1 || L > GAT_MAX_TRAJ_LEN || d < 0 || d >= kDistBins || val[L] >= kDistBins) {
      atomicOr(status, 1);
      continue;
    }
    atomicSub(&hist[val[L]], 1);
    atomicAdd(&hist[d], 1);
  }
  __syncthreads();
  // The cut: thread t scans distances [kPer t, kPer (t + 1)).
  constexpr int kPer = (kDistBins + kTopkBlock - 1) / kTopkBlock;
  const int lane = tid & 63, wv = tid >> 6;
  int32_t local = 0;
  for (int j = 0; j < kPer; ++j) {
    const int b = tid * kPer + j;
    if (b < kDistBins) local += hist[b];
  }
  int32_t incl = local;
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t y = __shfl_up(incl, o);
    if (lane >= o) incl += y;
  }
  if (lane == 63) red[wv] = incl;
  __syncthreads();
  int32_t before = incl - local;
  for (int j = 0; j < wv; ++j) before += red[j];
  if (before < kk && before + local >= kk) {
    int32_t acc = before;
    for (int j = 0; j < kPer; ++j) {
      const int b = tid * kPer + j;
      if (b >= kDistBins) break;
      if (acc + hist[b] >= kk) {
        sh_T = b;
        sh_below = acc;
        sh_at = hist[b];
        break;
      }
      acc += hist[b];
    }
  }
  __syncthreads();
  const int32_t T = sh_T;
  const int32_t r = kk - sh_below;
  if (T < 0) {
    if (tid == 0) atomicOr(status, 2);
    return;
  }
  // The distance histogram is done with; its space now holds the lists of the
  // lengths valued T or less (their lengths, and where their entries start in
  // the order below), the gathered ids, and this query's survivor ids where
  // those lie in global memory.
  const int32_t ns = s1 - s0;
  const int32_t pre = r + ns;
  constexpr int32_t kLists = 1024, kGather = Survivors::kInLds ? kDistBins - 2 * kLists : 1024;
  constexpr int32_t kStage = Survivors::kInLds ? 0 : kDistBins - 2 * kLists - kGather;
  constexpr int32_t kEntriesMax = 64 * kTopkBlock;
  int32_t* tl = hist;
  int32_t* first = hist + kLists;
  int32_t* g = hist + 2 * kLists;
  int32_t* st = g + kGather;
  const bool staged = ns <= kStage;
  if (tid == 0) sh_nt = 0;
  __syncthreads();
  if (staged)
    for (int32_t i = tid; i < ns; i += kTopkBlock) st[i] = sv.id(s0 + i);
  __syncthreads();
  // The survivor list's index of c, or -1.
  auto survivor = [&](int32_t c) -> int32_t {
    if (ns == 0) return -1;
    if (!staged) return survivor_index(sv, s0, s1, c);
    int32_t lo = 0, hi = ns;
    while (lo < hi) {
      const int32_t mid = lo + ((hi - lo) >> 1);
      if (st[mid] < c) lo = mid + 1;
      else hi = mid;
    }
    return lo < ns && st[lo] == c ? s0 + lo : -1;
  };
  auto take = [&](int32_t d, int32_t c) {
    const int32_t pos = atomicAdd(&n_out, 1);
    if (pos < kTopkMax) {
      out_d[pos] = d;
      out_i[pos] = c;
    }
  };
  // The r smallest ids at T.  Where T is common they lie among the first ids:
  // about r * nc / (candidates at T) of them, read in order, 2,048 at a time,
  // until r are found.  (Of 200,000 candidates a median of 20,000 lie at T: 500
  // ids for 50 results, where the lists of T's lengths hold 3,300 entries to
  // look through.)  Ids ordered by length can hide them further back; then the
  // lists below take over.
  bool scanned = false;
  if (int64_t(r) * nc <= int64_t(kScanRound) * (kScanRounds / 4) * sh_at) {
    int32_t have = 0;
    const int32_t kept = n_out;
    for (int32_t base = 0, round = 0; base < nc && have < r && round < kScanRounds; base += kScanRound, ++round) {
      int32_t len[kScanAhead];
#pragma unroll
      for (int j = 0; j < kScanAhead; ++j) {
        const int64_t c = int64_t(base) + j * kTopkBlock + tid;
        len[j] = c < nc ? clen[c] : 0;
      }
      uint64_t at[kScanAhead];
#pragma unroll
      for (int j = 0; j < kScanAhead; ++j) {
        bool is = false;
        if (len[j] >= 1 && len[j] <= GAT_MAX_TRAJ_LEN) {
          const int32_t i = survivor(base + j * kTopkBlock + tid);
          is = (i >= 0 ? sv.dist(i) : int32_t(val[len[j]])) == T;
        }
        at[j] = __ballot(is);
        if (lane == 0) part_at[j][wv] = __popcll(at[j]);
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < kScanAhead; ++j)
#pragma unroll
        for (int x = 0; x < kTopkBlock / 64; ++x) {
          if (x == wv && (at[j] >> lane & 1u)) {
            const int32_t before = have + int32_t(__builtin_amdgcn_mbcnt_hi(
                                              uint32_t(at[j] >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(at[j]), 0u)));
            if (before < r) take(T, base + j * kTopkBlock + tid);
          }
          have += part_at[j][x];
        }
      __syncthreads();  // part_at is read
    }
    scanned = have >= r;
    if (!scanned) {
      if (tid == 0) n_out = kept;
      __syncthreads();
    }
  }
#pragma unroll 8
  for (int L = 1 + tid; L < kLenBins; L += kTopkBlock)
    if (val[L] <= (scanned ? T - 1 : T) && len_off[L + 1] > len_off[L]) {
      const int32_t at = atomicAdd(&sh_nt, 1);
      if (at < kLists) tl[at] = L;
    }
  __syncthreads();
  const int32_t nt = sh_nt;
  auto is_survivor = [&](int32_t c) -> bool { return survivor(c) >= 0; };
  // Survivors below T.
  for (int32_t i = s0 + tid; i < s1; i += kTopkBlock) {
    const int32_t c = sv.id(i);
    const int32_t L = (c >= 0 && c < nc) ? clen[c] : 0;
    if (L < 1 || L > GAT_MAX_TRAJ_LEN) continue;
    if (sv.dist(i) < T) take(sv.dist(i), c);
  }
  // The r smallest ids at T by lists: the least id X with r candidates at T at
  // or below it.  Each length valued T holds its ids ascending and at most ns of them
  // are survivors (counted at their DP distance), so a list of at least r + ns
  // ids has r non-survivors at or below its (r + ns)-th id: the least such id
  // over those lists bounds X from above, and below that bound every list's
  // count of ids <= X lies in its first r + ns ids.
  int32_t bound = nc > 0 ? nc - 1 : 0;
  auto bound_by = [&](int L) {
    const int32_t o = len_off[L];
    if (val[L] == T && len_off[L + 1] - o >= pre) bound = min(bound, len_ids[o + pre - 1]);
  };
  if (scanned) {
    bound = 0;
  } else if (nt <= kLists) {
    for (int32_t t = tid; t < nt; t += kTopkBlock) bound_by(tl[t]);
  } else {
    for (int L = 1 + tid; L < kLenBins; L += kTopkBlock) bound_by(L);
  }
  for (int o = 32; o > 0; o >>= 1) bound = min(bound, __shfl_xor(bound, o));
  if ((tid & 63) == 0) red[tid >> 6] = bound;
  __syncthreads();
  bound = min(min(red[0], red[1]), min(red[2], red[3]));
  __syncthreads();  // every thread has read red before it is written again
  // The entries that matter, each list's in full below T and the first r + ns
  // at T, one per thread: a list per thread read its ids one after another, a
  // microsecond each, and so did every step of a search over them.  The
  // non-survivors below T go out, those at
  // T and up to the bound are gathered, and X is searched among the gathered.
  int32_t entries = kEntriesMax + 1;
  if (nt <= kLists) {
    constexpr int kPerList = kLists / kTopkBlock;
    int32_t cnt[kPerList], sum = 0;
#pragma unroll
    for (int j = 0; j < kPerList; ++j) {
      const int32_t t = tid * kPerList + j;
      cnt[j] = 0;
      if (t < nt) {
        const int L = tl[t];
        const int32_t size = len_off[L + 1] - len_off[L];
        // (Saturated: more than kEntriesMax takes the other way.)
        cnt[j] = min(val[L] < T ? size : min(size, pre), kEntriesMax + 1);
      }
      sum += cnt[j];
    }
    int32_t upto = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const int32_t y = __shfl_up(upto, o);
      if (lane >= o) upto += y;
    }
    if (lane == 63) red[wv] = upto;
    __syncthreads();
    int32_t at = upto - sum;
    for (int j = 0; j < wv; ++j) at += red[j];
    entries = red[0] + red[1] + red[2] + red[3];
#pragma unroll
    for (int j = 0; j < kPerList; ++j) {
      const int32_t t = tid * kPerList + j;
      if (t < nt) first[t] = at;
      at += cnt[j];
    }
  }
  if (tid == 0) sh_ng = 0;
  __syncthreads();  // first, sh_ng, and red read
  if (entries <= kEntriesMax) {
    for (int32_t e = tid; e < entries; e += kTopkBlock) {
      int32_t lo = 0, hi = nt - 1;  // the last list starting at or before e
      while (lo < hi) {
        const int32_t mid = (lo + hi + 1) >> 1;
        if (first[mid] <= e) lo = mid;
        else hi = mid - 1;
      }
      const int L = tl[lo];
      const int32_t c = len_ids[len_off[L] + (e - first[lo])];
      const bool below = val[L] < T;
      if ((!below && c > bound) || is_survivor(c)) continue;
      if (below) {
        take(val[L], c);
      } else {
        const int32_t pos = atomicAdd(&sh_ng, 1);
        if (pos < kGather) g[pos] = c;
      }
    }
    for (int32_t i = s0 + tid; i < s1 && !scanned; i += kTopkBlock) {
      const int32_t c = sv.id(i);
      if (sv.dist(i) != T || c > bound || c < 0 || c >= nc || clen[c] < 1 || clen[c] > GAT_MAX_TRAJ_LEN) continue;
      const int32_t pos = atomicAdd(&sh_ng, 1);
      if (pos < kGather) g[pos] = c;
    }
  } else {
    for (int L = 1 + tid; L < kLenBins; L += kTopkBlock) {
      if (val[L] >= T) continue;
      for (int32_t i = len_off[L], e = len_off[L + 1]; i < e; ++i)
        if (!is_survivor(len_ids[i])) take(val[L], len_ids[i]);
    }
  }
  __syncthreads();
  const int32_t ng = sh_ng;
  if (scanned) {
    // (The candidates at T are out already.)
  } else if (entries <= kEntriesMax && ng <= kGather) {
    int32_t lo = 0, hi = bound;
    while (lo < hi) {
      const int32_t mid = lo + ((hi - lo) >> 1);
      int32_t part = 0;
      for (int32_t i = tid; i < ng; i += kTopkBlock) part += g[i] <= mid ? 1 : 0;
      if (topk_block_sum(part, red) >= r) hi = mid;
      else lo = mid + 1;
    }
    for (int32_t i = tid; i < ng; i += kTopkBlock)
      if (g[i] <= lo) take(T, g[i]);
  } else {
    // More than fits: X by a binary search over ids with a search per list.
    auto list_le = [&](int L, int32_t X) -> int32_t {
      const int32_t size = len_off[L + 1] - len_off[L];
      return count_le(len_ids + len_off[L], size < pre ? size : pre, X);
    };
    auto ties_le = [&](int32_t X) -> int32_t {
      int32_t part = 0;
      for (int L = 1 + tid; L < kLenBins; L += kTopkBlock)
        if (val[L] == T) part += list_le(L, X);
      for (int32_t i = s0 + tid; i < s1; i += kTopkBlock) {
        const int32_t c = sv.id(i);
        if (c > X || c < 0 || c >= nc) continue;
        const int32_t L = clen[c];
        if (L < 1 || L > GAT_MAX_TRAJ_LEN) continue;
        part += (sv.dist(i) == T ? 1 : 0) - (val[L] == T ? 1 : 0);
      }
      return topk_block_sum(part, red);
    };
    int32_t lo = 0, hi = bound;
    while (lo < hi) {
      const int32_t mid = lo + ((hi - lo) >> 1);
      if (ties_le(mid) >= r) hi = mid;
      else lo = mid + 1;
    }
    const int32_t X = lo;
    for (int L = 1 + tid; L < kLenBins; L += kTopkBlock) {
      if (val[L] != T) continue;
      const int32_t* ids = len_ids + len_off[L];
      const int32_t u = list_le(L, X);
      for (int32_t i = 0; i < u; ++i)
        if (!is_survivor(ids[i])) take(T, ids[i]);
    }
    for (int32_t i = s0 + tid; i < s1; i += kTopkBlock) {
      const int32_t c = sv.id(i);
      if (c > X || c < 0 || c >= nc) continue;
      const int32_t L = clen[c];
      if (L < 1 || L > GAT_MAX_TRAJ_LEN) continue;
      if (sv.dist(i) == T) take(T, c);
    }
  }
  __syncthreads();
  const int32_t n = n_out;
  if (n != kk) {
    if (tid == 0) atomicOr(status, 2);
    return;
  }
  // In rank order through LDS: the results may be host memory, which takes
  // whole lines, not one word at a time.
  int32_t* rd = hist;
  int32_t* ri = hist + kTopkMax;
  for (int i = tid; i < n; i += kTopkBlock) {
    const int32_t d = out_d[i], c = out_i[i];
    int32_t rank = 0;
    for (int j = 0; j < n; ++j) rank += (out_d[j] < d || (out_d[j] == d && out_i[j] < c)) ? 1 : 0;
    rd[rank] = d;
    ri[rank] = c + 1;
  }
  __syncthreads();
  for (int i = tid; i < n; i += kTopkBlock) {
    out_dist[int64_t(q) * k + i] = rd[i];
    out_ids[int64_t(q) * k + i] = ri[i];
  }
}

__global__ __launch_bounds__(kTopkBlock) void edr_topk_kernel(
    const int32_t* __restrict__ ftable, int32_t w, const int32_t* __restrict__ qlen,
    const int32_t* __restrict__ clen, int32_t nc, const int32_t* __restrict__ len_ids,
    const int32_t* __restrict__ len_off, const int32_t* __restrict__ sstart, const int32_t* __restrict__ sid,
    const int32_t* __restrict__ sdist, int32_t k, int32_t kk, int32_t* __restrict__ out_ids,
    int32_t* __restrict__ out_dist, int32_t* __restrict__ status) {
  const int q = blockIdx.x;
  topk_query<false>(q, GlobalSurvivors{sid, sdist}, sstart[q], sstart[q + 1], ftable, w, qlen, clen, nc, len_ids,
                    len_off, k, kk, out_ids, out_dist, status);
}

// A batch's control words (gat_edr_merge): device memory, cleared at its start.
constexpr int kCtlCount = 0, kCtlLists = 2, kCtlStatus = 3, kCtlTicket = 7, kCtlWords = 32;
constexpr int kMergeMax = 1024;  // survivors of a query gathered in LDS

// The merge straight from the DP's pairs and distances, one workgroup per query
// (no reference counterpart): the query's survivors are picked out of all the
// batch's pairs, sorted by id in LDS and merged as edr_topk_kernel does, where
// separate launches built lists, sorted them and merged.  Reading every pair
// in every workgroup suits batches of few pairs.  The results may go to pinned
// host memory; the last workgroup to end writes the control words and the time
// after them.  The start's time goes elsewhere (stamp): the last workgroup, on
// another XCD as a rule, is ordered behind the atomics whose results its ticket
// depends on, not behind the first one's plain stores.
__global__ __launch_bounds__(kTopkBlock) void edr_merge_kernel(
    const int32_t* __restrict__ ftable, int32_t w, const int32_t* __restrict__ qlen, int32_t nq,
    const int32_t* __restrict__ clen, int32_t nc, const int32_t* __restrict__ len_ids,
    const int32_t* __restrict__ len_off, const int2* __restrict__ pairs, const int32_t* __restrict__ dist,
    uint32_t cap, int32_t k, int32_t kk, int32_t* __restrict__ out_ids, int32_t* __restrict__ out_dist,
    uint32_t* __restrict__ ctl, uint32_t* __restrict__ ctl_out, uint32_t* __restrict__ stamp) {
  __shared__ unsigned long long v[kMergeMax];
  __shared__ int32_t found, wrong;
  const int q = blockIdx.x, t = threadIdx.x;
  if (stamp && q == 0 && t == 0) store_clock(stamp);
  const unsigned long long total = *reinterpret_cast<const unsigned long long*>(ctl + kCtlCount);
  const uint32_t np = total > cap ? 0u : uint32_t(total);
  if (t == 0) found = wrong = 0;
  __syncthreads();
  constexpr uint32_t kAhead = 8;  // pairs per thread in flight
  for (uint32_t i = t; i < np; i += kTopkBlock * kAhead) {
    int2 p[kAhead];
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j) p[j] = pairs[min(i + j * kTopkBlock, np - 1)];
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j) {
      const uint32_t k0 = i + j * kTopkBlock;
      if (k0 >= np || p[j].x != q) continue;
      const int32_t at = atomicAdd(&found, 1);
      if (at < kMergeMax) v[at] = ((unsigned long long)(uint32_t(p[j].y)) << 32) | uint32_t(dist[k0]);
    }
  }
  __syncthreads();
  const int32_t m = found;
  if (total <= cap && m <= kMergeMax) {
    if (m > 1) {  // bitonic sort by id (distinct within a query)
      int P = 2;
      while (P < m) P <<= 1;
      for (int i = m + t; i < P; i += kTopkBlock) v[i] = ~0ull;
      __syncthreads();
      for (int a = 2; a <= P; a <<= 1)
        for (int b = a >> 1; b > 0; b >>= 1) {
          for (int i = t; i < P; i += kTopkBlock) {
            const int o = i ^ b;
            if (o > i) {
              const bool up = (i & a) == 0;
              const unsigned long long x = v[i], y = v[o];
              if ((x > y) == up) {
                v[i] = y;
                v[o] = x;
              }
            }
          }
          __syncthreads();
        }
    }
    topk_query<true>(q, LdsSurvivors{v}, 0, m, ftable, w, qlen, clen, nc, len_ids, len_off, k, kk, out_ids, out_dist,
                     &wrong);
  }
  __syncthreads();
  if (t >= 64) return;
  uint32_t ticket = 0;
  if (t == 0) {
    // The statuses are in before the ticket, which depends on what their
    // atomics return: a fence would write the whole L2 back, once per workgroup.
    uint32_t before = 0;
    if (m > kMergeMax) before |= atomicOr(ctl + kCtlLists, 2u);
    if (wrong) before |= atomicOr(ctl + kCtlStatus, uint32_t(wrong));
    ticket = atomicAdd(ctl + kCtlTicket, before == ~0u ? 2u : 1u);  // (never 2: statuses are small)
  }
  if (uint32_t(__builtin_amdgcn_readfirstlane(int(ticket))) == uint32_t(nq) - 1u) {
    if (t < kCtlWords) ctl_out[t] = atomicOr(ctl + t, 0u);
    if (t == 0) store_clock(ctl_out + kCtlWords);
  }
}

// out[a * w + L] = the all-mismatch value of lengths a and L in either order.
__global__ __launch_bounds__(256) void edr_length_table_kernel(const int32_t* __restrict__ table, int32_t w,
                                                               int32_t* __restrict__ out) {
  // 16 x 16 tiles on and above the diagonal, each written to both sides.
  __shared__ int32_t tile[16][17];
  const int x = threadIdx.x & 15, y = threadIdx.x >> 4;
  const int c0 = int(blockIdx.x) * 16, r0 = int(blockIdx.y) * 16;
  if (c0 < r0) return;
  const int r = r0 + y, c = c0 + x;
  int32_t v = 0;
  if (r < w && c < w) v = table[int64_t(min(r, c)) * w + max(r, c)];
  tile[y][x] = v;
  if (r < w && c < w) out[int64_t(r) * w + c] = v;
  __syncthreads();
  const int rr = c0 + y, cc = r0 + x;
  if (c0 != r0 && rr < w && cc < w) out[int64_t(rr) * w + cc] = tile[x][y];
}

// ---------------------------------------------------------------- device jobs
// The batch's job list built on the device from the filter's survivors, so a
// top-k batch runs filter -> jobs -> DP -> merge with no host round trip.  One
// workgroup: per pair the shorter and longer length and the length bucket
// (JobShape below), then a counting sort in LDS by (bucket, strips descending,
// longer length descending in sixteen steps of the bucket's length range) and
// jobs of up to four pairs of one strip count (one pair in the long buckets).
// Pairs of equal sort key keep no particular order: it only changes which pairs
// share a job.
constexpr int kJobThreads = 1024;
constexpr int64_t kJobsOneBlock = 131072;  // larger batches take the whole device
constexpr int kJobsScratchExtra = GAT_EDR_JOBS_SCRATCH_EXTRA;
constexpr int kStripsMax = GAT_MAX_TRAJ_LEN / 16 + 1;  // strips_of(n) is 0..128
constexpr int kJobGroups = 4 * kStripsMax;             // (bucket, strips)
constexpr int kLenSteps = 16;                          // longer length in 128-point steps
constexpr int kSortBins = kJobGroups * kLenSteps;
constexpr int kSortPer = (kSortBins + kJobThreads - 1) / kJobThreads;

// Exclusive scan of a[0..n) in LDS by the whole workgroup (n <= per *
// kJobThreads); returns the total.  red holds kJobThreads / 64 + 1 words.
template <int PER>
__device__ uint32_t block_exclusive_scan(uint32_t* a, int n, uint32_t* red) {
  const int t = threadIdx.x;
  uint32_t v[PER], sum = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = t * PER + k;
    v[k] = i < n ? a[i] : 0u;
    sum += v[k];
  }
  uint32_t incl = sum;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = uint32_t(__shfl_up(int(incl), d, 64));
    if ((t & 63) >= d) incl += y;
  }
  if ((t & 63) == 63) red[t / 64] = incl;
  __syncthreads();
  if (t == 0) {
    uint32_t run = 0;
    for (int w = 0; w < kJobThreads / 64; ++w) {
      const uint32_t x = red[w];
      red[w] = run;
      run += x;
    }
    red[kJobThreads / 64] = run;
  }
  __syncthreads();
  uint32_t base = red[t / 64] + incl - sum;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = t * PER + k;
    if (i < n) a[i] = base;
    base += v[k];
  }
  const uint32_t total = red[kJobThreads / 64];
  __syncthreads();
  return total;
}

// What a pair of n rows and m columns keeps its wave busy for, in VALU
// instructions per 16-step block: in a 16-lane segment, on one wave (64-lane
// strips of four rows per lane, the last of two or one) and over several
// (edr_pipe_kernel's schedule, with a lag of kLag blocks between strips and a
// barrier per block).  Grid::runBatched applies the same rules on the host.
__device__ __forceinline__ int64_t segment_cost(int n, int m) {
  const int rows = (n + 15) / 16, rest = rows & 3;
  return int64_t((m + 15 + 15) / 16) * (19 * (rows / 4) + (rest >= 2 ? 11 : 0) + ((rest & 1) ? 7 : 0));
}
__device__ __forceinline__ int64_t one_wave_cost(int n, int m) {
  const int rows = (n + 63) / 64, rest = rows & 3;
  return int64_t((m + 63 + 15) / 16) * (19 * (rows / 4) + (rest >= 2 ? 11 : 0) + ((rest & 1) ? 7 : 0));
}
__device__ __forceinline__ int64_t pipe_cost(int n, int m, int waves) {
  const int per = (n + 64 * waves - 1) / (64 * waves);
  const int k = per <= 1 ? 1 : per == 2 ? 2 : 4;
  const int64_t strips = (n + 64 * k - 1) / (64 * k), b = (m + 63 + 15) / 16;
  const int64_t P = b > int64_t(waves) * kLag ? b : int64_t(waves) * kLag;
  return (((strips - 1) / waves) * P + ((strips - 1) % waves) * kLag + b) * (k == 1 ? 9 : k == 2 ? 13 : 21);
}

struct JobRules {
  int32_t split, waves, every_long, cus;
};

// The bucket rules of a batch of np pairs.  A batch of 64 jobs per CU and more
// keeps every SIMD busy whatever its pairs: long means longer than max(split,
// 1024).  A smaller one (one round of waves) ends when its longest pair does:
// its `critical` length is the longest pair's schedule over several waves (or
// on one, when it may take no more), but not under half of what all pairs
// would take spread evenly in 16-lane segments (a wave that shares its SIMD
// waits out its steps' latency and issues about a quarter of the time: with
// twice the spread work the longest pairs ran 1,040 us on one wave, the whole
// DP 510 with half).  A pair then takes the cheapest form that ends in time: a
// 16-lane segment (a quarter of the instructions, up to four times the length,
// and four waves share a SIMD) up to half of critical and `split` columns, one
// wave up to all of it, several beyond.
struct JobShape {
  int mid;
  bool latency, multi;
  __device__ JobShape(const JobRules& r, uint32_t np) {
    latency = (int64_t(np) + 3) / 4 < int64_t(r.cus) * 16;
    mid = latency ? r.split : max(r.split, 1024);
    multi = latency && r.waves > 1;
  }
};

// A pair's share of critical: the longest schedule, and the spread work.
__device__ __forceinline__ int64_t critical_share(int n, int m, const JobRules& r, const JobShape& sh) {
  if (!sh.latency || n < 1) return 0;
  return sh.multi ? pipe_cost(n, m, r.waves) : one_wave_cost(n, m);
}
__device__ __forceinline__ int64_t critical_of(int64_t longest, int64_t work, const JobRules& r) {
  const int64_t spread = work / (4 * 4 * int64_t(r.cus)) / 2;  // four pairs a wave, four SIMDs a CU
  return longest > spread ? longest : spread;
}

// Sort key of a pair of shorter length n and longer m: (bucket, strips
// descending, longer length descending in sixteen steps of the bucket's
// range).
__device__ __forceinline__ uint32_t job_key(int n, int m, const JobRules& rules, const JobShape& sh,
                                            int64_t critical) {
  int bucket = m <= rules.split ? 0 : m <= sh.mid ? 1 : 2;
  if (sh.latency && n >= 1) {
    if (bucket == 0 && 2 * segment_cost(n, m) > critical) bucket = 2;
    if (bucket == 2 && sh.multi && (rules.every_long ? m > rules.split : one_wave_cost(n, m) > critical)) bucket = 3;
  }
  const int strips = (n + 15) / 16;
  const int top = bucket == 0 ? rules.split : bucket == 1 ? sh.mid : GAT_MAX_TRAJ_LEN;
  const int step = max(1, (top + kLenSteps - 1) / kLenSteps);
  const int len = m >= 1 ? min((m - 1) / step, kLenSteps - 1) : 0;
  return uint32_t((bucket * kStripsMax + (kStripsMax - 1 - strips)) * kLenSteps + (kLenSteps - 1 - len));
}

__global__ __launch_bounds__(kJobThreads) void edr_jobs_kernel(const int2* __restrict__ pairs,
                                                               const unsigned long long* __restrict__ count,
                                                               uint32_t cap, const int32_t* __restrict__ qlen,
                                                               int32_t nq, const int32_t* __restrict__ clen,
                                                               int32_t nc, JobRules rules, int2* __restrict__ sorted,
                                                               int32_t* __restrict__ origin,
                                                               int2* __restrict__ nm, Job* __restrict__ jobs,
                                                               int32_t* __restrict__ windows,
                                                               int32_t* __restrict__ status,
                                                               unsigned long long* __restrict__ cells,
                                                               uint32_t* __restrict__ stamp) {
  __shared__ uint32_t bins[kSortBins];
  __shared__ uint32_t gjobs[kJobGroups + 1];
  __shared__ uint32_t red[kJobThreads / 64 + 1];
  __shared__ unsigned long long red64[kJobThreads / 64];
  const int t = threadIdx.x;
  if (stamp && t == 0) store_clock(stamp);
  const unsigned long long total = *count;
  if (t == 0) *status = total > cap ? 1 : 0;
  if (total > cap) {  // uniform: nothing to run; the caller grows the buffers
    if (t < 8) windows[t] = 0;
    return;
  }
  const uint32_t np = uint32_t(total);
  // Lengths, the cell count and the several-wave threshold.
  const JobShape shape(rules, np);
  unsigned long long my_cells = 0;
  int64_t my_crit = 0, my_work = 0;
  for (uint32_t i = t; i < np; i += kJobThreads) {
    const int2 p = pairs[i];
    const bool ok = p.x >= 0 && p.x < nq && p.y >= 0 && p.y < nc;
    const int a = ok ? qlen[p.x] : 0, b = ok ? clen[p.y] : 0;
    const int n = min(a, b), m = max(a, b);
    nm[i] = make_int2(n, m);
    my_cells += (unsigned long long)(n) * (unsigned long long)(m);
    const int64_t c = critical_share(n, m, rules, shape);
    if (c > my_crit) my_crit = c;
    if (n >= 1) my_work += segment_cost(n, m);
  }
  for (int off = 32; off > 0; off >>= 1) {
    my_cells += __shfl_xor(my_cells, off);
    my_work += __shfl_xor(my_work, off);
    const int64_t o = __shfl_xor(my_crit, off);
    if (o > my_crit) my_crit = o;
  }
  __shared__ int64_t crit_w[kJobThreads / 64], work_w[kJobThreads / 64];
  if ((t & 63) == 0) {
    red64[t / 64] = my_cells;
    crit_w[t / 64] = my_crit;
    work_w[t / 64] = my_work;
  }
  for (int i = t; i < kSortBins; i += kJobThreads) bins[i] = 0;
  __syncthreads();
  int64_t longest = 0, work = 0;
  for (int w = 0; w < kJobThreads / 64; ++w) {
    longest = crit_w[w] > longest ? crit_w[w] : longest;
    work += work_w[w];
  }
  const int64_t critical = critical_of(longest, work, rules);
  if (t == 0) {
    unsigned long long c = 0;
    for (int w = 0; w < kJobThreads / 64; ++w) c += red64[w];
    *cells = c;
  }
  auto key_of = [&](int2 v) { return job_key(v.x, v.y, rules, shape, critical); };
  for (uint32_t i = t; i < np; i += kJobThreads) atomicAdd(&bins[key_of(nm[i])], 1u);
  __syncthreads();
  block_exclusive_scan<kSortPer>(bins, kSortBins, red);
  for (uint32_t i = t; i < np; i += kJobThreads) {
    const uint32_t pos = atomicAdd(&bins[key_of(nm[i])], 1u);
    sorted[pos] = pairs[i];
    if (origin) origin[pos] = int32_t(i);
  }
  __syncthreads();
  // bins[b] now ends bin b: group g spans [end of bin g*16 - 1, end of bin g*16 + 15).
  auto group_start = [&](int g) { return g == 0 ? 0u : bins[g * kLenSteps - 1]; };
  auto per_job = [](int g) { return g / kStripsMax >= 2 ? 1u : 4u; };
  for (int g = t; g < kJobGroups; g += kJobThreads) {
    const uint32_t len = bins[g * kLenSteps + kLenSteps - 1] - group_start(g);
    gjobs[g] = (len + per_job(g) - 1) / per_job(g);
  }
  __syncthreads();
  const uint32_t njobs = block_exclusive_scan<1>(gjobs, kJobGroups, red);
  if (t == 0) gjobs[kJobGroups] = njobs;
  __syncthreads();
  for (uint32_t j = t; j < njobs; j += kJobThreads) {
    int lo = 0, hi = kJobGroups - 1;  // the last group whose first job is at or below j
    while (lo < hi) {
      const int mid_g = (lo + hi + 1) / 2;
      if (gjobs[mid_g] <= j) lo = mid_g; else hi = mid_g - 1;
    }
    const uint32_t g = uint32_t(lo), k = j - gjobs[g], per = per_job(int(g));
    const uint32_t first = group_start(int(g)) + k * per;
    const uint32_t end = bins[g * kLenSteps + kLenSteps - 1];
    jobs[j] = Job{int32_t(first), int32_t(min(per, end - first))};
  }
  if (t < 4) {
    windows[2 * t] = int32_t(gjobs[t * kStripsMax]);
    windows[2 * t + 1] = int32_t(gjobs[(t + 1) * kStripsMax] - gjobs[t * kStripsMax]);
  }
}

// The same job list for large batches, over the whole device: lengths and
// the batch's cell count and several-wave threshold; global bin totals;
// their scan, the groups' job counts and the windows (one workgroup); the
// pairs to their bins (each workgroup counts its contiguous share in LDS,
// reserves its range of every bin with one atomic per bin, then places its
// pairs); the jobs.  Scratch after the capacity's (n, m): bin totals, bin
// cursors, group starts and group job offsets.
constexpr int kJobsBlock = 256;

__device__ __forceinline__ bool jobs_overflow(const unsigned long long* count, uint32_t cap, uint32_t* np) {
  const unsigned long long total = *count;
  *np = total > cap ? 0u : uint32_t(total);
  return total > cap;
}

__global__ __launch_bounds__(kJobsBlock) void edr_jobs_lengths_kernel(
    const int2* __restrict__ pairs, const unsigned long long* __restrict__ count, uint32_t cap,
    const int32_t* __restrict__ qlen, int32_t nq, const int32_t* __restrict__ clen, int32_t nc, JobRules rules,
    int2* __restrict__ nm, unsigned long long* __restrict__ cells, unsigned long long* __restrict__ crit,
    uint32_t* __restrict__ stamp) {
  if (stamp && blockIdx.x == 0 && threadIdx.x == 0) store_clock(stamp);
  uint32_t np;
  if (jobs_overflow(count, cap, &np)) return;
  const JobShape sh(rules, np);
  unsigned long long my_cells = 0, my_crit = 0, my_work = 0;
  for (uint32_t i = blockIdx.x * kJobsBlock + threadIdx.x; i < np; i += gridDim.x * kJobsBlock) {
    const int2 p = pairs[i];
    const bool ok = p.x >= 0 && p.x < nq && p.y >= 0 && p.y < nc;
    const int a = ok ? qlen[p.x] : 0, b = ok ? clen[p.y] : 0;
    const int n = min(a, b), m = max(a, b);
    nm[i] = make_int2(n, m);
    my_cells += (unsigned long long)(n) * (unsigned long long)(m);
    const unsigned long long c = (unsigned long long)critical_share(n, m, rules, sh);
    my_crit = c > my_crit ? c : my_crit;
    if (sh.latency && n >= 1) my_work += (unsigned long long)segment_cost(n, m);
  }
  for (int off = 32; off > 0; off >>= 1) {
    my_cells += __shfl_xor(my_cells, off);
    const unsigned long long o = __shfl_xor(my_crit, off);
    my_crit = o > my_crit ? o : my_crit;
    my_work += __shfl_xor(my_work, off);
  }
  if ((threadIdx.x & 63) == 0) {
    if (my_cells) atomicAdd(cells, my_cells);
    if (my_crit) atomicMax(crit, my_crit);
    if (my_work) atomicAdd(crit + 1, my_work);
  }
}

__device__ __forceinline__ void jobs_share(uint32_t np, uint32_t* lo, uint32_t* hi) {
  const uint32_t per = (np + gridDim.x - 1) / gridDim.x;
  *lo = min(np, blockIdx.x * per);
  *hi = min(np, *lo + per);
}

__global__ __launch_bounds__(kJobsBlock) void edr_jobs_hist_kernel(const unsigned long long* __restrict__ count,
                                                                   uint32_t cap, JobRules rules,
                                                                   const int2* __restrict__ nm,
                                                                   const unsigned long long* __restrict__ crit,
                                                                   uint32_t* __restrict__ gbins) {
  __shared__ uint32_t h[kSortBins];
  uint32_t np;
  if (jobs_overflow(count, cap, &np)) return;
  const JobShape sh(rules, np);
  const int64_t critical = critical_of(int64_t(crit[0]), int64_t(crit[1]), rules);
  for (int b = threadIdx.x; b < kSortBins; b += kJobsBlock) h[b] = 0;
  __syncthreads();
  uint32_t lo, hi;
  jobs_share(np, &lo, &hi);
  for (uint32_t i = lo + threadIdx.x; i < hi; i += kJobsBlock) {
    const int2 v = nm[i];
    atomicAdd(&h[job_key(v.x, v.y, rules, sh, critical)], 1u);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < kSortBins; b += kJobsBlock)
    if (h[b]) atomicAdd(gbins + b, h[b]);
}

__global__ __launch_bounds__(kJobThreads) void edr_jobs_scan_kernel(const unsigned long long* __restrict__ count,
                                                                   uint32_t cap, const uint32_t* __restrict__ gbins,
                                                                   uint32_t* __restrict__ gcur,
                                                                   uint32_t* __restrict__ gstart,
                                                                   uint32_t* __restrict__ gjobs_out,
                                                                   int32_t* __restrict__ windows,
                                                                   int32_t* __restrict__ status) {
  __shared__ uint32_t bins[kSortBins];
  __shared__ uint32_t gjobs[kJobGroups + 1];
  __shared__ uint32_t red[kJobThreads / 64 + 1];
  const int t = threadIdx.x;
  uint32_t np;
  if (jobs_overflow(count, cap, &np)) {
    if (t < 8) windows[t] = 0;
    if (t == 0) {
      atomicOr(status, 1);
      gjobs_out[kJobGroups] = 0;
    }
    return;
  }
  for (int b = t; b < kSortBins; b += kJobThreads) bins[b] = gbins[b];
  __syncthreads();
  block_exclusive_scan<kSortPer>(bins, kSortBins, red);
  for (int b = t; b < kSortBins; b += kJobThreads) gcur[b] = bins[b];
  auto per_job = [](int g) { return g / kStripsMax >= 2 ? 1u : 4u; };
  auto group_end = [&](int g) { return g + 1 < kJobGroups ? bins[(g + 1) * kLenSteps] : np; };
  for (int g = t; g < kJobGroups; g += kJobThreads) {
    const uint32_t first = bins[g * kLenSteps];
    gstart[g] = first;
    gjobs[g] = (group_end(g) - first + per_job(g) - 1) / per_job(g);
  }
  if (t == 0) gstart[kJobGroups] = np;
  __syncthreads();
  const uint32_t njobs = block_exclusive_scan<1>(gjobs, kJobGroups, red);
  for (int g = t; g < kJobGroups; g += kJobThreads) gjobs_out[g] = gjobs[g];
  if (t == 0) gjobs_out[kJobGroups] = njobs;
  if (t < 4) {
    const uint32_t a = gjobs[t * kStripsMax];
    const uint32_t b = t == 3 ? njobs : gjobs[(t + 1) * kStripsMax];
    windows[2 * t] = int32_t(a);
    windows[2 * t + 1] = int32_t(b - a);
  }
}

__global__ __launch_bounds__(kJobsBlock) void edr_jobs_scatter_kernel(
    const int2* __restrict__ pairs, const unsigned long long* __restrict__ count, uint32_t cap, JobRules rules,
    const int2* __restrict__ nm, const unsigned long long* __restrict__ crit, uint32_t* __restrict__ gcur,
    int2* __restrict__ sorted, int32_t* __restrict__ origin) {
  __shared__ uint32_t h[kSortBins];
  uint32_t np;
  if (jobs_overflow(count, cap, &np)) return;
  const JobShape sh(rules, np);
  const int64_t critical = critical_of(int64_t(crit[0]), int64_t(crit[1]), rules);
  for (int b = threadIdx.x; b < kSortBins; b += kJobsBlock) h[b] = 0;
  __syncthreads();
  uint32_t lo, hi;
  jobs_share(np, &lo, &hi);
  for (uint32_t i = lo + threadIdx.x; i < hi; i += kJobsBlock) {
    const int2 v = nm[i];
    atomicAdd(&h[job_key(v.x, v.y, rules, sh, critical)], 1u);
  }
  __syncthreads();
  // This workgroup's range of every bin it uses; h becomes its cursors.
  for (int b = threadIdx.x; b < kSortBins; b += kJobsBlock)
    if (h[b]) h[b] = atomicAdd(gcur + b, h[b]);
  __syncthreads();
  for (uint32_t i = lo + threadIdx.x; i < hi; i += kJobsBlock) {
    const int2 v = nm[i];
    const uint32_t pos = atomicAdd(&h[job_key(v.x, v.y, rules, sh, critical)], 1u);
    if (pos < np) {
      sorted[pos] = pairs[i];
      if (origin) origin[pos] = int32_t(i);
    }
  }
}

__global__ __launch_bounds__(kJobsBlock) void edr_jobs_write_kernel(const unsigned long long* __restrict__ count,
                                                                    uint32_t cap, const uint32_t* __restrict__ gstart,
                                                                    const uint32_t* __restrict__ gjobs_in,
                                                                    Job* __restrict__ jobs) {
  __shared__ uint32_t gs[kJobGroups + 1], gj[kJobGroups + 1];
  uint32_t np;
  if (jobs_overflow(count, cap, &np)) return;
  for (int g = threadIdx.x; g <= kJobGroups; g += kJobsBlock) {
    gs[g] = gstart[g];
    gj[g] = gjobs_in[g];
  }
  __syncthreads();
  const uint32_t njobs = gj[kJobGroups];
  for (uint32_t j = blockIdx.x * kJobsBlock + threadIdx.x; j < njobs; j += gridDim.x * kJobsBlock) {
    int lo = 0, hi = kJobGroups - 1;  // the last group whose first job is at or below j
    while (lo < hi) {
      const int mid_g = (lo + hi + 1) / 2;
      if (gj[mid_g] <= j) lo = mid_g; else hi = mid_g - 1;
    }
    const uint32_t per = lo / kStripsMax >= 2 ? 1u : 4u;
    const uint32_t first = gs[lo] + (j - gj[lo]) * per;
    jobs[j] = Job{int32_t(first), int32_t(min(per, gs[lo + 1] - first))};
  }
}

// Per-query survivor lists for edr_topk_kernel from the DP's sorted pairs and
// distances: counts in LDS, their scan as the start offsets, then each pair
// to its query's next slot (in no order; edr_lists_sort_kernel sorts by id).
constexpr int kListQueries = 8192;

__global__ __launch_bounds__(kJobThreads) void edr_lists_kernel(const int2* __restrict__ sorted,
                                                                const int32_t* __restrict__ dist,
                                                                const unsigned long long* __restrict__ count,
                                                                uint32_t cap, int32_t nq, int32_t* __restrict__ start,
                                                                int32_t* __restrict__ ids,
                                                                int32_t* __restrict__ dists) {
  __shared__ uint32_t cnt[kListQueries];
  __shared__ uint32_t red[kJobThreads / 64 + 1];
  const int t = threadIdx.x;
  const unsigned long long total = *count;
  const uint32_t np = total > cap ? 0u : uint32_t(total);
  for (int q = t; q < nq; q += kJobThreads) cnt[q] = 0;
  __syncthreads();
  for (uint32_t i = t; i < np; i += kJobThreads) {
    const int q = sorted[i].x;
    if (q >= 0 && q < nq) atomicAdd(&cnt[q], 1u);
  }
  __syncthreads();
  const uint32_t n = block_exclusive_scan<kListQueries / kJobThreads>(cnt, nq, red);
  for (int q = t; q < nq; q += kJobThreads) start[q] = int32_t(cnt[q]);
  if (t == 0) start[nq] = int32_t(n);
  __syncthreads();
  for (uint32_t i = t; i < np; i += kJobThreads) {
    const int2 p = sorted[i];
    if (p.x < 0 || p.x >= nq) continue;
    const uint32_t pos = atomicAdd(&cnt[p.x], 1u);
    ids[pos] = p.y;
    dists[pos] = dist[i];
  }
}

// Each query's survivors sorted by id (ids are distinct within a query): a
// bitonic sort in LDS of up to kSortMax (id, distance) pairs per workgroup;
// a query with more sets status bit 2 and keeps its list unsorted.
constexpr int kSortMax = 2048;
constexpr int kSortThreads = 256;

__global__ __launch_bounds__(kSortThreads) void edr_lists_sort_kernel(const int32_t* __restrict__ start,
                                                                      int32_t* __restrict__ ids,
                                                                      int32_t* __restrict__ dists,
                                                                      int32_t* __restrict__ status) {
  __shared__ unsigned long long v[kSortMax];
  const int q = blockIdx.x, t = threadIdx.x;
  const int s0 = start[q], m = start[q + 1] - s0;
  if (m <= 1) return;
  if (m > kSortMax) {
    if (t == 0) atomicOr(status, 2);
    return;
  }
  int P = 2;
  while (P < m) P <<= 1;
  for (int i = t; i < P; i += kSortThreads)
    v[i] = i < m ? ((unsigned long long)(uint32_t(ids[s0 + i])) << 32) | uint32_t(dists[s0 + i]) : ~0ull;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = t; i < P; i += kSortThreads) {
        const int o = i ^ j;
        if (o > i) {
          const bool up = (i & k) == 0;
          const unsigned long long x = v[i], y = v[o];
          if ((x > y) == up) {
            v[i] = y;
            v[o] = x;
          }
        }
      }
      __syncthreads();
    }
  for (int i = t; i < m; i += kSortThreads) {
    ids[s0 + i] = int32_t(v[i] >> 32);
    dists[s0 + i] = int32_t(uint32_t(v[i]));
  }
}

// Every (query, candidate) pair of nq x nc, pair i = (i / nc, i % nc).
__global__ __launch_bounds__(256) void edr_all_pairs_kernel(int32_t nq, int32_t nc, int2* __restrict__ pairs,
                                                            unsigned long long* __restrict__ count) {
  const uint64_t n = uint64_t(nq) * uint64_t(nc);
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += uint64_t(gridDim.x) * blockDim.x)
    pairs[i] = make_int2(int32_t(i / uint64_t(nc)), int32_t(i % uint64_t(nc)));
  if (blockIdx.x == 0 && threadIdx.x == 0) *count = n;
}

// out[origin[p]] = sorted_dist[p]: distances back in the pairs' first order.
__global__ __launch_bounds__(256) void edr_unsort_kernel(const int32_t* __restrict__ origin,
                                                         const int32_t* __restrict__ sorted_dist,
                                                         const unsigned long long* __restrict__ count, uint32_t cap,
                                                         int32_t* __restrict__ out) {
  const unsigned long long total = *count;
  const uint32_t n = total > cap ? 0u : uint32_t(total);
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const int32_t o = origin[p];
    if (o >= 0 && uint32_t(o) < n) out[o] = sorted_dist[p];
  }
}

}  // namespace

extern "C" int gat_edr_filter(const float* qbox, int32_t nq, const float* cbox, int32_t nc, double eps,
                              int32_t* pairs_out, int64_t capacity, uint64_t* count, void* stream) {
  GAT_REQUIRE(nq >= 0 && nc >= 0 && capacity >= 0 && nq <= 65535, "EDR filter: bad sizes");
  GAT_REQUIRE(count, "EDR filter: null count");
  hipStream_t s = gat::as_stream(stream);
  GAT_HIP_CHECK(hipMemsetAsync(count, 0, sizeof(uint64_t), s));
  if (nq == 0 || nc == 0) return GAT_OK;
  GAT_REQUIRE(qbox && cbox && (pairs_out || capacity == 0), "EDR filter: null pointer");
  GAT_REQUIRE(eps > 0, "EDR filter: eps must be positive");
  int64_t bx = (int64_t(nc) + 255) / 256;
  if (bx > 64) bx = 64;
  edr_filter_kernel<<<dim3(uint32_t(bx), uint32_t((nq + kFilterQ - 1) / kFilterQ)), dim3(256), 0, s>>>(
      reinterpret_cast<const float4*>(qbox), nq, reinterpret_cast<const float4*>(cbox), nc, gat_eps_threshold(eps),
      reinterpret_cast<int2*>(pairs_out), uint64_t(capacity), reinterpret_cast<unsigned long long*>(count));
  GAT_LAUNCH_CHECK("edr_filter_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_filter_grid_add(const float* qbox, int32_t nq, const float* cbox, int32_t nc,
                                       const gat_edr_cand_grid* grid, double eps, int32_t* pairs_out,
                                       int64_t capacity, uint64_t* count, uint32_t* stamp, void* stream) {
  GAT_REQUIRE(nq >= 0 && nc >= 0 && capacity >= 0, "EDR grid filter: bad sizes");
  GAT_REQUIRE(count && grid, "EDR grid filter: null count or grid");
  GAT_REQUIRE(grid->cells_per_side >= 1 && grid->cells_per_side <= 4096 && grid->nalways >= 0 &&
                  grid->cell_start_dev && (grid->nalways == 0 || grid->always_dev) && std::isfinite(grid->x0) &&
                  std::isfinite(grid->y0) && std::isfinite(grid->inv_x) && std::isfinite(grid->inv_y) &&
                  grid->inv_x >= 0.0f && grid->inv_y >= 0.0f,
              "EDR grid filter: bad grid");
  if (nq == 0 || nc == 0) return GAT_OK;
  GAT_REQUIRE(qbox && cbox && (pairs_out || capacity == 0), "EDR grid filter: null pointer");
  GAT_REQUIRE(eps > 0, "EDR grid filter: eps must be positive");
  const CandGrid gr{grid->cells_per_side,
                    grid->x0,
                    grid->y0,
                    grid->inv_x,
                    grid->inv_y,
                    grid->cell_start_dev,
                    grid->entry_id_dev,
                    reinterpret_cast<const float4*>(grid->entry_box_dev),
                    grid->always_dev,
                    grid->nalways};
  edr_filter_grid_kernel<<<dim3(uint32_t((nq + kGridFilterWaves - 1) / kGridFilterWaves)),
                           dim3(64 * kGridFilterWaves), 0, gat::as_stream(stream)>>>(
      reinterpret_cast<const float4*>(qbox), nq, reinterpret_cast<const float4*>(cbox), nc, gr,
      gat_eps_threshold(eps), reinterpret_cast<int2*>(pairs_out), uint64_t(capacity),
      reinterpret_cast<unsigned long long*>(count), stamp);
  GAT_LAUNCH_CHECK("edr_filter_grid_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_filter_grid(const float* qbox, int32_t nq, const float* cbox, int32_t nc,
                                   const gat_edr_cand_grid* grid, double eps, int32_t* pairs_out, int64_t capacity,
                                   uint64_t* count, void* stream) {
  GAT_REQUIRE(nq >= 0 && nc >= 0 && capacity >= 0, "EDR grid filter: bad sizes");
  GAT_REQUIRE(count && grid, "EDR grid filter: null count or grid");
  if (int rc = gat_fill_u32(reinterpret_cast<uint32_t*>(count), 0u, 2, stream)) return rc;
  return gat_edr_filter_grid_add(qbox, nq, cbox, nc, grid, eps, pairs_out, capacity, count, nullptr, stream);
}

extern "C" int gat_edr_topk(const int32_t* ftable, int32_t w, const int32_t* qlen, int32_t nq, const int32_t* clen,
                            int32_t nc, const int32_t* len_ids, const int32_t* len_off, const int32_t* surv_start,
                            const int32_t* surv_id, const int32_t* surv_dist, int32_t k, int32_t kk, int32_t* out_ids,
                            int32_t* out_dist, int32_t* status, void* stream) {
  GAT_REQUIRE(w == GAT_MAX_TRAJ_LEN + 1, "EDR top-k: the mismatch table must be %d wide", GAT_MAX_TRAJ_LEN + 1);
  GAT_REQUIRE(nq >= 0 && nc >= 0, "EDR top-k: bad sizes");
  GAT_REQUIRE(k >= 1 && k <= kTopkMax && kk >= 0 && kk <= k && kk <= nc,
              "EDR top-k: k outside 1..%d or kk outside 0..min(k, candidates)", kTopkMax);
  GAT_REQUIRE(status, "EDR top-k: null status");
  hipStream_t s = gat::as_stream(stream);
  GAT_HIP_CHECK(hipMemsetAsync(status, 0, sizeof(int32_t), s));
  if (nq == 0 || kk == 0) return GAT_OK;
  GAT_REQUIRE(ftable && qlen && clen && len_ids && len_off && surv_start && out_ids && out_dist,
              "EDR top-k: null pointer");
  edr_topk_kernel<<<dim3(uint32_t(nq)), dim3(kTopkBlock), 0, s>>>(ftable, w, qlen, clen, nc, len_ids, len_off,
                                                                  surv_start, surv_id, surv_dist, k, kk, out_ids,
                                                                  out_dist, status);
  GAT_LAUNCH_CHECK("edr_topk_kernel");
  return GAT_OK;
}

namespace {

// One wave per trajectory: its points, given as separate lon / lat arrays, go
// to the padded interleaved store at dst_off[t], and its box is reduced over
// the wave.  The store is NaN-filled first by the entry point.
__global__ __launch_bounds__(64) void edr_pack_kernel(const float* __restrict__ lon, const float* __restrict__ lat,
                                                      const int64_t* __restrict__ src_off,
                                                      const int64_t* __restrict__ dst_off, int32_t ntraj,
                                                      int64_t total, float2* __restrict__ xy,
                                                      float4* __restrict__ box) {
  for (int32_t t = int32_t(blockIdx.x); t < ntraj; t += int32_t(gridDim.x)) {
    const int64_t b = src_off[t], e = src_off[t + 1], d = dst_off[t];
    float xl = INFINITY, yl = INFINITY, xh = -INFINITY, yh = -INFINITY;
    for (int64_t i = b + int64_t(threadIdx.x); i < e; i += 64) {
      const float x = lon[i], y = lat[i];
      const int64_t at = d + (i - b);
      if (at >= 0 && at < total) xy[at] = make_float2(x, y);
      xl = fminf(xl, x);
      xh = fmaxf(xh, x);
      yl = fminf(yl, y);
      yh = fmaxf(yh, y);
    }
    for (int o = 32; o > 0; o >>= 1) {
      xl = fminf(xl, __shfl_xor(xl, o));
      xh = fmaxf(xh, __shfl_xor(xh, o));
      yl = fminf(yl, __shfl_xor(yl, o));
      yh = fmaxf(yh, __shfl_xor(yh, o));
    }
    if (threadIdx.x == 0) box[t] = make_float4(xl, yl, xh, yh);
  }
}

// A small batch's queries from pinned host memory in one launch: the metadata
// (source offsets, padded offsets as 64 and 32 bits, lengths) copied as it is,
// the padded store written whole (points, NaN elsewhere), the boxes, and a
// batch's control words cleared.  One wave per trajectory, which also writes
// the padding before it; the store's end is shared by all.  Two copies, a fill
// and the packing kernel took 25 us for one 128-point query.
__global__ __launch_bounds__(256) void edr_stage_queries_kernel(
    const uint32_t* __restrict__ meta, uint32_t meta_words, uint32_t* __restrict__ up, const int64_t* __restrict__ src,
    const int64_t* __restrict__ dst, int32_t ntraj, int64_t npoints, const float* __restrict__ lon,
    const float* __restrict__ lat, int64_t total, float2* __restrict__ xy, float4* __restrict__ box,
    uint32_t* __restrict__ ctl, uint32_t ctl_words, uint32_t* __restrict__ stamp) {
  const int64_t i0 = int64_t(blockIdx.x) * 256 + threadIdx.x, stride = int64_t(gridDim.x) * 256;
  for (int64_t i = i0; i < ctl_words; i += stride) ctl[i] = 0u;
  if (stamp && i0 == 0) store_clock(stamp);
  for (int64_t i = i0; i < meta_words; i += stride) up[i] = meta[i];
  const float2 nan2 = edr::nan_point();
  // Points end at: the last trajectory's end (the store's start when empty).
  const int64_t end = ntraj > 0 ? dst[ntraj - 1] + (npoints - src[ntraj - 1]) : 0;
  for (int64_t i = end + i0; i < total; i += stride) xy[i] = nan2;
  const int lane = threadIdx.x & 63;
  for (int64_t t = i0 / 64; t < ntraj; t += stride / 64) {
    const int64_t b = src[t], n = src[t + 1] - b, d = dst[t];
    for (int64_t i = d - kPad + lane; i < d; i += 64)
      if (i >= 0 && i < total) xy[i] = nan2;
    float4 bb = edr::empty_box();
    // Eight points per lane in flight: a read of host memory takes microseconds.
    constexpr int kAhead = 8;
    for (int64_t i = lane; i < n; i += 64 * kAhead) {
      float2 p[kAhead];
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int64_t at = b + min(i + 64 * k, n - 1);
        p[k] = make_float2(lon[at], lat[at]);
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int64_t at = i + 64 * k;
        if (at < n && d + at >= 0 && d + at < total) xy[d + at] = p[k];
        bb = edr::grow(bb, p[k]);  // (a repeated last point changes no box)
      }
    }
    bb = edr::segment_box<64>(bb);
    if (lane == 0) box[t] = bb;
  }
}

}  // namespace

extern "C" int gat_edr_stage_queries(const void* meta_pinned, int64_t meta_bytes, void* up, const int64_t* src_pinned,
                                     const int64_t* dst_pinned, int32_t ntraj, int64_t npoints,
                                     const float* lon_pinned, const float* lat_pinned, int64_t total, float* xy,
                                     float* box, uint32_t* ctl, int64_t ctl_words, uint32_t* stamp, void* stream) {
  GAT_REQUIRE(meta_bytes >= 0 && meta_bytes % 4 == 0 && meta_bytes / 4 <= int64_t(UINT32_MAX) && ntraj >= 0 &&
                  npoints >= 0 && total >= 0 && ctl_words >= 0 && ctl_words <= int64_t(UINT32_MAX),
              "EDR stage queries: bad sizes");
  GAT_REQUIRE((meta_bytes == 0 || (meta_pinned && up)) && (total == 0 || xy) && (ctl_words == 0 || ctl),
              "EDR stage queries: null pointer");
  GAT_REQUIRE(ntraj == 0 || (src_pinned && dst_pinned && box && (npoints == 0 || (lon_pinned && lat_pinned))),
              "EDR stage queries: null queries");
  int64_t blocks = (int64_t(ntraj) + 3) / 4;
  const int64_t fill = (total - npoints + 255) / 256;
  if (blocks < fill) blocks = fill;
  const int64_t most = int64_t(gat::cu_count()) * 8;
  blocks = blocks < 1 ? 1 : blocks > most ? most : blocks;
  edr_stage_queries_kernel<<<dim3(uint32_t(blocks)), dim3(256), 0, gat::as_stream(stream)>>>(
      static_cast<const uint32_t*>(meta_pinned), uint32_t(meta_bytes / 4), static_cast<uint32_t*>(up), src_pinned,
      dst_pinned, ntraj, npoints, lon_pinned, lat_pinned, total, reinterpret_cast<float2*>(xy),
      reinterpret_cast<float4*>(box), ctl, uint32_t(ctl_words), stamp);
  GAT_LAUNCH_CHECK("edr_stage_queries_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_length_table(const int32_t* table, int32_t w, int32_t* out, void* stream) {
  GAT_REQUIRE(w >= 0 && w <= GAT_MAX_TRAJ_LEN + 1, "EDR length table: width outside 0..%d", GAT_MAX_TRAJ_LEN + 1);
  if (w == 0) return GAT_OK;
  GAT_REQUIRE(table && out, "EDR length table: null pointer");
  const uint32_t tiles = uint32_t((w + 15) / 16);
  edr_length_table_kernel<<<dim3(tiles, tiles), dim3(256), 0, gat::as_stream(stream)>>>(table, w, out);
  GAT_LAUNCH_CHECK("edr_length_table_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_merge(const int32_t* length_table, int32_t w, const int32_t* qlen, int32_t nq,
                             const int32_t* clen, int32_t nc, const int32_t* len_ids, const int32_t* len_off,
                             const int32_t* pairs, const int32_t* dist, int64_t capacity, int32_t k, int32_t kk,
                             int32_t* out_ids, int32_t* out_dist, uint32_t* ctl, uint32_t* ctl_out, uint32_t* stamp,
                             void* stream) {
  GAT_REQUIRE(w == GAT_MAX_TRAJ_LEN + 1, "EDR merge: the length table must be %d wide", GAT_MAX_TRAJ_LEN + 1);
  GAT_REQUIRE(nq >= 1 && nc >= 0 && capacity >= 0 && capacity <= int64_t(INT32_MAX), "EDR merge: bad sizes");
  GAT_REQUIRE(k >= 1 && k <= kTopkMax && kk >= 0 && kk <= k && kk <= nc,
              "EDR merge: k outside 1..%d or kk outside 0..min(k, candidates)", kTopkMax);
  GAT_REQUIRE(length_table && qlen && clen && len_ids && len_off && pairs && dist && out_ids && out_dist && ctl &&
                  ctl_out,
              "EDR merge: null pointer");
  edr_merge_kernel<<<dim3(uint32_t(nq)), dim3(kTopkBlock), 0, gat::as_stream(stream)>>>(
      length_table, w, qlen, nq, clen, nc, len_ids, len_off, reinterpret_cast<const int2*>(pairs), dist,
      uint32_t(capacity), k, kk, out_ids, out_dist, ctl, ctl_out, stamp);
  GAT_LAUNCH_CHECK("edr_merge_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_pack_trajectories(const float* lon, const float* lat, const int64_t* src_off,
                                         const int64_t* dst_off, int32_t ntraj, int64_t total, float* xy, float* box,
                                         void* stream) {
  GAT_REQUIRE(ntraj >= 0 && total >= 0, "gat_edr_pack_trajectories: bad sizes");
  GAT_REQUIRE(total == 0 || xy, "gat_edr_pack_trajectories: null store");
  if (total > 0)
    if (int rc = gat_fill_u32(reinterpret_cast<uint32_t*>(xy), 0x7FC00000u, 2 * total, stream)) return rc;
  if (ntraj == 0) return GAT_OK;
  GAT_REQUIRE(lon && lat && src_off && dst_off && box, "gat_edr_pack_trajectories: null pointer");
  const int64_t cap = int64_t(gat::cu_count()) * 16;
  const uint32_t blocks = uint32_t(ntraj < cap ? ntraj : cap);
  edr_pack_kernel<<<dim3(blocks), dim3(64), 0, gat::as_stream(stream)>>>(
      lon, lat, src_off, dst_off, ntraj, total, reinterpret_cast<float2*>(xy), reinterpret_cast<float4*>(box));
  GAT_LAUNCH_CHECK("edr_pack_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_mismatch_table(int32_t maxlen, int32_t* out, void* stream) {
  GAT_REQUIRE(maxlen >= 0 && maxlen <= GAT_MAX_TRAJ_LEN, "mismatch table: maxlen outside 0..%d", GAT_MAX_TRAJ_LEN);
  GAT_REQUIRE(out, "mismatch table: null output");
  edr_mismatch_rows_kernel<<<dim3(1), dim3(64 * kTabWaves), 0, gat::as_stream(stream)>>>(maxlen, out);
  GAT_LAUNCH_CHECK("edr_mismatch_rows_kernel");
  if (maxlen > 0) {
    edr_mismatch_fill_kernel<<<dim3(uint32_t((maxlen + 63) / 64)), dim3(64), 0, gat::as_stream(stream)>>>(maxlen, out);
    GAT_LAUNCH_CHECK("edr_mismatch_fill_kernel");
  }
  return GAT_OK;
}

namespace {

// The launches of gat_edr_batched and gat_edr_pairs (jobs null, raw set); the
// job counter is cleared already.
int launch_edr(const int2* P, int64_t npairs, const Job* J, int64_t njobs, const int32_t* window, int32_t* counter,
               const float2* Q, const int64_t* qoff, const int32_t* qlen, int32_t nqueries, const float2* Cs,
               const int64_t* coff, const int32_t* clen, int32_t ncands, int32_t maxlen, float u, int32_t per_cu,
               int32_t lanes_per_pair, int32_t* out, const RawPairs& raw, hipStream_t s) {
  // LDS class: the smallest row buffer that holds maxlen columns (64-lane
  // pairs: 1024 or 2048).  Persistent grid: per_cu single-wave workgroups per
  // CU (default by class), capped by the work.
  const bool wide = lanes_per_pair >= 64;
  const int waves = lanes_per_pair / 64;  // > 1: one pair over several waves (edr_pipe_kernel)
  int cls = maxlen <= 256 ? 256 : maxlen <= 512 ? 512 : maxlen <= 1024 ? 1024 : GAT_MAX_TRAJ_LEN;
  if (wide && cls < 1024) cls = 1024;
  const int64_t pc = per_cu > 0 ? per_cu : waves > 1 ? 16 / waves : wide ? 16 : (cls <= 512 ? 20 : cls == 1024 ? 16 : 9);
  int64_t blocks = int64_t(gat::cu_count()) * pc;
  if (blocks > njobs) blocks = njobs;
  const dim3 grid{uint32_t(blocks)}, block{64};
  if (waves > 1) {
    const dim3 wblock{uint32_t(64 * waves)};
#define GAT_EDR_PIPE(M, W)                                                                                       \
  edr_pipe_kernel<M, W><<<grid, wblock, 0, s>>>(P, npairs, J, int32_t(njobs), window, counter, nqueries, ncands, Q, \
                                                qoff, qlen, Cs, coff, clen, u, out, raw)
    if (cls == 1024) {
      if (waves == 2) GAT_EDR_PIPE(1024, 2);
      else if (waves == 4) GAT_EDR_PIPE(1024, 4);
      else GAT_EDR_PIPE(1024, 8);
    } else {
      if (waves == 2) GAT_EDR_PIPE(GAT_MAX_TRAJ_LEN, 2);
      else if (waves == 4) GAT_EDR_PIPE(GAT_MAX_TRAJ_LEN, 4);
      else GAT_EDR_PIPE(GAT_MAX_TRAJ_LEN, 8);
    }
#undef GAT_EDR_PIPE
    GAT_LAUNCH_CHECK("edr_pipe_kernel");
    return GAT_OK;
  }
#define GAT_EDR_LAUNCH(M, SEG)                                                                                  \
  edr_wave_kernel<M, SEG><<<grid, block, 0, s>>>(P, npairs, J, int32_t(njobs), window, counter, nqueries, ncands, Q, \
                                                 qoff, qlen, Cs, coff, clen, u, out, raw)
  if (wide) {
    if (cls == 1024)
      GAT_EDR_LAUNCH(1024, 64);
    else
      GAT_EDR_LAUNCH(GAT_MAX_TRAJ_LEN, 64);
  } else {
    switch (cls) {
      case 256: GAT_EDR_LAUNCH(256, 16); break;
      case 512: GAT_EDR_LAUNCH(512, 16); break;
      case 1024: GAT_EDR_LAUNCH(1024, 16); break;
      default: GAT_EDR_LAUNCH(GAT_MAX_TRAJ_LEN, 16);
    }
  }
#undef GAT_EDR_LAUNCH
  GAT_LAUNCH_CHECK("edr_wave_kernel");
  return GAT_OK;
}

}  // namespace

static int run_bucket(const int32_t* pairs, int64_t npairs, const gat_edr_job* jobs, int64_t njobs,
                      const int32_t* window, int32_t* counter, bool clear, const float* qxy, const int64_t* qoff,
                      const int32_t* qlen, int32_t nqueries, const float* cxy, const int64_t* coff,
                      const int32_t* clen, int32_t ncands, int32_t maxlen, double eps, int32_t per_cu,
                      int32_t lanes_per_pair, uint32_t* stamp, int32_t* out, void* stream) {
  GAT_REQUIRE(npairs >= 0 && njobs >= 0 && njobs <= INT32_MAX && nqueries >= 0 && ncands >= 0,
              "EDR batched: bad sizes");
  GAT_REQUIRE(lanes_per_pair == 16 || lanes_per_pair == 64 || lanes_per_pair == 128 || lanes_per_pair == 256 ||
                  lanes_per_pair == 512,
              "EDR batched: lanes_per_pair must be 16, 64, 128, 256 or 512");
  if (njobs == 0) return GAT_OK;
  GAT_REQUIRE(pairs && jobs && counter && qxy && qoff && qlen && cxy && coff && clen && out,
              "EDR batched: null pointer");
  GAT_REQUIRE(maxlen >= 1 && maxlen <= GAT_MAX_TRAJ_LEN, "EDR batched: maxlen outside 1..%d", GAT_MAX_TRAJ_LEN);
  GAT_REQUIRE(eps > 0, "EDR batched: eps must be positive");
  GAT_REQUIRE(per_cu >= 0 && per_cu <= 64, "EDR batched: per_cu outside 0..64");
  // The job counter is cleared by a kernel, so the launch can be captured in a graph.
  if (clear)
    if (int rc = gat_fill_u32(reinterpret_cast<uint32_t*>(counter), 0u, 1, stream)) return rc;
  return launch_edr(reinterpret_cast<const int2*>(pairs), npairs, reinterpret_cast<const Job*>(jobs), njobs, window,
                    counter, reinterpret_cast<const float2*>(qxy), qoff, qlen, nqueries,
                    reinterpret_cast<const float2*>(cxy), coff, clen, ncands, maxlen, gat_eps_threshold(eps), per_cu,
                    lanes_per_pair, out, RawPairs{nullptr, nullptr, stamp}, gat::as_stream(stream));
}

extern "C" int gat_edr_bucket(const int32_t* pairs, int64_t npairs, const gat_edr_job* jobs, int64_t njobs,
                              const int32_t* window, int32_t* counter, const float* qxy, const int64_t* qoff,
                              const int32_t* qlen, int32_t nqueries, const float* cxy, const int64_t* coff,
                              const int32_t* clen, int32_t ncands, int32_t maxlen, double eps, int32_t per_cu,
                              int32_t lanes_per_pair, uint32_t* stamp, int32_t* out, void* stream) {
  return run_bucket(pairs, npairs, jobs, njobs, window, counter, false, qxy, qoff, qlen, nqueries, cxy, coff, clen,
                    ncands, maxlen, eps, per_cu, lanes_per_pair, stamp, out, stream);
}

extern "C" int gat_edr_batched(const int32_t* pairs, int64_t npairs, const gat_edr_job* jobs, int64_t njobs,
                               const int32_t* window, int32_t* counter, const float* qxy, const int64_t* qoff, const int32_t* qlen,
                               int32_t nqueries, const float* cxy, const int64_t* coff, const int32_t* clen,
                               int32_t ncands, int32_t maxlen, double eps, int32_t per_cu, int32_t lanes_per_pair,
                               int32_t* out, void* stream) {
  return run_bucket(pairs, npairs, jobs, njobs, window, counter, true, qxy, qoff, qlen, nqueries, cxy, coff, clen,
                    ncands, maxlen, eps, per_cu, lanes_per_pair, nullptr, out, stream);
}

extern "C" int gat_edr_pairs(const int32_t* pairs, const uint64_t* live, int64_t capacity, int32_t* counter,
                             const float* qxy, const int64_t* qoff, const int32_t* qlen, int32_t nqueries,
                             const float* cxy, const int64_t* coff, const int32_t* clen, int32_t ncands,
                             int32_t maxlen, double eps, int32_t lanes_per_pair, uint64_t* cells, uint32_t* stamp,
                             int32_t* out, void* stream) {
  GAT_REQUIRE(capacity >= 0 && capacity <= int64_t(INT32_MAX) - 8 && nqueries >= 0 && ncands >= 0,
              "EDR pairs: bad sizes");
  GAT_REQUIRE(lanes_per_pair == 64 || lanes_per_pair == 128 || lanes_per_pair == 256 || lanes_per_pair == 512,
              "EDR pairs: lanes_per_pair must be 64, 128, 256 or 512");
  if (capacity == 0) return GAT_OK;
  GAT_REQUIRE(pairs && live && counter && qxy && qoff && qlen && cxy && coff && clen && out && cells,
              "EDR pairs: null pointer");
  GAT_REQUIRE(maxlen >= 1 && maxlen <= GAT_MAX_TRAJ_LEN, "EDR pairs: maxlen outside 1..%d", GAT_MAX_TRAJ_LEN);
  GAT_REQUIRE(eps > 0, "EDR pairs: eps must be positive");
  return launch_edr(reinterpret_cast<const int2*>(pairs), capacity, nullptr, capacity, nullptr, counter,
                    reinterpret_cast<const float2*>(qxy), qoff, qlen, nqueries, reinterpret_cast<const float2*>(cxy),
                    coff, clen, ncands, maxlen, gat_eps_threshold(eps), 0, lanes_per_pair, out,
                    RawPairs{reinterpret_cast<const unsigned long long*>(live),
                             reinterpret_cast<unsigned long long*>(cells), stamp},
                    gat::as_stream(stream));
}

extern "C" int gat_edr_jobs_stamped(const int32_t* pairs, const uint64_t* count, int64_t capacity, const int32_t* qlen,
                                    int32_t nq, const int32_t* clen, int32_t nc, int32_t split, int32_t waves,
                                    int32_t every_long, int32_t* sorted, int32_t* origin, int32_t* scratch,
                                    gat_edr_job* jobs, int32_t* windows, int32_t* status, uint64_t* cells,
                                    uint32_t* stamp, void* stream) {
  GAT_REQUIRE(capacity >= 0 && capacity <= int64_t(INT32_MAX) - 8 && nq >= 0 && nc >= 0,
              "EDR jobs: bad sizes");
  GAT_REQUIRE(split >= 1 && split <= GAT_MAX_TRAJ_LEN && waves >= 1 && waves <= 8, "EDR jobs: bad rules");
  GAT_REQUIRE(pairs && count && qlen && clen && sorted && scratch && jobs && windows && status && cells,
              "EDR jobs: null pointer");
  const JobRules rules{split, waves, every_long ? 1 : 0, int32_t(gat::cu_count())};
  hipStream_t s = gat::as_stream(stream);
  const auto* P = reinterpret_cast<const int2*>(pairs);
  const auto* C = reinterpret_cast<const unsigned long long*>(count);
  auto* NM = reinterpret_cast<int2*>(scratch);
  auto* cells_u = reinterpret_cast<unsigned long long*>(cells);
  if (capacity <= kJobsOneBlock) {
    edr_jobs_kernel<<<dim3(1), dim3(kJobThreads), 0, s>>>(P, C, uint32_t(capacity), qlen, nq, clen, nc, rules,
                                                          reinterpret_cast<int2*>(sorted), origin, NM,
                                                          reinterpret_cast<Job*>(jobs), windows, status, cells_u,
                                                          stamp);
    GAT_LAUNCH_CHECK("edr_jobs_kernel");
    return GAT_OK;
  }
  // Scratch after the (n, m) pairs (8-byte aligned: 2 * capacity words): the
  // longest schedule and the spread work, bin totals, bin cursors, group starts, group job
  // offsets.
  static_assert(4 + 2 * kSortBins + 2 * (kJobGroups + 1) <= kJobsScratchExtra, "job scratch");
  auto* crit = reinterpret_cast<unsigned long long*>(scratch + 2 * capacity);
  uint32_t* gbins = reinterpret_cast<uint32_t*>(scratch + 2 * capacity + 4);
  uint32_t* gcur = gbins + kSortBins;
  uint32_t* gstart = gcur + kSortBins;
  uint32_t* gjobs = gstart + kJobGroups + 1;
  if (int rc = gat_fill_u32(reinterpret_cast<uint32_t*>(crit), 0u, 4 + kSortBins, stream)) return rc;
  if (int rc = gat_fill_u32(reinterpret_cast<uint32_t*>(status), 0u, 1, stream)) return rc;
  if (int rc = gat_fill_u32(reinterpret_cast<uint32_t*>(cells), 0u, 2, stream)) return rc;
  int64_t blocks = (capacity + 4095) / 4096;
  const int64_t most = int64_t(gat::cu_count()) * 4;
  if (blocks > most) blocks = most;
  if (blocks < 1) blocks = 1;
  const dim3 grid{uint32_t(blocks)}, block{kJobsBlock};
  const uint32_t cap = uint32_t(capacity);
  edr_jobs_lengths_kernel<<<grid, block, 0, s>>>(P, C, cap, qlen, nq, clen, nc, rules, NM, cells_u, crit, stamp);
  GAT_LAUNCH_CHECK("edr_jobs_lengths_kernel");
  edr_jobs_hist_kernel<<<grid, block, 0, s>>>(C, cap, rules, NM, crit, gbins);
  GAT_LAUNCH_CHECK("edr_jobs_hist_kernel");
  edr_jobs_scan_kernel<<<dim3(1), dim3(kJobThreads), 0, s>>>(C, cap, gbins, gcur, gstart, gjobs, windows, status);
  GAT_LAUNCH_CHECK("edr_jobs_scan_kernel");
  edr_jobs_scatter_kernel<<<grid, block, 0, s>>>(P, C, cap, rules, NM, crit, gcur, reinterpret_cast<int2*>(sorted),
                                                 origin);
  GAT_LAUNCH_CHECK("edr_jobs_scatter_kernel");
  edr_jobs_write_kernel<<<grid, block, 0, s>>>(C, cap, gstart, gjobs, reinterpret_cast<Job*>(jobs));
  GAT_LAUNCH_CHECK("edr_jobs_write_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_jobs(const int32_t* pairs, const uint64_t* count, int64_t capacity, const int32_t* qlen,
                            int32_t nq, const int32_t* clen, int32_t nc, int32_t split, int32_t waves,
                            int32_t every_long, int32_t* sorted, int32_t* origin, int32_t* scratch,
                            gat_edr_job* jobs, int32_t* windows, int32_t* status, uint64_t* cells, void* stream) {
  return gat_edr_jobs_stamped(pairs, count, capacity, qlen, nq, clen, nc, split, waves, every_long, sorted, origin,
                              scratch, jobs, windows, status, cells, nullptr, stream);
}

extern "C" int gat_edr_survivor_lists(const int32_t* sorted, const int32_t* dist, const uint64_t* count,
                                      int64_t capacity, int32_t nq, int32_t* start, int32_t* ids, int32_t* dists,
                                      int32_t* status, void* stream) {
  GAT_REQUIRE(capacity >= 0 && capacity <= int64_t(INT32_MAX) && nq >= 0 && nq <= kListQueries,
              "EDR survivor lists: at most %d queries", kListQueries);
  GAT_REQUIRE(sorted && dist && count && start && ids && dists && status, "EDR survivor lists: null pointer");
  if (nq == 0) return GAT_OK;
  hipStream_t s = gat::as_stream(stream);
  edr_lists_kernel<<<dim3(1), dim3(kJobThreads), 0, s>>>(reinterpret_cast<const int2*>(sorted), dist,
                                                          reinterpret_cast<const unsigned long long*>(count),
                                                          uint32_t(capacity), nq, start, ids, dists);
  GAT_LAUNCH_CHECK("edr_lists_kernel");
  edr_lists_sort_kernel<<<dim3(uint32_t(nq)), dim3(kSortThreads), 0, s>>>(start, ids, dists, status);
  GAT_LAUNCH_CHECK("edr_lists_sort_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_all_pairs(int32_t nq, int32_t nc, int32_t* pairs, uint64_t* count, void* stream) {
  GAT_REQUIRE(nq >= 0 && nc >= 0 && int64_t(nq) * nc <= int64_t(INT32_MAX), "EDR all pairs: bad sizes");
  GAT_REQUIRE(pairs && count, "EDR all pairs: null pointer");
  const int64_t n = int64_t(nq) * nc;
  int64_t blocks = (n + 255) / 256;
  const int64_t cap = int64_t(gat::cu_count()) * 16;
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  edr_all_pairs_kernel<<<dim3(uint32_t(blocks)), dim3(256), 0, gat::as_stream(stream)>>>(
      nq, nc, reinterpret_cast<int2*>(pairs), reinterpret_cast<unsigned long long*>(count));
  GAT_LAUNCH_CHECK("edr_all_pairs_kernel");
  return GAT_OK;
}

extern "C" int gat_edr_unsort(const int32_t* origin, const int32_t* sorted_dist, const uint64_t* count,
                              int64_t capacity, int32_t* out, void* stream) {
  GAT_REQUIRE(capacity >= 0 && capacity <= int64_t(INT32_MAX), "EDR unsort: bad capacity");
  GAT_REQUIRE(origin && sorted_dist && count && out, "EDR unsort: null pointer");
  int64_t blocks = (capacity + 255) / 256;
  const int64_t cap = int64_t(gat::cu_count()) * 16;
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  edr_unsort_kernel<<<dim3(uint32_t(blocks)), dim3(256), 0, gat::as_stream(stream)>>>(
      origin, sorted_dist, reinterpret_cast<const unsigned long long*>(count), uint32_t(capacity), out);
  GAT_LAUNCH_CHECK("edr_unsort_kernel");
  return GAT_OK;
}

