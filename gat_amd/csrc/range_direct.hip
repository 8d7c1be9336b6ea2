// The direct form of small range batches (a serving loop's, a caller's few
// rectangles), chained on the device with one host synchronisation: stage in,
// selection, output regions, refine, results out.  Such a batch is bound by its
// launches and by the latency of each step's dependent loads, not by bandwidth,
// so steps are merged (the upload is the kernel that clears the counters and
// reads the rectangles from pinned host memory; the readback is the kernel that
// writes the counts to it) and the refine reads the selection's (leaf,
// rectangle) entries itself.  One rectangle over 2.7M points took 138 us as
// nine launches, five copies and two synchronisations, and takes 66 us; 100
// rectangles of sides up to 0.05 over 1M trajectories took 525 us, and take 121.
#include "gat_common.hpp"

namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;

struct Node {
  float4 box;
  int32_t first_child;
  uint32_t start, count, flags;
};
static_assert(sizeof(Node) == sizeof(gat_tree_node), "node layout");

struct Store {
  const float2* xy;
  const uint32_t* id;
  const uint16_t* pid;
  uint64_t npoints;
  uint32_t pid_bits;
};

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
}
__device__ __forceinline__ uint32_t readlane_u(uint32_t v, uint32_t j) {
  return uint32_t(__builtin_amdgcn_readlane(int(v), int(j)));
}
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// MBB::pInBox (MBB.cpp:21-26): inclusive on all four edges; NaN is in no box.
__device__ __forceinline__ bool in_box(const float4& b, float x, float y) {
  return x <= b.z && x >= b.x && y <= b.w && y >= b.y;
}

__device__ __forceinline__ void store_u64(uint32_t* p, uint64_t v) {
  p[0] = uint32_t(v);
  p[1] = uint32_t(v >> 32);
}

constexpr int kSpans = 4;
struct Spans {
  uint32_t* p[kSpans];
  uint64_t end[kSpans];  // running totals of the spans' lengths
};

// Words of pinned host memory to the device, spans cleared, and the time.
__global__ __launch_bounds__(kBlock) void stage_in_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                          uint64_t words, Spans f, uint32_t* __restrict__ stamp) {
  const uint64_t i0 = uint64_t(blockIdx.x) * kBlock + threadIdx.x, stride = uint64_t(gridDim.x) * kBlock;
  if (stamp && i0 == 0) store_u64(stamp, wall_clock64());
  for (uint64_t i = i0; i < words; i += stride) dst[i] = src[i];
  for (uint64_t i = i0; i < f.end[kSpans - 1]; i += stride) {
    int k = 0;
    while (i >= f.end[k]) ++k;  // i < end[kSpans - 1], so k stays in range
    f.p[k][i - (k ? f.end[k - 1] : 0)] = 0u;
  }
}

// qbase = the exclusive sum of cand, qcount = 0, the total to counters[2..3]
// and the time to counters[14..15].  One workgroup: the batch is small.
__global__ __launch_bounds__(kBlock) void direct_regions_kernel(const uint64_t* __restrict__ cand, uint64_t nq,
                                                                uint64_t* __restrict__ qbase,
                                                                uint32_t* __restrict__ qcount,
                                                                uint32_t* __restrict__ counters) {
  __shared__ uint64_t wave_sum[kBlock / kWave];
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  uint64_t carry = 0;
  for (uint64_t b = 0; b < nq; b += kBlock) {
    const uint64_t i = b + t;
    const uint64_t v = i < nq ? cand[i] : 0;
    uint64_t incl = v;
    for (int d = 1; d < kWave; d <<= 1) {
      const uint64_t o = __shfl_up(incl, d);
      if (lane >= uint32_t(d)) incl += o;
    }
    __syncthreads();  // every thread has read the previous round's sums
    if (lane == kWave - 1) wave_sum[w] = incl;
    __syncthreads();
    uint64_t before = carry;
    for (uint32_t k = 0; k < kBlock / kWave; ++k) {
      if (k < w) before += wave_sum[k];
      carry += wave_sum[k];
    }
    if (i < nq) {
      qbase[i] = before + incl - v;
      qcount[i] = 0;
    }
  }
  if (t == 0) {
    store_u64(counters + 2, carry);
    store_u64(counters + 14, wall_clock64());
  }
}

// One wave refines four consecutive (leaf, rectangle) entries at a time, up to
// 256 points of each per round: their sixteen loads per lane are in flight
// together, and entries of the same rectangle (the selection lists a
// rectangle's leaves together) reserve their output slots with one atomic.
// With one entry and one atomic per wave, 100 rectangles over 1M trajectories
// took 70 us: the largest rectangle's 1,900 atomics on its counter one after
// another.
constexpr int kGroup = 4;
constexpr int kSlots = 4;  // 64-point slots per entry and round

template <bool kPacked>
__global__ __launch_bounds__(kBlock) void direct_refine_kernel(
    Store store, const uint2* __restrict__ lq, const unsigned long long* __restrict__ lq_total, uint64_t lq_cap,
    const Node* __restrict__ nodes, uint32_t nnodes, const float4* __restrict__ boxes, uint32_t nqueries,
    const uint64_t* __restrict__ qbase, uint32_t* __restrict__ qcount, int2* __restrict__ pairs, uint64_t capacity) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = uniform((blockIdx.x * kBlock + threadIdx.x) / kWave);
  const uint64_t nwaves = uint64_t(gridDim.x) * (kBlock / kWave);
  const uint64_t total = *lq_total;
  const uint64_t n = total < lq_cap ? total : lq_cap;
  const uint32_t pid_mask = (1u << store.pid_bits) - 1u;
  for (uint64_t g = wave; g * kGroup < n; g += nwaves) {
    // Lane e < 4: entry e.  Entries naming no leaf, no rectangle or points
    // past the store stay empty.
    uint32_t my_start = 0, my_count = 0, my_q = 0;
    if (lane < kGroup && g * kGroup + lane < n) {
      const uint2 e = lq[g * kGroup + lane];
      if (e.x < nnodes && e.y < nqueries) {
        my_start = nodes[e.x].start;
        my_count = nodes[e.x].count;
        my_q = e.y;
        if (uint64_t(my_start) + my_count > store.npoints) my_count = 0;
      }
    }
    uint32_t start[kGroup], count[kGroup], q[kGroup], most = 0;
    float4 box[kGroup];
#pragma unroll
    for (int e = 0; e < kGroup; ++e) {
      start[e] = readlane_u(my_start, e);
      count[e] = readlane_u(my_count, e);
      q[e] = readlane_u(my_q, e);
      most = most > count[e] ? most : count[e];
      box[e] = boxes[q[e]];
    }
    for (uint32_t base = 0; base < most; base += kSlots * kWave) {
      float2 v[kGroup][kSlots];
#pragma unroll
      for (int e = 0; e < kGroup; ++e)
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
          const uint32_t i = base + k * kWave + lane;
          v[e][k] = i < count[e] ? store.xy[uint64_t(start[e]) + i] : make_float2(__builtin_nanf(""), 0.0f);
        }
      // Bit kSlots * e + k: the lane's point of slot k of entry e is a hit (the
      // sixteen wave masks would crowd the SGPRs).
      uint32_t hit = 0, hits[kGroup];
#pragma unroll
      for (int e = 0; e < kGroup; ++e) {
        hits[e] = 0;
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
          const bool in = in_box(box[e], v[e][k].x, v[e][k].y);
          hit |= in ? 1u << (kSlots * e + k) : 0u;
          hits[e] += uint32_t(__popcll(__ballot(in)));
        }
      }
      if ((hits[0] | hits[1] | hits[2] | hits[3]) == 0) continue;
      uint32_t id[kGroup][kSlots], pid[kGroup][kSlots];
#pragma unroll
      for (int e = 0; e < kGroup; ++e)
#pragma unroll
        for (int k = 0; k < kSlots; ++k)
          if ((hit >> (kSlots * e + k)) & 1u) {
            const uint64_t at = uint64_t(start[e]) + base + k * kWave + lane;
            id[e][k] = store.id[at];
            if constexpr (!kPacked) pid[e][k] = store.pid[at];
          }
      // Entries next to each other of one rectangle form a run: its first
      // entry's lane reserves for all of it.
      uint32_t run_sum[kGroup], before[kGroup], lead[kGroup];
      run_sum[kGroup - 1] = hits[kGroup - 1];
#pragma unroll
      for (int e = kGroup - 2; e >= 0; --e) run_sum[e] = hits[e] + (q[e + 1] == q[e] ? run_sum[e + 1] : 0u);
      lead[0] = 0;
      before[0] = 0;
#pragma unroll
      for (int e = 1; e < kGroup; ++e) {
        const bool same = q[e] == q[e - 1];
        lead[e] = same ? lead[e - 1] : uint32_t(e);
        before[e] = same ? before[e - 1] + hits[e - 1] : 0u;
      }
      uint32_t add = 0, addq = 0;
#pragma unroll
      for (int e = 0; e < kGroup; ++e)
        if (lane == uint32_t(e) && lead[e] == uint32_t(e)) {
          add = run_sum[e];
          addq = q[e];
        }
      uint32_t got = 0;
      if (add > 0) got = atomicAdd(qcount + addq, add);
#pragma unroll
      for (int e = 0; e < kGroup; ++e) {
        if (hits[e] == 0) continue;
        uint64_t at0 = qbase[q[e]] + readlane_u(got, lead[e]) + before[e];
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
          const bool mine = (hit >> (kSlots * e + k)) & 1u;
          const uint64_t m = __ballot(mine);
          const uint64_t at = at0 + lanes_below(m);
          if (mine && at < capacity) {
            int2 p;
            if constexpr (kPacked) p = make_int2(int(id[e][k] >> store.pid_bits), int(id[e][k] & pid_mask));
            else p = make_int2(int(id[e][k]), int(pid[e][k]));
            gat::store_pair(pairs + at, p);
          }
          at0 += uint32_t(__popcll(m));
        }
      }
    }
  }
}

// The reference's result form: one byte per (rectangle, trajectory), set where
// the trajectory has a point in the rectangle.  direct_refine_kernel's reads
// without its slots: hits store the same byte, so no atomics.
template <bool kPacked>
__global__ __launch_bounds__(kBlock) void direct_bitmap_kernel(
    Store store, const uint2* __restrict__ lq, const unsigned long long* __restrict__ lq_total, uint64_t lq_cap,
    const Node* __restrict__ nodes, uint32_t nnodes, const float4* __restrict__ boxes, uint32_t nqueries,
    uint8_t* __restrict__ bitmap, uint64_t stride) {
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint64_t wave = uniform((blockIdx.x * kBlock + threadIdx.x) / kWave);
  const uint64_t nwaves = uint64_t(gridDim.x) * (kBlock / kWave);
  const uint64_t total = *lq_total;
  const uint64_t n = total < lq_cap ? total : lq_cap;
  for (uint64_t g = wave; g < n; g += nwaves) {
    const uint2 e = lq[g];
    const uint32_t leaf = uniform(e.x), q = uniform(e.y);
    if (leaf >= nnodes || q >= nqueries) continue;
    const uint32_t start = uniform(nodes[leaf].start), count = uniform(nodes[leaf].count);
    if (uint64_t(start) + count > store.npoints) continue;
    const float4 box = boxes[q];
    uint8_t* row = bitmap + uint64_t(q) * stride;
    for (uint32_t base = 0; base < count; base += kSlots * kWave) {
      float2 v[kSlots];
      uint32_t id[kSlots];
#pragma unroll
      for (int k = 0; k < kSlots; ++k) {
        const uint32_t i = min(base + k * kWave + lane, count - 1);
        v[k] = store.xy[uint64_t(start) + i];
        id[k] = store.id[uint64_t(start) + i];
      }
#pragma unroll
      for (int k = 0; k < kSlots; ++k) {  // (a repeated last point sets its byte again)
        const uint32_t tid = kPacked ? id[k] >> store.pid_bits : id[k];
        if (in_box(box, v[k].x, v[k].y) && tid < stride) row[tid] = 1;
      }
    }
  }
}

// Counters (16 words) and, from word 32, one bit per byte of the bitmap to
// pinned host memory: an eighth of the bytes on the way there, which set the
// time of this step (100 rectangles over 20,000 trajectories: 2 MB as bytes,
// 40 us; 250 KB as bits).  The bitmap is whole 32-byte groups of 0 and 1.
__global__ __launch_bounds__(kBlock) void bitmap_finish_kernel(const uint32_t* __restrict__ counters,
                                                               const uint4* __restrict__ bitmap, uint64_t groups,
                                                               uint32_t* __restrict__ host) {
  const uint64_t i0 = uint64_t(blockIdx.x) * kBlock + threadIdx.x, stride = uint64_t(gridDim.x) * kBlock;
  if (i0 < 16) host[i0] = counters[i0];
  for (uint64_t i = i0; i < groups; i += stride) {
    const uint4 a = bitmap[2 * i], b = bitmap[2 * i + 1];
    // Bytes b0..b3 of a word to bits 28..31 of the product, which have no
    // other terms below them to carry.
    auto nibble = [](uint32_t w) { return (w * 0x10204080u) >> 28; };
    host[32 + i] = nibble(a.x) | nibble(a.y) << 4 | nibble(a.z) << 8 | nibble(a.w) << 12 | nibble(b.x) << 16 |
                   nibble(b.y) << 20 | nibble(b.z) << 24 | nibble(b.w) << 28;
  }
}

// The batch's counters, the time, the counts and the regions to pinned host
// memory: words [0, 16) counters, [16, 18) the time, [32, 32 + nq) counts, then
// from the next even word the regions.
__global__ __launch_bounds__(kBlock) void direct_finish_kernel(const uint32_t* __restrict__ counters,
                                                               const uint32_t* __restrict__ qcount,
                                                               const uint64_t* __restrict__ qbase, uint64_t nq,
                                                               uint32_t* __restrict__ host) {
  const uint64_t i0 = uint64_t(blockIdx.x) * kBlock + threadIdx.x, stride = uint64_t(gridDim.x) * kBlock;
  if (i0 < 16) host[i0] = counters[i0];
  if (i0 == 0) store_u64(host + 16, wall_clock64());
  uint64_t* base = reinterpret_cast<uint64_t*>(host + 32 + ((nq + 1) & ~uint64_t(1)));
  for (uint64_t i = i0; i < nq; i += stride) {
    host[32 + i] = qcount[i];
    base[i] = qbase[i];
  }
}

// A batch's pairs gathered query after query for a program that reads them
// back: one copy per rectangle from its region costs about 10 us each, whatever
// its size.  at[q] = the pairs of the queries before q.
__global__ __launch_bounds__(kBlock) void gather_offsets_kernel(const uint32_t* __restrict__ qcount, uint64_t nq,
                                                                unsigned long long* __restrict__ at) {
  __shared__ uint64_t wave_sum[kBlock / kWave];
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  uint64_t carry = 0;
  for (uint64_t b = 0; b < nq; b += kBlock) {
    const uint64_t v = b + t < nq ? qcount[b + t] : 0;
    uint64_t incl = v;
    for (int d = 1; d < kWave; d <<= 1) {
      const uint64_t o = __shfl_up(incl, d);
      if (lane >= uint32_t(d)) incl += o;
    }
    __syncthreads();  // every thread has read the previous round's sums
    if (lane == kWave - 1) wave_sum[w] = incl;
    __syncthreads();
    uint64_t before = carry;
    for (uint32_t k = 0; k < kBlock / kWave; ++k) {
      if (k < w) before += wave_sum[k];
      carry += wave_sum[k];
    }
    if (b + t < nq) at[b + t] = before + incl - v;
  }
}

// Per-query regions: a workgroup per query and span of its pairs.
__global__ __launch_bounds__(kBlock) void gather_regions_kernel(const int2* __restrict__ pairs, uint64_t npairs,
                                                                const uint64_t* __restrict__ qbase,
                                                                const uint32_t* __restrict__ qcount, uint32_t nq,
                                                                const unsigned long long* __restrict__ at,
                                                                int2* __restrict__ out, uint64_t capacity) {
  for (uint32_t q = blockIdx.x; q < nq; q += gridDim.x) {
    const uint64_t b = qbase[q], n = qcount[q], to = at[q];
    for (uint64_t i = uint64_t(blockIdx.y) * kBlock + threadIdx.x; i < n; i += uint64_t(gridDim.y) * kBlock)
      if (b + i < npairs && to + i < capacity) out[to + i] = pairs[b + i];
  }
}

// Run-indexed pairs: a 16-lane row per run, which takes its place among its
// query's runs (at[q] moves on by the run's pairs).
__global__ __launch_bounds__(kBlock) void gather_runs_kernel(const int2* __restrict__ pairs, uint64_t npairs,
                                                             const gat_range_run* __restrict__ runs, uint64_t nruns,
                                                             uint32_t nq, unsigned long long* __restrict__ at,
                                                             int2* __restrict__ out, uint64_t capacity) {
  const uint32_t l = threadIdx.x & 15;
  const uint64_t nrows = uint64_t(gridDim.x) * (kBlock / 16);
  for (uint64_t r = (uint64_t(blockIdx.x) * kBlock + threadIdx.x) / 16; r < nruns; r += nrows) {
    const gat_range_run run = runs[r];
    if (run.count == 0 || run.q >= nq || run.first > npairs || run.count > npairs - run.first) continue;
    unsigned long long to = 0;
    if (l == 0) to = atomicAdd(at + run.q, (unsigned long long)run.count);
    to = __shfl(to, 0, 16);
    for (uint32_t i = l; i < run.count; i += 16)
      if (to + i < capacity) out[to + i] = pairs[run.first + i];
  }
}

int blocks_for(uint64_t n, uint64_t most) {
  uint64_t b = (n + kBlock - 1) / kBlock;
  if (b > most) b = most;
  return int(b == 0 ? 1 : b);
}

}  // namespace

extern "C" {

int gat_stage_in(void* dst, const void* src_pinned, int64_t bytes, int32_t nspans, uint32_t* const* spans,
                 const int64_t* words, uint32_t* stamp, void* stream) {
  GAT_REQUIRE(bytes >= 0 && bytes % 4 == 0 && (bytes == 0 || (dst && src_pinned)), "gat_stage_in: bad copy");
  GAT_REQUIRE(nspans >= 0 && nspans <= kSpans && (nspans == 0 || (spans && words)), "gat_stage_in: bad spans");
  Spans f{};
  uint64_t total = 0;
  for (int k = 0; k < kSpans; ++k) {
    if (k < nspans) {
      GAT_REQUIRE(words[k] >= 0 && (words[k] == 0 || spans[k]), "gat_stage_in: bad span");
      f.p[k] = spans[k];
      total += uint64_t(words[k]);
    }
    f.end[k] = total;
  }
  const uint64_t n = uint64_t(bytes) / 4 > total ? uint64_t(bytes) / 4 : total;
  stage_in_kernel<<<dim3{uint32_t(blocks_for(n, uint64_t(gat::cu_count()) * 4))}, dim3{uint32_t(kBlock)}, 0,
                    gat::as_stream(stream)>>>(static_cast<const uint32_t*>(src_pinned), static_cast<uint32_t*>(dst),
                                              uint64_t(bytes) / 4, f, stamp);
  GAT_LAUNCH_CHECK("stage_in_kernel");
  return GAT_OK;
}

int gat_direct_regions(const uint64_t* cand, int64_t nq, uint64_t* qbase, uint32_t* qcount, uint32_t* counters,
                       void* stream) {
  GAT_REQUIRE(nq >= 0 && counters && (nq == 0 || (cand && qbase && qcount)), "gat_direct_regions: bad arguments");
  direct_regions_kernel<<<dim3{1}, dim3{uint32_t(kBlock)}, 0, gat::as_stream(stream)>>>(cand, uint64_t(nq), qbase,
                                                                                        qcount, counters);
  GAT_LAUNCH_CHECK("direct_regions_kernel");
  return GAT_OK;
}

int gat_direct_refine(const gat_point_store* sp, const uint32_t* leaf_query, const uint64_t* lq_total,
                      int64_t lq_capacity, int64_t expected, const gat_tree_node* nodes, int64_t nnodes,
                      const float* boxes, int64_t nqueries, const uint64_t* qbase, uint32_t* qcount, int32_t* pairs,
                      int64_t capacity, void* stream) {
  GAT_REQUIRE(sp && sp->npoints >= 0 && sp->pid_bits >= 0 && sp->pid_bits < 32, "gat_direct_refine: bad store");
  GAT_REQUIRE(sp->npoints == 0 || (sp->xy_dev && sp->id_dev && (sp->pid_bits > 0 || sp->pid_dev)),
              "gat_direct_refine: null store array");
  GAT_REQUIRE(lq_total && nodes && nnodes >= 1 && nnodes < int64_t(INT32_MAX) && lq_capacity >= 0 && expected >= 0 &&
                  nqueries >= 0 && nqueries <= int64_t(UINT32_MAX) && capacity >= 0,
              "gat_direct_refine: bad sizes");
  if (lq_capacity == 0 || nqueries == 0) return GAT_OK;
  GAT_REQUIRE(leaf_query && boxes && qbase && qcount && (pairs || capacity == 0), "gat_direct_refine: null pointer");
  const Store st{reinterpret_cast<const float2*>(sp->xy_dev), sp->id_dev, sp->pid_dev, uint64_t(sp->npoints),
                 uint32_t(sp->pid_bits)};
  // The entry count is known on the device only: a grid for the expected
  // number, and a stride for what exceeds it.
  const int64_t most = int64_t(gat::cu_count()) * 16;
  int64_t blocks = (expected + kGroup * (kBlock / kWave) - 1) / (kGroup * (kBlock / kWave));
  blocks = blocks < 64 ? 64 : blocks > most ? most : blocks;
  const dim3 grid{uint32_t(blocks)}, block{uint32_t(kBlock)};
  hipStream_t s = gat::as_stream(stream);
  const auto* L = reinterpret_cast<const uint2*>(leaf_query);
  const auto* T = reinterpret_cast<const unsigned long long*>(lq_total);
  const auto* N = reinterpret_cast<const Node*>(nodes);
  const auto* B = reinterpret_cast<const float4*>(boxes);
  auto* P = reinterpret_cast<int2*>(pairs);
  if (sp->pid_bits > 0)
    direct_refine_kernel<true><<<grid, block, 0, s>>>(st, L, T, uint64_t(lq_capacity), N, uint32_t(nnodes), B,
                                                      uint32_t(nqueries), qbase, qcount, P, uint64_t(capacity));
  else
    direct_refine_kernel<false><<<grid, block, 0, s>>>(st, L, T, uint64_t(lq_capacity), N, uint32_t(nnodes), B,
                                                       uint32_t(nqueries), qbase, qcount, P, uint64_t(capacity));
  GAT_LAUNCH_CHECK("direct_refine_kernel");
  return GAT_OK;
}

int gat_direct_bitmap(const gat_point_store* sp, const uint32_t* leaf_query, const uint64_t* lq_total,
                      int64_t lq_capacity, int64_t expected, const gat_tree_node* nodes, int64_t nnodes,
                      const float* boxes, int64_t nqueries, uint8_t* bitmap, int64_t stride, void* stream) {
  GAT_REQUIRE(sp && sp->npoints >= 0 && sp->pid_bits >= 0 && sp->pid_bits < 32, "gat_direct_bitmap: bad store");
  GAT_REQUIRE(sp->npoints == 0 || (sp->xy_dev && sp->id_dev), "gat_direct_bitmap: null store array");
  GAT_REQUIRE(lq_total && nodes && nnodes >= 1 && nnodes < int64_t(INT32_MAX) && lq_capacity >= 0 && expected >= 0 &&
                  nqueries >= 0 && nqueries <= int64_t(UINT32_MAX) && stride >= 1,
              "gat_direct_bitmap: bad sizes");
  if (lq_capacity == 0 || nqueries == 0) return GAT_OK;
  GAT_REQUIRE(leaf_query && boxes && bitmap, "gat_direct_bitmap: null pointer");
  const Store st{reinterpret_cast<const float2*>(sp->xy_dev), sp->id_dev, sp->pid_dev, uint64_t(sp->npoints),
                 uint32_t(sp->pid_bits)};
  const int64_t most = int64_t(gat::cu_count()) * 16;
  int64_t blocks = (expected + kBlock / kWave - 1) / (kBlock / kWave);
  blocks = blocks < 64 ? 64 : blocks > most ? most : blocks;
  const dim3 grid{uint32_t(blocks)}, block{uint32_t(kBlock)};
  hipStream_t s = gat::as_stream(stream);
  const auto* L = reinterpret_cast<const uint2*>(leaf_query);
  const auto* T = reinterpret_cast<const unsigned long long*>(lq_total);
  const auto* N = reinterpret_cast<const Node*>(nodes);
  const auto* B = reinterpret_cast<const float4*>(boxes);
  if (sp->pid_bits > 0)
    direct_bitmap_kernel<true><<<grid, block, 0, s>>>(st, L, T, uint64_t(lq_capacity), N, uint32_t(nnodes), B,
                                                      uint32_t(nqueries), bitmap, uint64_t(stride));
  else
    direct_bitmap_kernel<false><<<grid, block, 0, s>>>(st, L, T, uint64_t(lq_capacity), N, uint32_t(nnodes), B,
                                                       uint32_t(nqueries), bitmap, uint64_t(stride));
  GAT_LAUNCH_CHECK("direct_bitmap_kernel");
  return GAT_OK;
}

int gat_bitmap_finish(const uint32_t* counters, const uint8_t* bitmap, int64_t bytes, uint32_t* out_pinned,
                      void* stream) {
  GAT_REQUIRE(bytes >= 0 && bytes % 32 == 0 && counters && out_pinned && (bytes == 0 || bitmap) &&
                  reinterpret_cast<uintptr_t>(bitmap) % 16 == 0,
              "gat_bitmap_finish: bad arguments");
  const uint64_t groups = uint64_t(bytes) / 32;
  bitmap_finish_kernel<<<dim3{uint32_t(blocks_for(groups, uint64_t(gat::cu_count()) * 8))}, dim3{uint32_t(kBlock)}, 0,
                         gat::as_stream(stream)>>>(counters, reinterpret_cast<const uint4*>(bitmap), groups,
                                                   out_pinned);
  GAT_LAUNCH_CHECK("bitmap_finish_kernel");
  return GAT_OK;
}

int64_t gat_direct_words(int64_t nq) { return nq < 0 ? 0 : 32 + ((nq + 1) & ~int64_t(1)) + 2 * nq; }

int gat_direct_finish(const uint32_t* counters, const uint32_t* qcount, const uint64_t* qbase, int64_t nq,
                      uint32_t* out_pinned, void* stream) {
  GAT_REQUIRE(nq >= 0 && counters && out_pinned && (nq == 0 || (qcount && qbase)), "gat_direct_finish: bad arguments");
  direct_finish_kernel<<<dim3{uint32_t(blocks_for(uint64_t(nq), 64))}, dim3{uint32_t(kBlock)}, 0,
                         gat::as_stream(stream)>>>(counters, qcount, qbase, uint64_t(nq), out_pinned);
  GAT_LAUNCH_CHECK("direct_finish_kernel");
  return GAT_OK;
}

int gat_gather_pairs(const int32_t* pairs, int64_t npairs, const uint64_t* qbase, const gat_range_run* runs,
                     int64_t nruns, const uint32_t* qcount, int64_t nq, uint64_t* at, int32_t* out, int64_t capacity,
                     void* stream) {
  GAT_REQUIRE(npairs >= 0 && nruns >= 0 && capacity >= 0 && nq >= 0 && nq <= int64_t(UINT32_MAX),
              "gat_gather_pairs: bad sizes");
  GAT_REQUIRE((qbase == nullptr) != (runs == nullptr) || nq == 0 || (!qbase && nruns == 0),
              "gat_gather_pairs: regions or runs, not both");
  if (nq == 0) return GAT_OK;
  GAT_REQUIRE(qcount && at && (capacity == 0 || out) && (npairs == 0 || pairs), "gat_gather_pairs: null pointer");
  hipStream_t s = gat::as_stream(stream);
  auto* A = reinterpret_cast<unsigned long long*>(at);
  const auto* P = reinterpret_cast<const int2*>(pairs);
  auto* O = reinterpret_cast<int2*>(out);
  gather_offsets_kernel<<<dim3{1}, dim3{uint32_t(kBlock)}, 0, s>>>(qcount, uint64_t(nq), A);
  GAT_LAUNCH_CHECK("gather_offsets_kernel");
  const int64_t most = int64_t(gat::cu_count()) * 8;
  if (qbase) {
    const int64_t blocks = nq < most ? nq : most;
    const int64_t split = most / blocks < 32 ? most / blocks : 32;  // at least 1
    gather_regions_kernel<<<dim3{uint32_t(blocks), uint32_t(split)}, dim3{uint32_t(kBlock)}, 0, s>>>(
        P, uint64_t(npairs), qbase, qcount, uint32_t(nq), A, O, uint64_t(capacity));
    GAT_LAUNCH_CHECK("gather_regions_kernel");
  } else if (nruns > 0) {
    gather_runs_kernel<<<dim3{uint32_t(blocks_for(uint64_t(nruns) * 16, uint64_t(most)))}, dim3{uint32_t(kBlock)}, 0,
                         s>>>(P, uint64_t(npairs), runs, uint64_t(nruns), uint32_t(nq), A, O, uint64_t(capacity));
    GAT_LAUNCH_CHECK("gather_runs_kernel");
  }
  return GAT_OK;
}

int gat_wall_clock_khz(int32_t* khz) {
  GAT_REQUIRE(khz, "gat_wall_clock_khz: null output");
  int dev = 0, rate = 0;
  GAT_HIP_CHECK(hipGetDevice(&dev));
  GAT_HIP_CHECK(hipDeviceGetAttribute(&rate, hipDeviceAttributeWallClockRate, dev));
  GAT_REQUIRE(rate > 0, "gat_wall_clock_khz: the device reports no rate");
  *khz = rate;
  return GAT_OK;
}

}  // extern "C"
