// EDR kernels for gfx950: the dynamic program of Grid::SimilarityExecuter
// (Grid.cpp:1222-1318) behind top-k trajectory similarity.
//
// The reference's cell rule (Grid.cpp:1288-1300) is not the textbook minimum:
// with M = D[r-1][c-1] + s, U = D[r-1][c] + 1 and L = D[r][c-1] + 1 it returns M
// when M is strictly smallest, L when L is strictly smallest, and U otherwise —
// including M == L < U.  Every kernel here evaluates that rule exactly.
//
// This file holds the plain drop-in for EDRDistance_Batch (kernel.cu:249-501):
// one wave per (query, candidate) task, in the order given.  The reference
// runs a workgroup per task, anti-diagonal by anti-diagonal with a barrier
// each, and stops at 1024 points (kernel.cu:263); here a wave sweeps the table
// in strips of up to 256 rows with its neighbours in registers (edr_dp.hpp),
// for lengths up to GAT_MAX_TRAJ_LEN.
#include "edr_dp.hpp"
#include "gat_common.hpp"

namespace {

constexpr int kMaxLen = GAT_MAX_TRAJ_LEN;

// The handler's stores carry no padding and its lengths are known on the
// device only, so every column load is checked and the row buffer is sized
// for the longest trajectory (8.8 KB of LDS: 16 waves per CU).
__global__ __launch_bounds__(64, 4) void edr_plain_kernel(
    int ntasks, const gat_edr_task* __restrict__ tasks, const float2* __restrict__ qxy, const int32_t* __restrict__ qoff,
    const int32_t* __restrict__ qlen, const float2* __restrict__ cxy, const int64_t* __restrict__ coff,
    const int32_t* __restrict__ clen, float u, int32_t* __restrict__ result) {
  // Columns from -63 on, the first a feed reads (column 1) 16-byte aligned.
  __shared__ __align__(16) int32_t above[edr::kOff64 + kMaxLen + 64 + edr::kBlk][1];
  const int t = blockIdx.x;
  const int l = threadIdx.x;
  if (t >= ntasks) return;
  const gat_edr_task task = tasks[t];
  const int qn = __builtin_amdgcn_readfirstlane(qlen[task.qid]);
  const int cn = __builtin_amdgcn_readfirstlane(clen[t]);
  // Rows are the shorter trajectory; on equal lengths the query (Grid.cpp:1234-1247).
  const bool query_rows = cn >= qn;
  const int n = query_rows ? qn : cn;
  const int m = query_rows ? cn : qn;
  if (n < 0 || m > kMaxLen) {  // rejected by the host wrapper; never indexes out of bounds
    if (l == 0) result[t] = -1;
    return;
  }
  if (n == 0) {  // D[0][m] = m (Grid.cpp:1269-1272)
    if (l == 0) result[t] = m;
    return;
  }
  const float2* R = query_rows ? qxy + qoff[task.qid] : cxy + coff[t];
  const float2* C = query_rows ? cxy + coff[t] : qxy + qoff[task.qid];
  for (int i = l; i < m + edr::kOff64 + 64 + edr::kBlk; i += 64) above[i][0] = i - edr::kOff64;
  const int ns[1] = {n}, ms[1] = {m};
  bool mine = false;
  const int res = edr::sweep_pairs<64, true>(R, n, C, m, n, m, ns, ms, u, above, 0, l, &mine);
  if (mine) result[t] = res + n;  // D = E + n
}

}  // namespace

extern "C" {

int gatEDRDistanceBatchHandler(int queryTaskNum, const gat_edr_task* tasks, const float* query_xy,
                               const int32_t* query_offset, const int32_t* query_length, const float* cand_xy,
                               const int64_t* cand_offset, const int32_t* cand_length, double eps, int32_t* result,
                               void* stream) {
  GAT_REQUIRE(queryTaskNum >= 0, "EDR batch: negative task count");
  if (queryTaskNum == 0) return GAT_OK;
  GAT_REQUIRE(tasks && query_xy && query_offset && query_length && cand_xy && cand_offset && cand_length && result,
              "EDR batch: null pointer");
  GAT_REQUIRE(eps > 0, "EDR batch: eps must be positive");
  edr_plain_kernel<<<dim3(uint32_t(queryTaskNum)), dim3(64), 0, gat::as_stream(stream)>>>(
      queryTaskNum, tasks, reinterpret_cast<const float2*>(query_xy), query_offset, query_length,
      reinterpret_cast<const float2*>(cand_xy), cand_offset, cand_length, gat_eps_threshold(eps), result);
  GAT_LAUNCH_CHECK("edr_plain_kernel");
  return GAT_OK;
}

}  // extern "C"
