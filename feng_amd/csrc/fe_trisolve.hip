// Exact ILU(0) application of small systems in one launch (the PCILU solves
// of the reference's GMRES runs, feLinearSystemPETSc.cpp:900-1031).
//
// z = U^-1 L^-1 v over the dependency levels of both triangles is a chain of
// levels with a few dozen rows each: what bounds it is the latency of one
// level times their number, not the entries (138 levels per triangle for
// 3,481 unknowns of cubic triangles, 25 rows a level).  So the whole chain
// runs in one workgroup with the solution vector in LDS: a level costs an LDS
// gather, a reduction over a row's lanes in registers and a barrier that waits for
// LDS only, while the matrix entries of the next steps (kept in the order of
// the schedule, so that a wavefront reads them contiguously) are already in
// flight to registers.  Measured at 3,481 unknowns: 42.4 ms -> 14.3 ms for
// 100 GMRES steps against one workgroup per run of levels that gathered the
// solution from global memory (376 -> 99 us per application).
//
// A step is up to TB / LPR rows of one level, LPR lanes a row, K entries a
// lane (K of the step's longest row), one of them the row's own right-hand
// side; an entry is 16 bytes (value, LDS offset of its column), read by one
// load whose address is a scalar plus the lane.  The rule (feTriSolveBuild):
// the vector and the steps have to fit the LDS, a row at most 16 kMaxK
// entries, and the levels must be narrow (at most kMaxSteps steps a level on
// average: about 2.4 us at 0.3 us a step, where a launch per level costs 4.8 us
// and spreads the rows over many workgroups).
#include "fe_hip_internal.h"

#include <algorithm>
#include <vector>

struct FeTriSolve {
  bool usable = false;
  int steps = 0, K = 0, LPR = 0, TB = 0;
  int64_t slots = 0;
  int4 *d_step = nullptr;   // first slot, lanes in use, K, 0
  int *d_map = nullptr;     // slot -> entry of G (< nnzL), nnzL + entry of G^T, -2 - row: the row's own
                            // right-hand side in the lower solve, -2 - n - row in the upper one, -1 none
  uint4 *d_ent = nullptr;   // slot -> value, LDS offset of the column
};

namespace {

constexpr int kMaxTB = 512;
constexpr int kMaxK = 6;          // entries per lane
constexpr int kMaxN = 16384;      // the solution: 128 KB of LDS
constexpr int kMaxStep = 1920;    // the steps' descriptors: 30 KB of LDS
constexpr int kMaxSteps = 8;
constexpr int kAhead = 4;         // steps whose entries are in flight

// Values in schedule order: the strict entries of G = I - L and of
// G^T = I - D^-1 U, and per row the factor of its right-hand side (1, 1 / u_ii).
__global__ void triPack(int64_t slots, const int *__restrict__ map, int nnzL, const double *__restrict__ gL,
                        const double *__restrict__ gU, int n, const double *__restrict__ dinv, uint4 *__restrict__ ent)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(t >= slots) return;
  const int m = map[t];
  double v = 0.;
  if(m >= 0) v = m < nnzL ? gL[m] : gU[m - nnzL];
  else if(m <= -2) v = -2 - m < n ? 1. : dinv[-2 - m - n];
  *(double *)(ent + t) = v;
}

// Sum over the LPR (4, 8, 16) lanes of a row, in every one of them: lane ^ 1,
// lane ^ 2, then the mirrored half-row of 8 and row of 16 (whose halves
// already agree).
template <int CTRL>
__device__ __forceinline__ double dppMove(double v)
{
  const unsigned long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffull), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((unsigned long long)(unsigned)lo | (unsigned long long)(unsigned)hi << 32);
}
template <int LPR>
__device__ __forceinline__ double rowSum(double v)
{
  v += dppMove<0xB1>(v);                           // quad_perm [1, 0, 3, 2]
  v += dppMove<0x4E>(v);                           // quad_perm [2, 3, 0, 1]
  if constexpr(LPR >= 8) v += dppMove<0x141>(v);   // row_half_mirror
  if constexpr(LPR >= 16) v += dppMove<0x140>(v);  // row_mirror
  return v;
}

// Orders the LDS accesses of the workgroup without waiting for the loads of
// the coming steps (__syncthreads would drain them).
__device__ __forceinline__ void ldsBarrier()
{
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int TB, int LPR, int KM>
__global__ __launch_bounds__(TB) void triSolve(int n, int steps, const int4 *__restrict__ step,
                                               const uint4 *__restrict__ ent, const double *__restrict__ v,
                                               double *__restrict__ z)
{
  __shared__ double x[kMaxN];
  __shared__ int4 ds[kMaxStep + 1];
  const int t = threadIdx.x;
  for(int i = t; i < n; i += TB) x[i] = v[i];
  for(int s = t; s <= steps; s += TB) ds[s] = s < steps ? step[s] : make_int4(0, 0, 0, 0);
  __syncthreads();
  const int wave0 = __builtin_amdgcn_readfirstlane(t & ~63);
  uint4 e[kAhead][KM];
  int lanes[kAhead];
  int4 next = ds[0];  // descriptor of the step fetched next, read a step ahead
  // The loads are unconditional (slots 0 .. TB - 1 are empty entries, lanes
  // past the step's repeat its last one), so their number is known and the
  // wait for one step's entries leaves the later steps' in flight.
  auto fetch = [&](int s, int u) {
    const int base = __builtin_amdgcn_readfirstlane(next.x), use = __builtin_amdgcn_readfirstlane(next.y),
              K = __builtin_amdgcn_readfirstlane(next.z);
    next = ds[min(s + 1, steps)];
    lanes[u] = use;
    const int o = use > 0 ? min(t, use - 1) : t;
#pragma unroll
    for(int q = 0; q < KM; ++q) {
      const uint4 *p = ent + (q < K ? base + q * use : 0);
      e[u][q] = p[o];
    }
    __builtin_amdgcn_sched_barrier(0);  // the steps' loads stay in step order
  };
#pragma unroll
  for(int u = 0; u < kAhead; ++u) fetch(u, u);
  for(int s0 = 0; s0 < steps; s0 += kAhead) {
#pragma unroll
    for(int u = 0; u < kAhead; ++u) {
      if(wave0 < lanes[u]) {
        double g[KM];
#pragma unroll
        for(int q = 0; q < KM; ++q) g[q] = *(const double *)((const char *)x + e[u][q].z);
        double acc = 0.;
#pragma unroll
        for(int q = 0; q < KM; ++q)
          acc += __longlong_as_double((unsigned long long)e[u][q].x | (unsigned long long)e[u][q].y << 32) * g[q];
        acc = rowSum<LPR>(acc);
        // a row's own entry is the first of its first lane
        if(t < lanes[u] && t % LPR == 0) *(double *)((char *)x + e[u][0].z) = acc;
      }
      ldsBarrier();
      fetch(s0 + u + kAhead, u);
    }
  }
  for(int i = t; i < n; i += TB) z[i] = x[i];
}

template <typename T>
int upload(fe_hip_ctx *ctx, T **d, const std::vector<T> &h)
{
  if(int rc = feAlloc(ctx, d, std::max<size_t>(1, h.size()))) return rc;
  if(!h.empty()) FE_HIP_TRY(ctx, hipMemcpy(*d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice));
  return FE_STATUS_OK;
}

}  // namespace

int feTriSolveBuild(fe_hip_ctx *ctx)
{
  if(ctx->tri) return FE_STATUS_OK;
  ctx->tri = new FeTriSolve();
  FeTriSolve &T = *ctx->tri;
  const FePrecond &P = ctx->pc;
  const int n = ctx->n;
  if(n > kMaxN || P.nnzL + P.nnzU >= (int64_t)1 << 30) return FE_STATUS_OK;
  std::vector<int> ia[2], ja[2], lr[2];
  const int *dIa[2] = {P.d_iaL, P.d_iaU}, *dJa[2] = {P.d_jaL, P.d_jaU}, *dRows[2] = {P.d_levelRows, P.d_levelRowsU};
  const std::vector<int> *lp[2] = {&P.levelPtr, &P.levelPtrU};
  const int64_t nz[2] = {P.nnzL, P.nnzU};
  int64_t levels = 0, lanesUsed = 0;
  int longest = 0;  // entries of a row, its own right-hand side among them
  for(int t = 0; t < 2; ++t) {
    ia[t].resize(n + 1);
    ja[t].resize(nz[t]);
    lr[t].resize(n);
    FE_HIP_TRY(ctx, hipMemcpy(ia[t].data(), dIa[t], sizeof(int) * (n + 1), hipMemcpyDeviceToHost));
    FE_HIP_TRY(ctx, hipMemcpy(ja[t].data(), dJa[t], sizeof(int) * nz[t], hipMemcpyDeviceToHost));
    FE_HIP_TRY(ctx, hipMemcpy(lr[t].data(), dRows[t], sizeof(int) * n, hipMemcpyDeviceToHost));
    for(int i = 0; i < n; ++i) longest = std::max(longest, ia[t][i + 1] - ia[t][i]);
    levels += (int64_t)lp[t]->size() - 1;
  }
  // lanes a row: about half the longest row, so that K is 2 to 4 and short
  // rows waste little; a workgroup of 256 where the levels fill no more
  T.LPR = longest <= 10 ? 4 : longest <= 24 ? 8 : 16;
  lanesUsed = 2 * (int64_t)n * T.LPR;
  T.TB = lanesUsed <= 256 * levels ? 256 : kMaxTB;
  const int kRows = T.TB / T.LPR;
  int64_t steps = 0;
  for(int t = 0; t < 2; ++t)
    for(size_t l = 0; l + 1 < lp[t]->size(); ++l) steps += ((*lp[t])[l + 1] - (*lp[t])[l] + kRows - 1) / kRows;
  if(longest > kMaxK * T.LPR || steps > kMaxStep || steps > kMaxSteps * levels) return FE_STATUS_OK;
  std::vector<int4> step;
  std::vector<int> map(T.TB, -1), col(T.TB, 0);  // slots 0 .. TB - 1: empty entries
  for(int t = 0; t < 2; ++t) {
    for(size_t l = 0; l + 1 < lp[t]->size(); ++l) {
      const int e = (*lp[t])[l + 1];
      for(int b = (*lp[t])[l]; b < e; b += kRows) {
        const int cnt = std::min(kRows, e - b), use = cnt * T.LPR;
        int K = 0;
        for(int r = 0; r < cnt; ++r) {
          const int i = lr[t][b + r];
          K = std::max(K, (ia[t][i + 1] - ia[t][i] + T.LPR - 1) / T.LPR);
        }
        const size_t base = map.size();
        step.push_back(make_int4((int)base, use, K, 0));
        T.K = std::max(T.K, K);
        map.resize(base + (size_t)K * use, -1);
        col.resize(map.size(), 0);
        for(int r = 0; r < cnt; ++r) {
          const int i = lr[t][b + r];
          // entry m of a row: lane m % LPR, its slot m / LPR
          auto slot = [&](int m) { return base + (size_t)(m / T.LPR) * use + r * T.LPR + m % T.LPR; };
          for(int m = 0; m < K * T.LPR; ++m) col[slot(m)] = 8 * i;
          map[slot(0)] = -2 - i - (t ? n : 0);
          int m = 1;
          for(int k = ia[t][i]; k < ia[t][i + 1]; ++k) {
            if(ja[t][k] == i) continue;  // the unit diagonal
            map[slot(m)] = k + (t ? (int)P.nnzL : 0);
            col[slot(m)] = 8 * ja[t][k];
            ++m;
          }
        }
      }
    }
  }
  T.steps = (int)step.size();
  T.slots = (int64_t)map.size();
  std::vector<uint4> ent(map.size());
  for(size_t q = 0; q < ent.size(); ++q) ent[q] = make_uint4(0, 0, (unsigned)col[q], 0);
  if(upload(ctx, &T.d_step, step) || upload(ctx, &T.d_map, map) || upload(ctx, &T.d_ent, ent))
    return FE_STATUS_OUT_OF_MEMORY;
  T.usable = true;
  return FE_STATUS_OK;
}

bool feTriSolveUsable(const fe_hip_ctx *ctx) { return ctx->tri && ctx->tri->usable; }

int feTriSolvePack(fe_hip_ctx *ctx)
{
  FeTriSolve &T = *ctx->tri;
  const FePrecond &P = ctx->pc;
  hipLaunchKernelGGL(triPack, dim3((unsigned)((T.slots + 255) / 256)), dim3(256), 0, ctx->stream, T.slots, T.d_map,
                     (int)P.nnzL, P.d_gL64, P.d_gU64, ctx->n, P.d_dinv64, T.d_ent);
  FE_HIP_TRY(ctx, hipGetLastError());
  return FE_STATUS_OK;
}

namespace {

template <int TB, int LPR>
void launchTri(fe_hip_ctx *ctx, const FeTriSolve &T, const double *v, double *z)
{
#define FE_TRI(KM_) \
  hipLaunchKernelGGL((triSolve<TB, LPR, KM_>), dim3(1), dim3(TB), 0, ctx->stream, ctx->n, T.steps, T.d_step, T.d_ent, v, z)
  switch(T.K) {
    case 1: FE_TRI(1); break;
    case 2: FE_TRI(2); break;
    case 3: FE_TRI(3); break;
    case 4: FE_TRI(4); break;
    case 5: FE_TRI(5); break;
    default: FE_TRI(6); break;
  }
#undef FE_TRI
}

}  // namespace

int feTriSolveApply(fe_hip_ctx *ctx, const double *v, double *z)
{
  const FeTriSolve &T = *ctx->tri;
  if(T.TB == 256) {
    if(T.LPR == 4) launchTri<256, 4>(ctx, T, v, z);
    else if(T.LPR == 8) launchTri<256, 8>(ctx, T, v, z);
    else launchTri<256, 16>(ctx, T, v, z);
  } else {
    if(T.LPR == 4) launchTri<512, 4>(ctx, T, v, z);
    else if(T.LPR == 8) launchTri<512, 8>(ctx, T, v, z);
    else launchTri<512, 16>(ctx, T, v, z);
  }
  FE_HIP_TRY(ctx, hipGetLastError());
  return FE_STATUS_OK;
}

void feTriSolveRelease(fe_hip_ctx *ctx)
{
  delete ctx->tri;  // device buffers are owned by the context
  ctx->tri = nullptr;
}
