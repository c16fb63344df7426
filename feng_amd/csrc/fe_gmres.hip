// Restarted GMRES(m) on the device (the KSPGMRES the reference's
// Navier-Stokes runs select, feLinearSystemPETSc.cpp:900-1031; restart 30 by
// PETSc default, 50 in the configs), FP64, right preconditioned so the
// monitored residual is the true residual of A x = b.
//
// Arnoldi uses classical Gram-Schmidt (PETSc's default orthogonalization,
// no refinement), or with one reorthogonalization (CGS2, `gmres_orth` 2).
// The whole solve stays on the device: the projections, the Hessenberg
// column with its Givens rotations, the stop test, the triangular solve of a
// cycle's end and the true residual of a restart.  A step is the
// preconditioner, the product and three launches --
//   gmDots : block partials of (V_k, w), k <= j (rows x groups of vectors)
//   gmAxpy : h = folded partials, w -= V h, block partials of (w, w)
//   gmNext : V_j+1 = w / ||w||; one extra block rotates the Hessenberg column
//            and posts the step and the stop code to a pinned mailbox
// -- and the host only launches: it stays at most kGmAhead steps ahead of the
// mailbox and never waits for a value inside a cycle.  What bounds a step of
// up to some 10^5 unknowns is the latency of its dependent launches, so the
// reductions are folded by their consumers (the partials are kept to
// kGmChunks per vector so that every block can fold them all).  Kovasznay
// flow, Taylor-Hood 36^2 / 112^2 (n = 11,307 / 111,779), one Newton solve:
// 70.5 / 179.5 ms with a host-driven form (4 stream synchronizations and
// 1024-block reductions per step), 28.3 / 93.3 ms with this one.
//
// Preconditioners: Jacobi, or ILU(0) (exact incomplete factors from
// fe_precond.hip, PETSc's PCILU) applied by exact triangular solves
// scheduled by dependency levels -- y = L^-1 r over the levels of the lower
// triangle, z = U^-1 y over those of the upper one; the rows of a level are
// independent, a level of many rows is one launch, a run of consecutive
// levels of few rows is one workgroup with a barrier between levels -- or,
// with `ilu_sweeps` = k > 0, by k Jacobi iterations per factor (the parallel
// approximate triangular solve: y <- r - L_strict y, z <- D^-1 (y - U_strict z)).
#include "fe_hip_internal.h"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <vector>

namespace {

constexpr int kTB = 256;
constexpr int kG = 1024;

template <int LPR>
__global__ __launch_bounds__(kTB) void spmv64(int n, const int *__restrict__ ia, const int *__restrict__ ja,
                                              const double *__restrict__ val, const double *__restrict__ x,
                                              double *__restrict__ y)
{
  constexpr int RPB = kTB / LPR;
  const int sub = threadIdx.x % LPR;
  const int nChunks = (n + RPB - 1) / RPB;
  for(int chunk = blockIdx.x; chunk < nChunks; chunk += gridDim.x) {
    const int row = chunk * RPB + threadIdx.x / LPR;
    double s = 0.;
    if(row < n)
      s = feRowDot<FeKs<LPR>::value, LPR>(ja, val, ia[row] + sub, ia[row + 1], [&](int j) { return x[j]; });
#pragma unroll
    for(int o = LPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, LPR);
    if(sub == 0 && row < n) y[row] = s;
  }
}

// out_i = scale_i * in0_i + sum_{j != i} g_ij v_j over a unit-diagonal factor.
__global__ __launch_bounds__(kTB) void factorSweep(int n, const int *__restrict__ ia, const int *__restrict__ ja,
                                                   const double *__restrict__ g, const double *__restrict__ scale,
                                                   const double *__restrict__ in0, const double *__restrict__ v,
                                                   double *__restrict__ out)
{
  for(int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    double s = scale ? scale[i] * in0[i] : in0[i];
    for(int k = ia[i]; k < ia[i + 1]; ++k) {
      const int j = ja[k];
      if(j != i) s += g[k] * (scale ? v[j] : v[j]);
    }
    out[i] = s;
  }
}

constexpr int kTriLPR = 8;      // lanes per row of the exact triangular solves
constexpr int kTriRunTB = 1024;  // workgroup of a run of small levels
constexpr int kTriSmall = 256;   // levels of at most this many rows join a run

// Row i of an exact triangular solve: out_i = (scale ? scale_i in0_i : in0_i)
// + sum_{j != i} g_ij out_j, the out_j of earlier levels.  kTriLPR lanes per
// row; every lane of the group takes part in the reduction.
__device__ __forceinline__ void triRow(bool on, int i, int sub, const int *__restrict__ ia, const int *__restrict__ ja,
                                       const double *__restrict__ g, const double *__restrict__ scale,
                                       const double *__restrict__ in0, double *out)
{
  double s = 0.;
  if(on)
    for(int k = ia[i] + sub; k < ia[i + 1]; k += kTriLPR) {
      const int j = ja[k];
      if(j != i) s += g[k] * out[j];
    }
#pragma unroll
  for(int o = kTriLPR / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, kTriLPR);
  if(on && sub == 0) out[i] = (scale ? scale[i] * in0[i] : in0[i]) + s;
}

// One level of many rows.
__global__ __launch_bounds__(256) void triLevel(const int *__restrict__ rows, int count, const int *__restrict__ ia,
                                                const int *__restrict__ ja, const double *__restrict__ g,
                                                const double *__restrict__ scale, const double *__restrict__ in0,
                                                double *out)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = t / kTriLPR, sub = t % kTriLPR;
  const bool on = r < count;
  triRow(on, on ? rows[r] : 0, sub, ia, ja, g, scale, in0, out);
}

// Levels l0 .. l1 - 1, each of few rows, in one workgroup: a barrier between
// levels orders the writes of one level before the reads of the next.
__global__ __launch_bounds__(kTriRunTB) void triLevelRun(const int *__restrict__ levelPtr, int l0, int l1,
                                                         const int *__restrict__ rows, const int *__restrict__ ia,
                                                         const int *__restrict__ ja, const double *__restrict__ g,
                                                         const double *__restrict__ scale,
                                                         const double *__restrict__ in0, double *out)
{
  constexpr int RPP = kTriRunTB / kTriLPR;  // rows per pass
  const int sub = threadIdx.x % kTriLPR;
  for(int l = l0; l < l1; ++l) {
    const int b = levelPtr[l], cnt = levelPtr[l + 1] - b;
    for(int r0 = 0; r0 < cnt; r0 += RPP) {
      const int r = r0 + (int)threadIdx.x / kTriLPR;
      const bool on = r < cnt;
      triRow(on, on ? rows[b + r] : 0, sub, ia, ja, g, scale, in0, out);
    }
    __syncthreads();
  }
}

// Segments of the exact solves over the levels in levelPtr.
std::vector<FePrecond::TriSeg> triPlan(const std::vector<int> &levelPtr)
{
  std::vector<FePrecond::TriSeg> plan;
  const int nl = (int)levelPtr.size() - 1;
  int runStart = -1;
  for(int l = 0; l < nl; ++l) {
    const int cnt = levelPtr[l + 1] - levelPtr[l];
    if(cnt <= kTriSmall) {
      if(runStart < 0) runStart = l;
      continue;
    }
    if(runStart >= 0) plan.push_back({runStart, l, true});
    runStart = -1;
    plan.push_back({l, l + 1, false});
  }
  if(runStart >= 0) plan.push_back({runStart, nl, true});
  return plan;
}

__global__ void scaleVec(int n, const double *__restrict__ d, const double *__restrict__ x, double *__restrict__ y)
{
  for(int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) y[i] = d[i] * x[i];
}

__global__ void jacobiDiag(int n, const int *__restrict__ diag, const double *__restrict__ val,
                           double *__restrict__ dinv)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  const double d = diag[i] >= 0 ? val[diag[i]] : 0.;
  dinv[i] = d != 0. ? 1. / d : 1.;
}

constexpr int kGmAhead = 2;      // steps the host launches ahead of the last posted one
constexpr int kGmChunks = 128;   // row chunks of the dot products: partials per vector that every block folds
constexpr int kGmMaxVec = 128;   // vectors of one cycle (restart + 1 at most)
constexpr int kGmNorm = 512;     // blocks (norm partials) of the row kernels
constexpr size_t kGmKeep = (size_t)256 << 20;  // bytes of a workspace kept for the next solve

// Device state of a solve: rotations, the least-squares right-hand side, the
// last cycle's coefficients, norms.
struct GmState {
  double cs[kGmMaxVec], sn[kGmMaxVec], g[kGmMaxVec + 1], y[kGmMaxVec];
  double bn, target, res;
  int stopped;  // this cycle has stopped: its later steps post nothing
};
// What the host sees (pinned): posted step << 2 | code in one word, so a step
// and its code are never seen apart.  Codes: 0 go on, 1 the estimate of a
// step met the target (or the space is exhausted), 2 the true residual of a
// restart did, 3 diverged or not a number.
struct GmMailbox {
  unsigned long long word;
};
__device__ __forceinline__ void gmPost(GmMailbox *mb, unsigned long long step, int code)
{
  __hip_atomic_store(&mb->word, step << 2 | (unsigned long long)code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// part[c * KP + k] = sum over rows of chunk c of V_k w, k < nv; block
// (chunk, group of 8 vectors), two vectors per wavefront.
template <int KP>
__global__ __launch_bounds__(kTB) void gmDots(int n, int nv, int rows, const double *__restrict__ V, size_t ld,
                                              const double *__restrict__ w, double *__restrict__ part)
{
  const int lane = threadIdx.x & 63, k = blockIdx.y * 8 + (threadIdx.x >> 6) * 2;
  if(k >= nv) return;
  const bool two = k + 1 < nv;
  const double *v0 = V + (size_t)k * ld, *v1 = V + (size_t)(two ? k + 1 : k) * ld;
  const int r0 = blockIdx.x * rows, r1 = min(n, r0 + rows);
  double s0 = 0., s1 = 0.;
  constexpr int U = 8;
  int i = r0 + lane;
  for(; i + 64 * (U - 1) < r1; i += 64 * U) {
    double a[U], b[U], c[U];
#pragma unroll
    for(int u = 0; u < U; ++u) {
      a[u] = w[i + 64 * u];
      b[u] = v0[i + 64 * u];
      c[u] = v1[i + 64 * u];
    }
#pragma unroll
    for(int u = 0; u < U; ++u) {
      s0 += a[u] * b[u];
      s1 += a[u] * c[u];
    }
  }
  for(; i < r1; i += 64) {
    const double a = w[i];
    s0 += a * v0[i];
    s1 += a * v1[i];
  }
  s0 = feWaveSum(s0);
  s1 = feWaveSum(s1);
  if(lane == 0) {
    part[(size_t)blockIdx.x * KP + k] = s0;
    if(two) part[(size_t)blockIdx.x * KP + k + 1] = s1;
  }
}

// h = sum of the C chunk partials (the same order in every block);
// w -= sum_k h_k V_k; block partials of (w, w).  Block 0 stores the
// Hessenberg column (adds to it in a reorthogonalization).
template <int KP>
__global__ __launch_bounds__(kTB) void gmAxpy(int n, int nv, int C, const double *__restrict__ part,
                                              const double *__restrict__ V, size_t ld, double *__restrict__ w,
                                              double *__restrict__ hcol, int add, double *__restrict__ normPart)
{
  constexpr int NG = kTB / KP;
  __shared__ double hp[NG][KP], hs[KP];
  __shared__ double lds[kTB / 64 + 1];
  {
    const int k = threadIdx.x % KP, gq = threadIdx.x / KP;
    double s = 0.;
    if(k < nv) {
#pragma unroll 8
      for(int c = gq; c < C; c += NG) s += part[(size_t)c * KP + k];
    }
    hp[gq][k] = s;
    __syncthreads();
    if(gq == 0) {
      double t = 0.;
#pragma unroll
      for(int q = 0; q < NG; ++q) t += hp[q][k];
      hs[k] = t;
      if(blockIdx.x == 0 && k < nv) hcol[k] = add ? hcol[k] + t : t;
    }
    __syncthreads();
  }
  double nn = 0.;
  for(int i = blockIdx.x * kTB + threadIdx.x; i < n; i += gridDim.x * kTB) {
    double s = w[i];
    int k = 0;
    for(; k + 8 <= nv; k += 8) {
      double v[8];
#pragma unroll
      for(int u = 0; u < 8; ++u) v[u] = V[(size_t)(k + u) * ld + i];
#pragma unroll
      for(int u = 0; u < 8; ++u) s -= hs[k + u] * v[u];
    }
    for(; k < nv; ++k) s -= hs[k] * V[(size_t)k * ld + i];
    w[i] = s;
    nn += s * s;
  }
  feStoreBlockSum(nn, normPart, lds);
}

// Blocks >= 1: out = w / ||w|| (0 when w = 0), the norm folded from G
// partials.  Block 0: step j's Hessenberg column through the rotations, its
// own rotation, the residual estimate, the post.  H: column k at k (m + 1).
__global__ __launch_bounds__(kTB) void gmNext(int n, const double *__restrict__ w, const double *__restrict__ normPart,
                                              int G, double *__restrict__ out, int j, double *__restrict__ hcol,
                                              GmState *st, GmMailbox *mb, unsigned long long step)
{
  __shared__ double lds[kTB / 64 + 1];
  __shared__ double cs[kGmMaxVec], sn[kGmMaxVec], h[kGmMaxVec];
  const double wn = sqrt(feFoldPartials(normPart, G, lds));
  if(blockIdx.x > 0) {
    const double a = wn > 0. ? 1. / wn : 0.;
    for(int i = (blockIdx.x - 1) * kTB + threadIdx.x; i < n; i += (gridDim.x - 1) * kTB) out[i] = a * w[i];
    return;
  }
  for(int k = threadIdx.x; k <= j; k += kTB) {
    h[k] = hcol[k];
    if(k < j) {
      cs[k] = st->cs[k];
      sn[k] = st->sn[k];
    }
  }
  __syncthreads();
  if(threadIdx.x == 0) {
    double a = h[0];
#pragma unroll 4
    for(int k = 0; k < j; ++k) {
      const double b = h[k + 1];
      h[k] = cs[k] * a + sn[k] * b;
      a = -sn[k] * a + cs[k] * b;
    }
    const double rr = sqrt(a * a + wn * wn);
    const double c = rr > 0. ? a / rr : 1., s = rr > 0. ? wn / rr : 0.;
    h[j] = rr;
    st->cs[j] = c;
    st->sn[j] = s;
    const double g = st->g[j], gn = -s * g;
    st->g[j] = c * g;
    st->g[j + 1] = gn;
    if(!st->stopped) {
      const bool stop = fabs(gn) <= st->target || wn == 0.;
      if(stop) st->stopped = 1;
      gmPost(mb, step, stop ? 1 : 0);
    }
  }
  __syncthreads();
  for(int k = threadIdx.x; k <= j; k += kTB) hcol[k] = h[k];
}

// Start of a cycle from the residual r: V_0 = r / ||r||; block 0 tests the
// true residual (the first call also sets ||b|| and the target) and posts.
__global__ __launch_bounds__(kTB) void gmStart(int n, const double *__restrict__ r, const double *__restrict__ normPart,
                                               int G, double *__restrict__ out, int first, double rtol, double atol,
                                               double dtol, GmState *st, GmMailbox *mb, unsigned long long step)
{
  __shared__ double lds[kTB / 64 + 1];
  const double beta = sqrt(feFoldPartials(normPart, G, lds));
  if(blockIdx.x > 0) {
    const double a = 1. / beta;
    for(int i = (blockIdx.x - 1) * kTB + threadIdx.x; i < n; i += (gridDim.x - 1) * kTB) out[i] = a * r[i];
    return;
  }
  if(threadIdx.x == 0) {
    if(first) {
      st->bn = beta;
      st->target = fmax(rtol * beta, atol);
    }
    st->g[0] = beta;
    st->res = beta;
    int code = 0;
    if(beta <= st->target) code = 2;
    else if(!(beta == beta) || beta / st->bn > dtol) code = 3;
    st->stopped = code;  // steps launched past a stop post nothing
    gmPost(mb, step, code);
  }
}

// y = R^-1 g of a cycle of jn steps: back substitution by columns, the
// triangle in LDS (packed).
__global__ __launch_bounds__(kGmMaxVec) void gmSolveY(int jn, int ldh, const double *__restrict__ H, GmState *st)
{
  __shared__ double R[kGmMaxVec * (kGmMaxVec - 1) / 2];
  __shared__ double y[kGmMaxVec];
  const int t = threadIdx.x;
  for(int k = 0; k < jn; ++k)
    if(t <= k) R[k * (k + 1) / 2 + t] = H[(size_t)k * ldh + t];
  double g = t < jn ? st->g[t] : 0.;
  __syncthreads();
  for(int k = jn - 1; k >= 0; --k) {
    const double *Rk = R + k * (k + 1) / 2;
    if(t == k) y[k] = g / Rk[k];
    __syncthreads();
    if(t < k) g -= Rk[t] * y[k];
  }
  if(t < jn) st->y[t] = y[t];
}

// w = sum_k y_k V_k
__global__ __launch_bounds__(kTB) void gmCombine(int n, int nv, const double *__restrict__ V, size_t ld,
                                                 const GmState *st, double *__restrict__ w)
{
  __shared__ double ys[kGmMaxVec];
  for(int k = threadIdx.x; k < nv; k += kTB) ys[k] = st->y[k];
  __syncthreads();
  for(int i = blockIdx.x * kTB + threadIdx.x; i < n; i += gridDim.x * kTB) {
    double s = 0.;
    int k = 0;
    for(; k + 8 <= nv; k += 8) {
      double v[8];
#pragma unroll
      for(int u = 0; u < 8; ++u) v[u] = V[(size_t)(k + u) * ld + i];
#pragma unroll
      for(int u = 0; u < 8; ++u) s += ys[k + u] * v[u];
    }
    for(; k < nv; ++k) s += ys[k] * V[(size_t)k * ld + i];
    w[i] = s;
  }
}

__global__ void axpyKernel(int n, double a, const double *__restrict__ x, double *__restrict__ y)
{
  for(int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) y[i] += a * x[i];
}

// r = b - ax; block partials of (r, r).
__global__ __launch_bounds__(kTB) void gmResidual(int n, const double *__restrict__ b, const double *__restrict__ ax,
                                                  double *__restrict__ r, double *__restrict__ normPart)
{
  __shared__ double lds[kTB / 64 + 1];
  double s = 0.;
  for(int i = blockIdx.x * kTB + threadIdx.x; i < n; i += gridDim.x * kTB) {
    const double v = b[i] - ax[i];
    r[i] = v;
    s += v * v;
  }
  feStoreBlockSum(s, normPart, lds);
}

// Block maxima of |x|, |b|, |ax - b|: part[3 block + 0 .. 2].
__global__ __launch_bounds__(kTB) void gmMaxAbs(int n, const double *__restrict__ x, const double *__restrict__ b,
                                                const double *__restrict__ ax, double *__restrict__ part)
{
  __shared__ double red[3][kTB / 64];
  double m[3] = {0., 0., 0.};
  for(int i = blockIdx.x * kTB + threadIdx.x; i < n; i += gridDim.x * kTB) {
    m[0] = fmax(m[0], fabs(x[i]));
    m[1] = fmax(m[1], fabs(b[i]));
    m[2] = fmax(m[2], fabs(ax[i] - b[i]));
  }
#pragma unroll
  for(int q = 0; q < 3; ++q) {
#pragma unroll
    for(int o = 32; o > 0; o >>= 1) m[q] = fmax(m[q], __shfl_xor(m[q], o, 64));
    if((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = m[q];
  }
  __syncthreads();
  if(threadIdx.x < 3) {
    double v = 0.;
    for(int q = 0; q < kTB / 64; ++q) v = fmax(v, red[threadIdx.x][q]);
    part[3 * blockIdx.x + threadIdx.x] = v;
  }
}

struct Gm {
  fe_hip_ctx *ctx;
  int n, m;
  size_t ld;
  double *V, *w, *z, *t1, *t2, *x, *r, *dinvJ, *part, *normPart, *H;
  GmState *st;
  GmMailbox *mbHost, *mbDev;
  int pc;
  int sweeps;
  int C, rows;  // row chunks of the dot products
  int gRow;     // blocks of the row kernels

  void spmv(const double *x_, double *y_)
  {
    const int L = ctx->spmvLanes;
#define FE_SP(LL) hipLaunchKernelGGL(spmv64<LL>, dim3(kG), dim3(kTB), 0, ctx->stream, n, ctx->d_ia, ctx->d_ja, ctx->d_val, x_, y_)
    switch(L) {
      case 1: FE_SP(1); break;
      case 2: FE_SP(2); break;
      case 4: FE_SP(4); break;
      case 8: FE_SP(8); break;
      case 16: FE_SP(16); break;
      default: FE_SP(32); break;
    }
#undef FE_SP
  }

  // z = M^-1 v
  int precond(const double *v, double *out)
  {
    if(pc == FE_PC_JACOBI) {
      hipLaunchKernelGGL(scaleVec, dim3(kG), dim3(kTB), 0, ctx->stream, n, dinvJ, v, out);
      return FE_STATUS_OK;
    }
    if(pc == FE_PC_NONE) {
      FE_HIP_TRY(ctx, hipMemcpyAsync(out, v, sizeof(double) * n, hipMemcpyDeviceToDevice, ctx->stream));
      return FE_STATUS_OK;
    }
    if(pc == FE_PC_FIELDSPLIT) return feFieldSplitApply(ctx, v, out);
    FePrecond &P = ctx->pc;
    if(sweeps == 0 && feTriSolveUsable(ctx)) return feTriSolveApply(ctx, v, out);
    if(sweeps == 0) {
      // exact: y = L^-1 v (G_L = I - L_strict: y_i = v_i + sum_j<i g_ij y_j), then
      // z = U^-1 y (z_i = y_i / u_ii + sum_j>i g_ij z_j with g_ij = -u_ij / u_ii)
      if(P.triL.empty()) P.triL = triPlan(P.levelPtr);
      if(P.triU.empty()) P.triU = triPlan(P.levelPtrU);
      auto solve = [&](const std::vector<FePrecond::TriSeg> &plan, const std::vector<int> &lp, const int *dLp,
                       const int *rows, const int *tia, const int *tja, const double *tg, const double *scale,
                       const double *in0, double *o) {
        for(const FePrecond::TriSeg &sg : plan) {
          if(sg.run) {
            hipLaunchKernelGGL(triLevelRun, dim3(1), dim3(kTriRunTB), 0, ctx->stream, dLp, sg.l0, sg.l1, rows, tia,
                               tja, tg, scale, in0, o);
          } else {
            const int b = lp[sg.l0], cnt = lp[sg.l0 + 1] - b;
            hipLaunchKernelGGL(triLevel, dim3((cnt * kTriLPR + 255) / 256), dim3(256), 0, ctx->stream, rows + b, cnt,
                               tia, tja, tg, scale, in0, o);
          }
        }
      };
      solve(P.triL, P.levelPtr, P.d_levelPtr, P.d_levelRows, P.d_iaL, P.d_jaL, P.d_gL64, nullptr, v, t1);
      solve(P.triU, P.levelPtrU, P.d_levelPtrU, P.d_levelRowsU, P.d_iaU, P.d_jaU, P.d_gU64, P.d_dinv64, t1, out);
      return FE_STATUS_OK;
    }
    // L sweeps: y_{k+1} = v + G_L,strict y_k (G_L = -L_strict), y_0 = v
    const double *cur = v;
    double *bufs[2] = {t1, t2};
    int bi = 0;
    for(int s = 0; s < sweeps; ++s) {
      hipLaunchKernelGGL(factorSweep, dim3(kG), dim3(kTB), 0, ctx->stream, n, P.d_iaL, P.d_jaL, P.d_gL64,
                         (const double *)nullptr, v, cur, bufs[bi]);
      cur = bufs[bi];
      bi ^= 1;
    }
    // keep y in t_y (copy if it aliases the U-sweep buffers)
    const double *y = cur;
    // U sweeps: z_{k+1} = D^-1 y + G_U,strict z_k (G_U = -D^-1 U_strict), z_0 = D^-1 y
    double *zb[2] = {out, (y == t1) ? t2 : t1};
    hipLaunchKernelGGL(scaleVec, dim3(kG), dim3(kTB), 0, ctx->stream, n, P.d_dinv64, y, zb[0]);
    int zi = 0;
    for(int s = 0; s < sweeps; ++s) {
      hipLaunchKernelGGL(factorSweep, dim3(kG), dim3(kTB), 0, ctx->stream, n, P.d_iaU, P.d_jaU, P.d_gU64,
                         P.d_dinv64, y, zb[zi], zb[zi ^ 1]);
      zi ^= 1;
    }
    if(zb[zi] != out)
      FE_HIP_TRY(ctx, hipMemcpyAsync(out, zb[zi], sizeof(double) * n, hipMemcpyDeviceToDevice, ctx->stream));
    return FE_STATUS_OK;
  }

  // profiling: an event pair around a launch (timed: the A products of the
  // Arnoldi steps, the dominant kernel, and whole steps)
  int mark(FeKernelTimer &t)
  {
    if(t.used + 1 > t.ev.size())
      for(int q = 0; q < 64; ++q) {
        hipEvent_t e;
        FE_HIP_TRY(ctx, hipEventCreate(&e));
        t.ev.push_back(e);
      }
    FE_HIP_TRY(ctx, hipEventRecord(t.ev[t.used++], ctx->stream));
    return FE_STATUS_OK;
  }
  // complete pairs into the totals (the stream has been synchronized); an
  // open pair's first event moves to the front
  int collect(FeKernelTimer &t)
  {
    size_t q = 0;
    for(; q + 1 < t.used; q += 2) {
      float ms = 0.f;
      FE_HIP_TRY(ctx, hipEventElapsedTime(&ms, t.ev[q], t.ev[q + 1]));
      t.total_ms += ms;
      t.launches++;
    }
    if(q < t.used) std::swap(t.ev[0], t.ev[q]);
    t.used -= q;
    return FE_STATUS_OK;
  }

  // w -= V V^T w over nv vectors, the coefficients into hcol (added to it in
  // a reorthogonalization), the partials of (w, w)
  void project(int nv, double *hcol, int add)
  {
    const dim3 gd(C, (nv + 7) / 8);
    if(nv <= 64) {
      hipLaunchKernelGGL(gmDots<64>, gd, dim3(kTB), 0, ctx->stream, n, nv, rows, V, ld, w, part);
      hipLaunchKernelGGL(gmAxpy<64>, dim3(gRow), dim3(kTB), 0, ctx->stream, n, nv, C, part, V, ld, w, hcol, add,
                         normPart);
    } else {
      hipLaunchKernelGGL(gmDots<128>, gd, dim3(kTB), 0, ctx->stream, n, nv, rows, V, ld, w, part);
      hipLaunchKernelGGL(gmAxpy<128>, dim3(gRow), dim3(kTB), 0, ctx->stream, n, nv, C, part, V, ld, w, hcol, add,
                         normPart);
    }
  }

  // Waits until the device has posted `step` or a nonzero code; the stream
  // draining ends the wait too (nothing left to wait for).  Returns the word.
  unsigned long long waitFor(unsigned long long step)
  {
    volatile unsigned long long *word = &mbHost->word;
    unsigned long long v = *word;
    for(int spin = 1; (v >> 2) < step && !(v & 3); ++spin) {
      if((spin & 255) == 0 && hipStreamQuery(ctx->stream) != hipErrorNotReady) {
        v = *word;
        break;
      }
      v = *word;
    }
    return v;
  }
};

}  // namespace

// Workspace of the GMRES solves of a context, kept between them up to kGmKeep
// bytes (allocating 50 MB takes longer than a step; above, solves take tens of
// milliseconds and give (restart + 8) n values back).
struct FeGmres {
  double *work = nullptr;
  size_t count = 0;
  GmState *st = nullptr;
  GmMailbox *mbHost = nullptr, *mbDev = nullptr;
};

void feGmresRelease(fe_hip_ctx *ctx)
{
  if(ctx->gmres && ctx->gmres->mbHost) (void)hipHostFree(ctx->gmres->mbHost);
  delete ctx->gmres;  // device buffers are owned by the context
  ctx->gmres = nullptr;
}

int feSolveGmres(fe_hip_ctx *ctx, const fe_hip_solver_opts *o, double *du, fe_hip_solve_stats *stats)
{
  FE_REQUIRE(ctx, o->precision == FE_PREC_FP64, "GMRES runs in FP64");
  FE_REQUIRE(ctx,
             o->pc == FE_PC_NONE || o->pc == FE_PC_JACOBI || o->pc == FE_PC_ILU0 || o->pc == FE_PC_BJ_ILU0 ||
                 o->pc == FE_PC_FIELDSPLIT,
             "GMRES takes the NONE, JACOBI, ILU0 or FIELDSPLIT preconditioner");
  const int n = ctx->n;
  const int m = std::max(2, std::min(o->restart, 120));
  Gm g;
  g.ctx = ctx;
  g.n = n;
  g.m = m;
  g.ld = ((size_t)n + 63) & ~(size_t)63;
  g.pc = (o->pc == FE_PC_BJ_ILU0) ? FE_PC_ILU0 : o->pc;
  g.sweeps = std::max(0, ctx->pc.sweeps);
  // dot products: chunks of at least 512 rows, at most kGmChunks of them
  g.C = std::max(1, std::min(kGmChunks, n / 512));
  g.rows = (n + g.C - 1) / g.C;
  g.gRow = std::max(1, std::min(kGmNorm, (n + kTB - 1) / kTB));
  const int ldh = m + 1;
  const size_t need = g.ld * (m + 1) + 7 * g.ld + (size_t)kGmChunks * kGmMaxVec + 3 * kGmNorm + (size_t)ldh * m;
  if(!ctx->gmres) ctx->gmres = new FeGmres();
  FeGmres &W = *ctx->gmres;
  if(W.count < need) {
    if(W.work) feFree(ctx, W.work);
    W.work = nullptr;
    W.count = 0;
    if(feAlloc(ctx, &W.work, need)) return FE_STATUS_OUT_OF_MEMORY;
    W.count = need;
  }
  if(!W.st && feAlloc(ctx, &W.st, 1)) return FE_STATUS_OUT_OF_MEMORY;
  if(!W.mbHost) {
    FE_HIP_TRY(ctx, hipHostMalloc((void **)&W.mbHost, sizeof(GmMailbox), hipHostMallocMapped | hipHostMallocCoherent));
    FE_HIP_TRY(ctx, hipHostGetDevicePointer((void **)&W.mbDev, W.mbHost, 0));
  }
  g.V = W.work;
  g.w = g.V + g.ld * (m + 1);
  g.z = g.w + g.ld;
  g.t1 = g.z + g.ld;
  g.t2 = g.t1 + g.ld;
  g.x = g.t2 + g.ld;
  g.r = g.x + g.ld;
  g.dinvJ = g.r + g.ld;
  g.part = g.dinvJ + g.ld;
  g.normPart = g.part + (size_t)kGmChunks * kGmMaxVec;
  g.H = g.normPart + 3 * kGmNorm;
  g.st = W.st;
  g.mbHost = W.mbHost;
  g.mbDev = W.mbDev;
  *(volatile unsigned long long *)&W.mbHost->word = 0;  // no kernel of this context is running: the stream is idle

  hipEvent_t ev[3];
  for(hipEvent_t &e : ev) FE_HIP_TRY(ctx, hipEventCreate(&e));
  FE_HIP_TRY(ctx, hipEventRecord(ev[0], ctx->stream));
  ctx->spmvTimer = FeKernelTimer{std::move(ctx->spmvTimer.ev)};
  ctx->iterTimer = FeKernelTimer{std::move(ctx->iterTimer.ev)};
  if(g.pc == FE_PC_ILU0) {
    if(int rc = fePrecondFactor(ctx)) return rc;
    if(g.sweeps == 0) {
      if(int rc = feTriSolveBuild(ctx)) return rc;
      if(feTriSolveUsable(ctx))
        if(int rc = feTriSolvePack(ctx)) return rc;
    }
  } else if(g.pc == FE_PC_FIELDSPLIT) {
    if(int rc = feFieldSplitSetup(ctx)) return rc;
  } else if(g.pc == FE_PC_JACOBI) {
    hipLaunchKernelGGL(jacobiDiag, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, ctx->d_diag, ctx->d_val, g.dinvJ);
  }
  FE_HIP_TRY(ctx, hipEventRecord(ev[1], ctx->stream));

  // Level-scheduled exact solves (hundreds of launches) hide the host's round
  // trip by themselves, and a step launched past a stop costs another
  // application: cycles of one or two steps, as at the FP64 floor of a system
  // (P4 triangles, n = 16,129), took 12 ms a step with kGmAhead, 8 with one.
  const unsigned long long ahead = g.pc == FE_PC_ILU0 && g.sweeps == 0 && !feTriSolveUsable(ctx) ? 1 : kGmAhead;
  const int gNext = 1 + std::min(kG, (n + kTB - 1) / kTB);
  int iters = 0, outer = 0, converged = 0, reason = 0;
  unsigned long long step = 0;  // posted steps: one per cycle start and per Arnoldi step
  bool expectStop = false;
  FE_HIP_TRY(ctx, hipMemsetAsync(g.x, 0, sizeof(double) * n, ctx->stream));
  for(;;) {
    // r = b - A x, V_0 = r / ||r||, the test of the true residual
    g.spmv(g.x, g.w);
    hipLaunchKernelGGL(gmResidual, dim3(g.gRow), dim3(kTB), 0, ctx->stream, n, ctx->d_rhs, g.w, g.r, g.normPart);
    hipLaunchKernelGGL(gmStart, dim3(gNext), dim3(kTB), 0, ctx->stream, n, g.r, g.normPart, g.gRow, g.V,
                       outer == 0 ? 1 : 0, o->rtol, o->atol, o->dtol, g.st, g.mbDev, ++step);
    FE_HIP_TRY(ctx, hipGetLastError());
    // a cycle after a met estimate, or past the budget, usually does not run:
    // its start is waited for instead of launched past
    const bool last = iters >= o->max_iter;
    unsigned long long word = 0;
    if(expectStop || last) word = g.waitFor(step);
    const unsigned long long base = step;
    int j = 0, jn = 0;
    for(; !(word & 3) && !last && j < m && iters + j < o->max_iter; ++j) {
      if(step >= ahead) {
        word = g.waitFor(step - ahead + 1);
        if(word & 3) break;
      }
      double *vj = g.V + g.ld * j, *hcol = g.H + (size_t)j * ldh;
      if(ctx->profiling)
        if(int rc = g.mark(ctx->iterTimer)) return rc;
      if(int rc = g.precond(vj, g.z)) return rc;
      // profiling: events around the A product (the dominant kernel of the
      // Arnoldi steps), read at the end of the solve
      if(ctx->profiling)
        if(int rc = g.mark(ctx->spmvTimer)) return rc;
      g.spmv(g.z, g.w);
      if(ctx->profiling)
        if(int rc = g.mark(ctx->spmvTimer)) return rc;
      g.project(j + 1, hcol, 0);
      if(ctx->gmresOrth == 2) g.project(j + 1, hcol, 1);
      hipLaunchKernelGGL(gmNext, dim3(gNext), dim3(kTB), 0, ctx->stream, n, g.w, g.normPart, g.gRow, vj + g.ld, j, hcol,
                         g.st, g.mbDev, ++step);
      if(ctx->profiling)
        if(int rc = g.mark(ctx->iterTimer)) return rc;
      FE_HIP_TRY(ctx, hipGetLastError());
    }
    // every launched step's code decides how many columns the cycle keeps
    word = g.waitFor(step);
    const int code = (int)(word & 3);
    if(code == 0 && (word >> 2) < step) {  // the stream drained without the post: a failed launch
      FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
      FE_REQUIRE(ctx, (*(volatile unsigned long long *)&g.mbHost->word >> 2) >= step, "GMRES: a step did not post");
    }
    if(!last) outer++;
    if(code >= 2) {  // at the cycle's start
      converged = code == 2;
      reason = code == 2 ? 2 : last ? -3 : -4;
      break;
    }
    if(last) {
      reason = -3;
      break;
    }
    jn = code == 1 ? (int)((word >> 2) - base) : j;
    expectStop = code == 1;
    iters += jn;
    // y = R^-1 g, x += M^-1 (V y)
    hipLaunchKernelGGL(gmSolveY, dim3(1), dim3(kGmMaxVec), 0, ctx->stream, jn, ldh, g.H, g.st);
    hipLaunchKernelGGL(gmCombine, dim3(std::min(kG, (n + kTB - 1) / kTB)), dim3(kTB), 0, ctx->stream, n, jn, g.V, g.ld,
                       g.st, g.w);
    if(int rc = g.precond(g.w, g.z)) return rc;
    hipLaunchKernelGGL(axpyKernel, dim3(kG), dim3(kTB), 0, ctx->stream, n, 1., g.z, g.x);
    FE_HIP_TRY(ctx, hipGetLastError());
    *(volatile unsigned long long *)&g.mbHost->word = step << 2;  // the device posts nothing until the next start
  }
  FE_HIP_TRY(ctx, hipMemcpyAsync(ctx->d_du, g.x, sizeof(double) * n, hipMemcpyDeviceToDevice, ctx->stream));
  FE_HIP_TRY(ctx, hipEventRecord(ev[2], ctx->stream));
  if(stats) {
    // infinity norms: du, b, A du - b
    g.spmv(g.x, g.w);
    hipLaunchKernelGGL(gmMaxAbs, dim3(g.gRow), dim3(kTB), 0, ctx->stream, n, g.x, ctx->d_rhs, g.w, g.normPart);
  }
  std::vector<double> mx(3 * g.gRow), tail(3);
  static_assert(offsetof(GmState, res) == offsetof(GmState, bn) + 2 * sizeof(double), "bn, target, res together");
  FE_HIP_TRY(ctx, hipMemcpyAsync(mx.data(), g.normPart, sizeof(double) * mx.size(), hipMemcpyDeviceToHost, ctx->stream));
  FE_HIP_TRY(ctx, hipMemcpyAsync(tail.data(), &g.st->bn, 3 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  float ms = 0.f, setupMs = 0.f;
  FE_HIP_TRY(ctx, hipEventElapsedTime(&ms, ev[0], ev[2]));
  FE_HIP_TRY(ctx, hipEventElapsedTime(&setupMs, ev[0], ev[1]));
  for(hipEvent_t &e : ev) (void)hipEventDestroy(e);
  if(ctx->profiling) {
    if(int rc = g.collect(ctx->spmvTimer)) return rc;
    if(int rc = g.collect(ctx->iterTimer)) return rc;
    ctx->spmvTimer.used = ctx->iterTimer.used = 0;
  }
  if(stats) {
    memset(stats, 0, sizeof(*stats));
    double mv[3] = {0., 0., 0.};
    for(size_t q = 0; q < mx.size(); ++q) mv[q % 3] = std::max(mv[q % 3], mx[q]);
    stats->iterations = iters;
    stats->outer_iterations = tail[0] == 0. ? 0 : outer;  // no cycle for a zero right-hand side
    stats->converged = converged;
    stats->reason = reason;
    stats->relres_fp64 = tail[0] > 0. ? tail[2] / tail[0] : 0.;
    stats->norm_dx_inf = mv[0];
    stats->norm_rhs_inf = mv[1];
    stats->norm_axb_inf = mv[2];
    stats->ms_solve = ms;
    stats->ms_setup = setupMs;
  }
  if(du) FE_HIP_TRY(ctx, hipMemcpy(du, g.x, sizeof(double) * n, hipMemcpyDeviceToHost));
  if(W.count * sizeof(double) > kGmKeep) {  // the stream is idle
    feFree(ctx, W.work);
    W.work = nullptr;
    W.count = 0;
  }
  return FE_STATUS_OK;
}
