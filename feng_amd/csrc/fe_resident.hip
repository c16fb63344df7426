// Jacobi-PCG with all iterations in one launch (the KSPCG / PCJACOBI of the
// reference's options, feLinearSystemPETSc.cpp:900-1031): the pipelined
// recurrences of fe_krylov.hip's tileIter (Ghysels & Vanroose 2014), with the
// matrix in registers.
//
// What bounded the launch-per-iteration form below some 10^5 unknowns was not
// the matrix but the chain inside a launch -- dispatch, row bounds, columns
// and values, gather, reduction, each a trip to memory that the previous
// launch's end had emptied the caches for: 9.2 us for the 27 k entries of a
// 64 x 64 Poisson problem, 14.5 us at 48^3 tetrahedra.  Here a workgroup of
// up to 1024 threads owns a range of rows, one thread a row: its entries (FP64
// values, 16-bit positions), x, r, w, s, z, p and 1 / a_ii stay in registers
// for the whole solve, the gathered vector m lives in LDS with the values of
// other workgroups' rows behind the own ones, and an iteration is one
// exchange (fe_resident.h) of m and the three partial sums plus two
// workgroup barriers; the start, the check of the true residual and a restart
// are exchanges of the same loop, so a solve is one launch and one
// synchronization.  An iteration, launch-per-iteration -> here: 64^2 P1
// triangles (n = 3,969) 11.2 -> 3.0 us, 500^2 (249,001) 18.7 -> 5.9 us, 100^2
// P2 16.2 -> 4.5 us, tetrahedra at 16^3 14.1 -> 3.1, 32^3 15.2 -> 4.0, 48^3
// 16.9 -> 5.5, 64^3 24.0 -> 6.2 us.  What is left is the trip of a stored word
// to another workgroup's poll (about 1.5 us), the LDS gathers and the barriers.
//
// The rule (resUsable): one row a thread on the CUs of the device (n <= 1024 x
// CUs, 262,144 on 256), rows of at most 24 entries (48 + 12 registers), and
// the rows of other workgroups that one gathers have to fit the LDS.  Larger
// systems are bound by the matrix traffic, which the tiled kernels stream.
#include "fe_resident.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

using namespace fe_res;

// What a solve returns to the host, and per workgroup the largest |x|, |b|,
// |b - A x| of its rows behind it.
struct ResOut {
  int reason, iters, outer, gaveUp;
  double bn, rn;
};

struct FeResident {
  bool built = false, usable = false;
  int G = 0, RW = 0, TB = 0, E = 0, H = 0;  // workgroups, rows and threads of one, entries a row, gathered rows at most
  unsigned *d_idx = nullptr;      // per workgroup E / 2 x TB packed pairs of LDS positions
  int *d_hcol = nullptr, *d_hcnt = nullptr;
  unsigned long long *d_buf = nullptr;  // kResBufs x (n values, 3 G partial sums)
  ResOut *d_out = nullptr, *h_out = nullptr;  // h_out: pinned copy
};

namespace {

constexpr int kResH = 8192;       // gathered rows of other workgroups at most
constexpr int kResLds = 150 * 1024;
constexpr int kResRows = 512;     // rows a workgroup below the full device: 2.85 us an iteration at 3,969 unknowns
                                  // (256 rows 2.99, 1024 rows 3.13), 3.79 at 32^3 tetrahedra (4.09, 4.09)

struct ResArgs {
  int n, G, RW, H, hcap;
  const int *ia, *ja;
  const double *val;
  const unsigned *idx;
  const int *hcol, *hcnt;
  const double *b;
  double *x;
  unsigned long long *buf;
  ResOut *out;
  double *maxima;
  double rtol, atol, dtol;
  int maxit;
};

// LDS positions of a workgroup's entries: own rows first, then the other
// columns its rows touch, in increasing order (a bitmap over all columns and
// its prefix sums).  flag[0] = the most such columns, flag[1] = the longest row.
__global__ __launch_bounds__(1024) void resPattern(int n, int RW, int E, int TB, int hcap, const int *__restrict__ ia,
                                                   const int *__restrict__ ja, unsigned short *__restrict__ idx,
                                                   int *__restrict__ hcol, int *__restrict__ hcnt, int *flag)
{
  __shared__ unsigned bits[8192];
  __shared__ int base[8192];
  __shared__ int sums[1024];
  const int wg = blockIdx.x, t = threadIdx.x;
  const int r0 = wg * RW, r1 = min(n, r0 + RW), nw = (n + 31) / 32;
  for(int q = t; q < nw; q += 1024) bits[q] = 0u;
  __syncthreads();
  const int k0 = ia[r0], k1 = ia[r1];
  for(int k = k0 + t; k < k1; k += 1024) {
    const int j = ja[k];
    if(j < r0 || j >= r1) atomicOr(&bits[j >> 5], 1u << (j & 31));
  }
  __syncthreads();
  const int per = (nw + 1023) / 1024, q0 = min(nw, t * per), q1 = min(nw, q0 + per);
  int s = 0;
  for(int q = q0; q < q1; ++q) s += __popc(bits[q]);
  sums[t] = s;
  __syncthreads();
  for(int o = 1; o < 1024; o <<= 1) {
    const int v = t >= o ? sums[t - o] : 0;
    __syncthreads();
    sums[t] += v;
    __syncthreads();
  }
  int c = sums[t] - s;
  for(int q = q0; q < q1; ++q) {
    base[q] = c;
    unsigned b = bits[q];
    while(b) {
      const int u = __ffs(b) - 1;
      if(c < hcap) hcol[(size_t)wg * hcap + c] = 32 * q + u;
      ++c;
      b &= b - 1;
    }
  }
  __syncthreads();
  if(t == 0) {
    hcnt[wg] = sums[1023];
    atomicMax(&flag[0], sums[1023]);
  }
  const int row = r0 + t;
  if(t < TB) {
    int kb = 0, len = 0;
    if(row < r1) {
      kb = ia[row];
      len = ia[row + 1] - kb;
      if(len > E) atomicMax(&flag[1], len);
    }
    for(int e = 0; e < E; ++e) {
      int p = min(t, RW - 1);  // no entry: value 0 at the own row
      if(e < len) {
        const int j = ja[kb + e];
        p = j >= r0 && j < r1 ? j - r0 : RW + base[j >> 5] + __popc(bits[j >> 5] & ((1u << (j & 31)) - 1u));
      }
      idx[(((size_t)wg * (E / 2) + e / 2) * TB + t) * 2 + (e & 1)] = (unsigned short)min(p, 65535);
    }
  }
}

__global__ void resLongest(int n, const int *__restrict__ ia, int *flag)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int len = i < n ? ia[i + 1] - ia[i] : 0;
#pragma unroll
  for(int o = 32; o > 0; o >>= 1) len = max(len, __shfl_xor(len, o, 64));
  if((threadIdx.x & 63) == 0) atomicMax(flag, len);
}

__global__ void resFill(size_t count, unsigned long long *__restrict__ buf, ResOut *out)
{
  for(size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
    buf[i] = kSentinel;
  if(blockIdx.x == 0 && threadIdx.x == 0) *out = ResOut{0, 0, 0, 0, 0., 0.};
}

// What the values gathered by an exchange are, and its partial sums: the
// start of a recurrence (D^-1 r; (r, r)), an iteration (m = D^-1 w; gamma,
// delta, rho), the check of the true residual (x; none).
enum { kResStart, kResIterate, kResCheck };

template <int TB, int E>
__global__ __launch_bounds__(TB) void resJacobi(ResArgs a)
{
  // slots a thread polls in one go: the partial sums by all, or by the first
  // wavefronts alone when the others cover the gathered values
  constexpr bool kSplit = TB == 512;
  constexpr int kSums = kSplit ? 0 : 3, kHeld = kSplit ? 6 : 3, kPoll = kSums + kHeld;
  extern __shared__ double lds[];           // two regions of own + gathered values
  __shared__ double wsum[3][16], psum[3][TB / 64];
  __shared__ int gaveUp;
  const int wg = blockIdx.x, t = threadIdx.x, G = a.G, RW = a.RW, stride = RW + a.H;
  const int row = wg * RW + t;
  const bool own = t < RW && row < a.n;
  const size_t bufLen = (size_t)a.n + 3 * (size_t)G;
  const int hc = a.hcnt[wg];
  const int *hcol = a.hcol + (size_t)wg * a.hcap;
  const int sumThreads = (G + 63) & ~63, h0 = kSplit ? t - sumThreads : t, hStep = kSplit ? TB - sumThreads : TB;
  if(t == 0) gaveUp = 0;
  // entries, 1 / a_ii, vectors
  double v[E];
  unsigned ix[E / 2];
  double d = 1., x = 0., r = 0., w = 0., s = 0., z = 0., p = 0.;
#pragma unroll
  for(int e = 0; e < E / 2; ++e) ix[e] = a.idx[((size_t)wg * (E / 2) + e) * TB + t];
  {
    int kb = 0, len = 0;
    if(own) {
      kb = a.ia[row];
      len = a.ia[row + 1] - kb;
      r = a.b[row];
    }
    double dg = 0.;
#pragma unroll
    for(int e = 0; e < E; ++e) {
      v[e] = 0.;
      if(e < len) {
        v[e] = a.val[kb + e];
        if(a.ja[kb + e] == row) dg = v[e];
      }
    }
    if(own) d = dg != 0. ? 1. / dg : 1.;
  }
  int hcl[kHeld];
#pragma unroll
  for(int q = 0; q < kHeld; ++q) hcl[q] = h0 >= 0 && h0 + q * hStep < hc ? hcol[h0 + q * hStep] : -1;
  // the value others gather and the partial sums of the next exchange
  double m = d * r, p0 = r * r, p1 = 0., p2 = 0.;
  // uniform state (every workgroup folds the same sums in the same order)
  double alphaP = __builtin_inf(), gammaP = 1., bn = 0., rn = 0., target = 0., tol2 = 0.;
  int phase = kResStart, code = 0, it = 0, outer = 0, breakdowns = 0, reason = 0;
  resBarrier();
  for(int q = 0;; ++q) {
    unsigned long long *buf = a.buf + (q & 3) * bufLen;
    double *reg = lds + (q & 1) * stride;
    // publish: own values, then the workgroup's sums
    resStoresDone();  // the resets of the previous exchange
    if(own) resStore(buf + row, m);
    if(t < RW) reg[t] = m;
    p0 = resWaveSum(own ? p0 : 0.);
    p1 = resWaveSum(own ? p1 : 0.);
    p2 = resWaveSum(own ? p2 : 0.);
    if((t & 63) == 0) {
      psum[0][t >> 6] = p0;
      psum[1][t >> 6] = p1;
      psum[2][t >> 6] = p2;
    }
    resBarrier();
    if(t < 3) {
      double sum = 0.;
#pragma unroll
      for(int k = 0; k < TB / 64; ++k) sum += psum[t][k];
      resStore(buf + a.n + t * G + wg, sum);
    }
    // collect the others'
    double f0 = 0., f1 = 0., f2 = 0.;
    {
      unsigned long long pv[kPoll];
      int at[kPoll];
#pragma unroll
      for(int k = 0; k < kHeld; ++k) at[kSums + k] = hcl[k];
#pragma unroll
      for(int k = 0; k < 3; ++k)
        if(!kSplit || t < sumThreads) at[k] = t < G ? a.n + k * G + t : -1;
      bool ok = resPoll<kPoll>(buf, at, pv);
#pragma unroll
      for(int k = 0; k < kHeld; ++k)
        if(hcl[k] >= 0) reg[RW + h0 + k * hStep] = __longlong_as_double((long long)pv[kSums + k]);
      for(int h = h0 + kHeld * hStep; h0 >= 0 && h < hc && ok; h += hStep) {
        const int a1[1] = {hcol[h]};
        unsigned long long v1[1];
        ok = resPoll<1>(buf, a1, v1);
        reg[RW + h] = __longlong_as_double((long long)v1[0]);
      }
      if(t < G) {
        f0 = __longlong_as_double((long long)pv[0]);
        f1 = __longlong_as_double((long long)pv[1]);
        f2 = __longlong_as_double((long long)pv[2]);
      }
      if(!ok) gaveUp = 1;
    }
    if(t < sumThreads) {
      f0 = resWaveSum(f0);
      f1 = resWaveSum(f1);
      f2 = resWaveSum(f2);
      if((t & 63) == 0) {
        wsum[0][t >> 6] = f0;
        wsum[1][t >> 6] = f1;
        wsum[2][t >> 6] = f2;
      }
    }
    resBarrier();
    if(gaveUp) break;
    double gamma = 0., delta = 0., rho = 0.;
    for(int k = 0; k < (G + 63) / 64; ++k) {
      gamma += wsum[0][k];
      delta += wsum[1][k];
      rho += wsum[2][k];
    }
    gamma = resUniform(gamma);
    delta = resUniform(delta);
    rho = resUniform(rho);
    {  // the slots of exchange q + 2 are empty again
      unsigned long long *rs = a.buf + ((q + 2) & 3) * bufLen;
      if(own) resStore(rs + row, kSentinel);
      if(t < 3) resStore(rs + a.n + t * G + wg, kSentinel);
    }
    double alpha = 0., beta = 0.;
    if(phase == kResIterate) {
      if(!(rho > tol2) || it >= a.maxit) {
        code = rho <= tol2 ? 1 : (rho == rho ? 2 : 4);
      } else {
        beta = resUniform(gamma / gammaP);
        const double den = delta - beta * gamma / alphaP;
        if(den > 0.) {
          alpha = resUniform(gamma / den);
          gammaP = gamma;
          alphaP = alpha;
          ++it;
        } else {
          code = 3;  // breakdown: the preconditioned operator is not SPD
        }
      }
      if(code) {  // gather x for the true residual
        phase = kResCheck;
        m = x;
        p0 = p1 = p2 = 0.;
        continue;
      }
    }
    if(phase == kResStart) {
      rn = resUniform(sqrt(gamma));  // ||b||, or the true residual's norm
      if(outer == 0) {
        bn = rn;
        target = resUniform(fmax(a.rtol * bn, a.atol));
        tol2 = resUniform(target * target * 0.25);
        if(bn == 0.) {
          reason = 2;
          break;
        }
      } else {
        if(rn <= target) reason = 2;
        else if(code == 4 || !(rn == rn)) reason = -9;
        else if(it >= a.maxit) reason = -3;
        else if(rn / bn > a.dtol) reason = -4;
        else if(code == 3 && ++breakdowns > 20) reason = -3;
        if(reason) break;
        // again from the true residual: after a breakdown, or when the
        // recursive residual met a target the true one has not (aim lower)
        if(code != 3) tol2 = resUniform(0.01 * tol2);
        code = 0;
      }
      s = z = p = 0.;
      gammaP = 1.;
      alphaP = __builtin_inf();
    }
    double y = 0.;
#pragma unroll
    for(int e = 0; e < E / 2; ++e) {
      asm volatile("" : "+v"(ix[e]));  // unpacked here, not kept unpacked across the loop
      y += v[2 * e] * reg[ix[e] & 0xffffu];
      y += v[2 * e + 1] * reg[ix[e] >> 16];
    }
    if(phase == kResCheck) {
      r = own ? a.b[row] - y : 0.;
      m = d * r;
      p0 = r * r;
      ++outer;
      phase = kResStart;
      continue;
    }
    if(phase == kResStart) {
      w = y;
      phase = kResIterate;
      if(outer == 0) x = 0.;
    } else {
      z = y + beta * z;
      s = w + beta * s;
      p = d * r + beta * p;
      x = x + alpha * p;
      r = r - alpha * s;
      w = w - alpha * z;
    }
    m = d * w;
    const double u = d * r;
    p0 = r * u;
    p1 = w * u;
    p2 = r * r;
  }
  if(t == 0) {
    if(gaveUp) __hip_atomic_store(&a.out->gaveUp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if(wg == 0) {
      a.out->reason = reason;
      a.out->iters = it;
      a.out->outer = outer;
      a.out->bn = bn;
      a.out->rn = rn;
    }
  }
  if(own) a.x[row] = x;
  // the workgroup's largest |x|, |b|, |b - A x|
  double mx[3] = {own ? fabs(x) : 0., own ? fabs(a.b[row]) : 0., own ? fabs(r) : 0.};
#pragma unroll
  for(int k = 0; k < 3; ++k) {
#pragma unroll
    for(int o = 32; o > 0; o >>= 1) mx[k] = fmax(mx[k], __shfl_xor(mx[k], o, 64));
    if((t & 63) == 0) psum[k][t >> 6] = mx[k];
  }
  resBarrier();
  if(t < 3) {
    double mm = 0.;
    for(int k = 0; k < TB / 64; ++k) mm = fmax(mm, psum[t][k]);
    a.maxima[3 * wg + t] = mm;
  }
}

template <int TB, int E>
int launchRes(fe_hip_ctx *ctx, FeResident &R, const ResArgs &a, size_t lds, bool *fits)
{
  const void *f = (const void *)resJacobi<TB, E>;
  int perCu = 0, cus = 0;
  *fits = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess &&
          hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, f, TB, lds) == hipSuccess &&
          hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) == hipSuccess &&
          perCu * cus >= R.G;
  if(!*fits) {
    (void)hipGetLastError();
    return FE_STATUS_OK;
  }
  hipLaunchKernelGGL((resJacobi<TB, E>), dim3(R.G), dim3(TB), lds, ctx->stream, a);
  FE_HIP_TRY(ctx, hipGetLastError());
  return FE_STATUS_OK;
}

template <int TB>
int launchResE(fe_hip_ctx *ctx, FeResident &R, const ResArgs &a, size_t lds, bool *fits)
{
  if(R.E == 8) return launchRes<TB, 8>(ctx, R, a, lds, fits);
  if(R.E == 16) return launchRes<TB, 16>(ctx, R, a, lds, fits);
  return launchRes<TB, 24>(ctx, R, a, lds, fits);
}

int resBuild(fe_hip_ctx *ctx, FeResident &R)
{
  R.built = true;
  const int n = ctx->n;
  int cus = 0;
  FE_HIP_TRY(ctx, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
  cus = std::min(cus, 256);  // one thread per workgroup's partial sums
  if(n < 1 || n > cus * 1024) return FE_STATUS_OK;
  R.G = std::min(cus, (n + kResRows - 1) / kResRows);
  R.RW = (n + R.G - 1) / R.G;
  R.G = (n + R.RW - 1) / R.RW;
  R.TB = R.RW <= 512 ? 512 : 1024;
  int *flag = nullptr;
  if(feAlloc(ctx, &flag, 2)) return FE_STATUS_OUT_OF_MEMORY;
  int hf[2] = {0, 0};
  FE_HIP_TRY(ctx, hipMemsetAsync(flag, 0, 2 * sizeof(int), ctx->stream));
  hipLaunchKernelGGL(resLongest, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, ctx->d_ia, flag + 1);
  FE_HIP_TRY(ctx, hipMemcpyAsync(hf, flag, sizeof(hf), hipMemcpyDeviceToHost, ctx->stream));
  FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  R.E = hf[1] <= 8 ? 8 : hf[1] <= 16 ? 16 : 24;
  if(hf[1] > 24) {
    feFree(ctx, flag);
    return FE_STATUS_OK;
  }
  const int hcap = std::min(kResH, kResLds / 16 - R.RW);
  if(feAlloc(ctx, &R.d_idx, (size_t)R.G * (R.E / 2) * R.TB) || feAlloc(ctx, &R.d_hcol, (size_t)R.G * hcap) ||
     feAlloc(ctx, &R.d_hcnt, R.G) || feAlloc(ctx, &R.d_buf, kResBufs * ((size_t)n + 3 * (size_t)R.G)) ||
     feAlloc(ctx, (char **)&R.d_out, sizeof(ResOut) + 3 * sizeof(double) * R.G))
    return FE_STATUS_OUT_OF_MEMORY;
  FE_HIP_TRY(ctx, hipHostMalloc((void **)&R.h_out, sizeof(ResOut) + 3 * sizeof(double) * R.G));
  hipLaunchKernelGGL(resPattern, dim3(R.G), dim3(1024), 0, ctx->stream, n, R.RW, R.E, R.TB, hcap, ctx->d_ia, ctx->d_ja,
                     (unsigned short *)R.d_idx, R.d_hcol, R.d_hcnt, flag);
  FE_HIP_TRY(ctx, hipGetLastError());
  FE_HIP_TRY(ctx, hipMemcpyAsync(hf, flag, sizeof(hf), hipMemcpyDeviceToHost, ctx->stream));
  FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  feFree(ctx, flag);
  R.H = hf[0];
  R.usable = R.H <= hcap;
  return FE_STATUS_OK;
}

}  // namespace

std::mutex &feResidentMutex(int device)
{
  static std::mutex m[64];
  return m[device & 63];
}

int feResidentJacobi(fe_hip_ctx *ctx, const fe_hip_solver_opts *o, double *x, FeResidentResult *res)
{
  res->ran = false;
  if(!ctx->resident || ctx->residentGaveUp) return FE_STATUS_OK;
  if(!ctx->res) ctx->res = new FeResident();
  FeResident &R = *ctx->res;
  if(!R.built)
    if(int rc = resBuild(ctx, R)) return rc;
  if(!R.usable) return FE_STATUS_OK;
  const int hcap = std::min(kResH, kResLds / 16 - R.RW);
  const ResArgs a{ctx->n,     R.G,     R.RW, R.H,     hcap,    ctx->d_ia, ctx->d_ja,       ctx->d_val, R.d_idx, R.d_hcol,
                  R.d_hcnt,   ctx->d_rhs, x, R.d_buf, R.d_out, (double *)(R.d_out + 1), o->rtol, o->atol, o->dtol, o->max_iter};
  const size_t lds = 2 * (size_t)(R.RW + R.H) * sizeof(double);
  const size_t cells = kResBufs * ((size_t)ctx->n + 3 * (size_t)R.G);
  bool fits = false;
  {
    std::lock_guard<std::mutex> lock(feResidentMutex(ctx->device));
    if(ctx->profiling)
      if(int rc = feTimerMark(ctx, ctx->spmvTimer)) return rc;
    hipLaunchKernelGGL(resFill, dim3((unsigned)std::min<size_t>(1024, (cells + 255) / 256)), dim3(256), 0, ctx->stream,
                       cells, R.d_buf, R.d_out);
    int rc = FE_STATUS_OK;
    if(R.TB == 512) rc = launchResE<512>(ctx, R, a, lds, &fits);
    else rc = launchResE<1024>(ctx, R, a, lds, &fits);
    if(rc) return rc;
    if(fits) {
      if(ctx->profiling)
        if(int rc2 = feTimerMark(ctx, ctx->spmvTimer)) return rc2;
      FE_HIP_TRY(ctx, hipMemcpyAsync(R.h_out, R.d_out, sizeof(ResOut) + 3 * sizeof(double) * R.G, hipMemcpyDeviceToHost,
                                     ctx->stream));
    }
    FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  }
  if(!fits) {
    ctx->spmvTimer.used = 0;
    R.usable = false;
    return FE_STATUS_OK;
  }
  const ResOut &out = *R.h_out;
  if(out.gaveUp || out.reason == 0) {  // a wait ran out: the other kernels take over
    ctx->spmvTimer.used = 0;
    ctx->residentGaveUp = true;
    return FE_STATUS_OK;
  }
  res->ran = true;
  res->reason = out.reason;
  res->iters = out.iters;
  res->outer = out.outer;
  res->relres = out.bn > 0. ? out.rn / out.bn : 0.;
  const double *mx = (const double *)(R.h_out + 1);
  for(int k = 0; k < 3; ++k) res->inf[k] = 0.;
  for(int k = 0; k < 3 * R.G; ++k) res->inf[k % 3] = std::max(res->inf[k % 3], mx[k]);
  if(ctx->profiling) {  // the launch's time over its iterations
    float ms = 0.f;
    FeKernelTimer &t = ctx->spmvTimer;
    FE_HIP_TRY(ctx, hipEventElapsedTime(&ms, t.ev[t.used - 2], t.ev[t.used - 1]));
    t.total_ms += ms;
    t.launches += std::max(1, out.iters);
    t.used = 0;
  }
  return FE_STATUS_OK;
}

void feResidentRelease(fe_hip_ctx *ctx)
{
  if(ctx->res && ctx->res->h_out) (void)hipHostFree(ctx->res->h_out);
  delete ctx->res;  // device buffers are owned by the context
  ctx->res = nullptr;
}
