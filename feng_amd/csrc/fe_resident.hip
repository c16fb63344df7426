// Jacobi-PCG, and split-preconditioned PCG (resSplit), with all iterations in
// one launch (the KSPCG / PCJACOBI of the reference's options,
// feLinearSystemPETSc.cpp:900-1031): the pipelined recurrences of
// fe_krylov.hip's tileIter (Ghysels & Vanroose 2014), with the matrix in
// registers.
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
// The rule (resBuild): one row a thread on the CUs of the device (n <= 1024 x
// CUs, 262,144 on 256), rows of at most 24 entries (48 + 12 registers), and
// the rows of other workgroups that one gathers have to fit the LDS.  Larger
// systems are bound by the matrix traffic, which the tiled kernels stream.
// resSplit: rows of at most 16 entries above 512 x CUs rows (131,072), where
// workgroups have 1024 threads and no registers for longer ones.
#include "fe_resident.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

using namespace fe_res;

// What a solve returns to the host, and per workgroup the largest |x|, |b|,
// |b - A x| of its rows behind it.
struct ResOut {
  int reason, iters, outer, gaveUp, ended, pad;
  double bn, rn;
};

struct FeResident {
  bool built = false, usable = false;
  int G = 0, RW = 0, TB = 0, E = 0, H = 0;  // workgroups, rows and threads of one, entries a row, gathered rows at most
  unsigned *d_idx = nullptr;      // per workgroup E / 2 x TB packed pairs of LDS positions
  int *d_hcol = nullptr, *d_hcnt = nullptr;
  unsigned long long *d_buf = nullptr;  // kResBufs x (n values, 3 G partial sums)
  ResOut *d_out = nullptr, *h_out = nullptr;  // h_out: pinned copy
  int splitState = 0;             // split PCG: 1 ready, -1 the factor's pattern is not the matrix's
  int *d_pos = nullptr;
  unsigned long long *d_splitBuf = nullptr;
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
  int refine;      // FE_PREC_FP32_IR: the targets are tested before the first iteration too, with a bound on
                   // the restarts, as in that loop
  int wait;  // ticks
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
  if(blockIdx.x == 0 && threadIdx.x == 0) *out = ResOut{0, 0, 0, 0, 0, 0, 0., 0.};
}

// The workgroup's largest |x|, |b|, |b - A x|.
template <int TB>
__device__ __forceinline__ void resMaxima(bool own, double x, double b, double r, double (&part)[3][TB / 64], double *out)
{
  const int t = threadIdx.x;
  double mx[3] = {own ? fabs(x) : 0., fabs(b), own ? fabs(r) : 0.};
#pragma unroll
  for(int k = 0; k < 3; ++k) {
#pragma unroll
    for(int o = 32; o > 0; o >>= 1) mx[k] = fmax(mx[k], __shfl_xor(mx[k], o, 64));
    if((t & 63) == 0) part[k][t >> 6] = mx[k];
  }
  resBarrier();
  if(t < 3) {
    double mm = 0.;
    for(int k = 0; k < TB / 64; ++k) mm = fmax(mm, part[t][k]);
    out[t] = mm;
  }
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
  __shared__ int gaveUp, wait, refine;
  const int wg = blockIdx.x, t = threadIdx.x, G = a.G, RW = a.RW, stride = RW + a.H;
  const int row = wg * RW + t;
  const bool own = t < RW && row < a.n;
  const size_t bufLen = (size_t)a.n + 3 * (size_t)G;
  const int hc = a.hcnt[wg];
  const int *hcol = a.hcol + (size_t)wg * a.hcap;
  const int sumThreads = (G + 63) & ~63, h0 = kSplit ? t - sumThreads : t, hStep = kSplit ? TB - sumThreads : TB;
  if(t == 0) {
    gaveUp = 0;
    wait = a.wait;
    refine = a.refine;
  }
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
      bool ok = resPoll<kPoll>(buf, at, pv, wait);
#pragma unroll
      for(int k = 0; k < kHeld; ++k)
        if(hcl[k] >= 0) reg[RW + h0 + k * hStep] = __longlong_as_double((long long)pv[kSums + k]);
      for(int h = h0 + kHeld * hStep; h0 >= 0 && h < hc && ok; h += hStep) {
        const int a1[1] = {hcol[h]};
        unsigned long long v1[1];
        ok = resPoll<1>(buf, a1, v1, wait);
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
        if(bn == 0.) reason = 2;
        else if(refine && rn <= target) reason = 2;
        else if(refine && a.maxit <= 0) reason = -3;
        if(reason) break;
      } else {
        if(rn <= target) reason = 2;
        else if(code == 4 || !(rn == rn)) reason = -9;
        else if(it >= a.maxit && !refine) reason = -3;
        else if(rn / bn > a.dtol) reason = -4;
        else if(code == 3 && ++breakdowns > 20) reason = -3;
        else if(refine && outer >= kResOuter) reason = kResLimit;
        else if(it >= a.maxit) reason = -3;
        if(reason) break;
        // again from the true residual: after a breakdown, or when the
        // recursive residual met a target the true one has not (aim lower; the
        // bounded restarts of a refined solve keep the target)
        if(code != 3 && !refine) tol2 = resUniform(0.01 * tol2);
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
      a.out->ended = 1;
      a.out->reason = reason == kResLimit ? 0 : reason;
      a.out->iters = it;
      a.out->outer = outer;
      a.out->bn = bn;
      a.out->rn = rn;
    }
  }
  if(own) a.x[row] = x;
  resMaxima<TB>(own, x, own ? a.b[row] : 0., r, psum, a.maxima + 3 * wg);
}

// Split-preconditioned PCG, M^-1 = G^T D^-1 G with FP32 factor values (IC(0)
// or the learned factor), as a resident kernel: the pipelined recurrences of
// fe_krylov.hip's spIter.  The factor has the pattern of the matrix, so it
// adds one FP32 value per entry to the registers and no positions: G takes
// the entries up to the diagonal, G^T those from it.  An iteration is three
// exchanges, each with the slots of its own kind,
//   w with the three sums:  t = D^-1 G w      (columns below the own rows)
//   t:                      m = G^T t         (columns above)
//   m:                      n = A m, then the vector updates,
// where the launch-per-iteration form has three kernels that read the entries
// again.
// Solve with the factor's set-up, launches -> here: learned factor, P1
// tetrahedra 30^3 (n = 24,389) 2.46 -> 0.96 ms, 45^3 (85,184) 4.40 -> 1.73, 64^3
// (250,047, 1024 threads, part of the entries spilled) 8.70 -> 4.88; IC(0), P1
// triangles 160^2 6.26 -> 3.25, P2 60^2 8.45 -> 4.00.  An iteration is bound by
// its three trips of a stored word to another workgroup's poll.
//
// Slots come in three sets: after the sums of round k every workgroup has left
// round k - 1, whose slots are emptied then and polled again in round k + 2;
// the resets are complete before the sums of round k + 1 are published.
struct SplitArgs {
  ResArgs r;
  const int *pos;          // per workgroup E x TB: 2 k (G) or 2 k + 1 (G^T) of each entry, -1: none
  const float *gL, *gU, *dinv;
};

constexpr int kSplitSets = 3;

// Positions of a row's entries in the factor's two CSR forms; flag: entries of
// the factor outside the matrix's pattern.
__global__ void splitPattern(int n, int RW, int E, int TB, const int *__restrict__ ia, const int *__restrict__ ja,
                             const int *__restrict__ iaL, const int *__restrict__ jaL, const int *__restrict__ iaU,
                             const int *__restrict__ jaU, int *__restrict__ pos, int *flag)
{
  const int wg = blockIdx.x;
  for(int t = threadIdx.x; t < TB; t += blockDim.x) {
    const int row = wg * RW + t;
    const bool own = t < RW && row < n;
    const int kb = own ? ia[row] : 0, len = own ? ia[row + 1] - kb : 0;
    int nl = 0, nu = 0;
    for(int e = 0; e < E; ++e) {
      int f = -1;
      if(e < len) {
        const int j = ja[kb + e];
        const int *fa = j <= row ? iaL : iaU, *fj = j <= row ? jaL : jaU;
        for(int k = fa[row]; k < fa[row + 1] && f < 0; ++k)
          if(fj[k] == j) f = 2 * k + (j > row);
        if(f >= 0) j <= row ? ++nl : ++nu;
      }
      pos[((size_t)wg * E + e) * TB + t] = f;
    }
    if(own && (nl != iaL[row + 1] - iaL[row] || nu + 1 != iaU[row + 1] - iaU[row])) atomicMax(flag, 1);
  }
}

template <int TB, int E>
__global__ __launch_bounds__(TB) void resSplit(SplitArgs sa)
{
  const ResArgs &a = sa.r;
  constexpr int kHeld = TB == 512 ? 3 : 2;
  extern __shared__ double lds[];           // two regions of own + gathered values
  __shared__ double wsum[3][4], psum[3][TB / 64];
  __shared__ int gaveUp, wait, below;
  const int wg = blockIdx.x, t = threadIdx.x, G = a.G, RW = a.RW, stride = RW + a.H;
  const int r0 = wg * RW, row = r0 + t;
  const bool own = t < RW && row < a.n;
  const int oT = a.n, oM = 2 * a.n, oS = 3 * a.n;
  const size_t bufLen = 3 * ((size_t)a.n + G);
  const int hc = a.hcnt[wg];
  const int *hcol = a.hcol + (size_t)wg * a.hcap;
  if(t == 0) {
    gaveUp = 0;
    wait = a.wait;
    below = 0;
  }
  for(int q = t; q < 2 * stride; q += TB) lds[q] = 0.;  // a factor reads only the columns of its half
  __syncthreads();
  for(int h = t; h < hc; h += TB)
    if(hcol[h] < r0) atomicAdd(&below, 1);
  double v[E];
  float g[E], dinv = 0.f;
  unsigned ix[E / 2], low = 0, up = 0;  // bits: entries up to, from the diagonal
  double x = 0., r = 0., u = 0., w = 0., z = 0., q = 0., s = 0., p = 0., m = 0.;
#pragma unroll
  for(int e = 0; e < E / 2; ++e) ix[e] = a.idx[((size_t)wg * (E / 2) + e) * TB + t];
  {
    int kb = 0, len = 0;
    if(own) {
      kb = a.ia[row];
      len = a.ia[row + 1] - kb;
      r = a.b[row];
      dinv = sa.dinv[row];
    }
#pragma unroll
    for(int e = 0; e < E; ++e) {
      const int f = sa.pos[((size_t)wg * E + e) * TB + t];
      v[e] = e < len ? a.val[kb + e] : 0.;
      g[e] = f < 0 ? 0.f : f & 1 ? sa.gU[f >> 1] : sa.gL[f >> 1];
      if(e < len) {
        const int j = a.ja[kb + e];
        if(j <= row) low |= 1u << e;
        if(j >= row) up |= 1u << e;
      }
    }
  }
  int hcl[kHeld];
#pragma unroll
  for(int k = 0; k < kHeld; ++k) hcl[k] = t + k * TB < hc ? hcol[t + k * TB] : -1;
  resBarrier();
  const int hLow = below;  // hcol increases: these come first
  unsigned long long *buf = a.buf;
  int turn = 0;
  double *reg = lds;
  // Own value into the slots o + row and the region, the others' gathered rows
  // [h0, h1) from theirs; with kSum three partial sums, folded into f.
  auto exchange = [&](auto withSums, int o, double own1, int h0, int h1, const double (&sum)[3], double (&f)[3]) -> bool {
    constexpr bool kSum = decltype(withSums)::value;
    reg = lds + turn * stride;
    turn ^= 1;
    if(own) resStore(buf + o + row, own1);
    if(t < RW) reg[t] = own1;
    if constexpr(kSum) {
#pragma unroll
      for(int j = 0; j < 3; ++j) {
        const double ws = resWaveSum(own ? sum[j] : 0.);
        if((t & 63) == 0) psum[j][t >> 6] = ws;
      }
      resBarrier();
      if(t < 3) {
        double ws = 0.;
#pragma unroll
        for(int k = 0; k < TB / 64; ++k) ws += psum[t][k];
        resStore(buf + oS + t * G + wg, ws);
      }
    }
    constexpr int kS = kSum ? 3 : 0;
    unsigned long long pv[kS + kHeld];
    int at[kS + kHeld];
    if constexpr(kSum) {
#pragma unroll
      for(int j = 0; j < 3; ++j) at[j] = t < G ? oS + j * G + t : -1;
    }
#pragma unroll
    for(int k = 0; k < kHeld; ++k) {
      const int h = t + k * TB;
      at[kS + k] = h >= h0 && h < h1 ? o + hcl[k] : -1;
    }
    bool ok = resPoll<kS + kHeld>(buf, at, pv, wait);
#pragma unroll
    for(int k = 0; k < kHeld; ++k)
      if(at[kS + k] >= 0) reg[RW + t + k * TB] = __longlong_as_double((long long)pv[kS + k]);
    for(int h = t + kHeld * TB; h < h1 && ok; h += TB) {
      if(h < h0) continue;
      const int a1[1] = {o + hcol[h]};
      unsigned long long v1[1];
      ok = resPoll<1>(buf, a1, v1, wait);
      reg[RW + h] = __longlong_as_double((long long)v1[0]);
    }
    if(!ok) gaveUp = 1;
    if constexpr(kSum) {
      if(t < ((G + 63) & ~63)) {
#pragma unroll
        for(int j = 0; j < 3; ++j) {
          const double ws = resWaveSum(t < G ? __longlong_as_double((long long)pv[j]) : 0.);
          if((t & 63) == 0) wsum[j][t >> 6] = ws;
        }
      }
    }
    resBarrier();
    if(gaveUp) return false;
    if constexpr(kSum) {
#pragma unroll
      for(int j = 0; j < 3; ++j) {
        double ws = 0.;
        for(int k = 0; k < (G + 63) / 64; ++k) ws += wsum[j][k];
        f[j] = resUniform(ws);
      }
    }
    return true;
  };
  auto product = [&]() {  // the matrix
    double y = 0.;
#pragma unroll
    for(int e = 0; e < E / 2; ++e) {
      asm volatile("" : "+v"(ix[e]));  // unpacked here, not kept unpacked across the loop
      y += v[2 * e] * reg[ix[e] & 0xffffu];
      y += v[2 * e + 1] * reg[ix[e] >> 16];
      if constexpr(TB == 1024 || E == 24)
        if(e % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" : "+v"(y));
    return y;
  };
  auto factor = [&](unsigned half) {  // G or G^T: the entries with their bit set
    double y = 0.;
    asm volatile("" : "+v"(half));
#pragma unroll
    for(int e = 0; e < E / 2; ++e) {
      asm volatile("" : "+v"(ix[e]), "+v"(g[2 * e]), "+v"(g[2 * e + 1]));  // nor converted
      const float g0 = half & (1u << (2 * e)) ? g[2 * e] : 0.f, g1 = half & (2u << (2 * e)) ? g[2 * e + 1] : 0.f;
      y += (double)g0 * reg[ix[e] & 0xffffu];
      y += (double)g1 * reg[ix[e] >> 16];
      if constexpr(TB == 1024 || E == 24)
        if(e % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // eight reads in flight, not a register for each
    }
    asm volatile("" : "+v"(y));  // summed here, not where it is used
    return y;
  };
  using Yes = std::true_type;
  using No = std::false_type;
  // uniform state (every workgroup folds the same sums in the same order)
  double alphaP = __builtin_inf(), gammaP = 1., bn = 0., rn = 0., target = 0., tol2 = 0.;
  int code = 0, it = 0, outer = 0, breakdowns = 0, reason = 0;
  bool start = true;
  for(int k = 0;; ++k) {
    buf = a.buf + (k % kSplitSets) * bufLen;
    double sum[3] = {r * r, 0., 0.}, f[3];
    if(!start) {
      sum[0] = r * u;
      sum[1] = w * u;
      sum[2] = r * r;
    }
    resStoresDone();  // the resets of the previous round
    if(!exchange(Yes{}, 0, start ? r : w, 0, hLow, sum, f)) break;
    {  // the slots of round k + 2 are empty again
      unsigned long long *rs = a.buf + ((k + 2) % kSplitSets) * bufLen;
      if(own) {
        resStore(rs + row, kSentinel);
        resStore(rs + oT + row, kSentinel);
        resStore(rs + oM + row, kSentinel);
      }
      if(t < 3) resStore(rs + oS + t * G + wg, kSentinel);
    }
    double alpha = 0., beta = 0.;
    if(start) {
      rn = resUniform(sqrt(f[0]));  // ||b||, or the true residual's norm
      if(outer == 0) {
        bn = rn;
        target = resUniform(fmax(a.rtol * bn, a.atol));
        tol2 = resUniform(target * target * 0.25);
        if(bn == 0. || rn <= target) reason = 2;
        else if(a.maxit <= 0) reason = -3;
      } else {
        if(rn <= target) reason = 2;
        else if(code == 4 || !(rn == rn)) reason = -9;
        else if(code == 3 && ++breakdowns > 20) reason = -3;
        else if(rn / bn > a.dtol) reason = -4;
        else if(outer >= kResOuter) reason = kResLimit;
        else if(it >= a.maxit) reason = -3;
        code = 0;  // again from the true residual
      }
      if(reason) break;
      z = q = s = p = 0.;
      gammaP = 1.;
      alphaP = __builtin_inf();
    } else {
      if(!(f[2] > tol2) || it >= a.maxit) {
        code = f[2] <= tol2 ? 1 : (f[2] == f[2] ? 2 : 4);
      } else {
        beta = resUniform(f[0] / gammaP);
        const double den = f[1] - beta * f[0] / alphaP;
        if(den > 0.) {
          alpha = resUniform(f[0] / den);
          gammaP = f[0];
          alphaP = alpha;
          ++it;
        } else {
          code = 3;  // breakdown: the preconditioned operator is not SPD
        }
      }
      if(code) {  // the true residual
        if(!exchange(No{}, oM, x, 0, hc, sum, f)) break;
        r = own ? a.b[row] - product() : 0.;
        ++outer;
        start = true;
        continue;
      }
    }
    const double tv = (double)dinv * factor(low);
    if(!exchange(No{}, oT, tv, hLow, hc, sum, f)) break;
    m = factor(up);
    if(!exchange(No{}, oM, m, 0, hc, sum, f)) break;
    const double y = product();
    if(start) {
      u = m;
      w = y;
      start = false;
    } else {
      z = y + beta * z;
      q = m + beta * q;
      s = w + beta * s;
      p = u + beta * p;
      x = x + alpha * p;
      r = r - alpha * s;
      u = u - alpha * q;
      w = w - alpha * z;
    }
  }
  if(t == 0) {
    if(gaveUp) __hip_atomic_store(&a.out->gaveUp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if(wg == 0) {
      a.out->ended = 1;
      a.out->reason = reason == kResLimit ? 0 : reason;
      a.out->iters = it;
      a.out->outer = outer;
      a.out->bn = bn;
      a.out->rn = rn;
    }
  }
  if(own) a.x[row] = x;
  resMaxima<TB>(own, x, own ? a.b[row] : 0., r, psum, a.maxima + 3 * wg);
}

template <typename Args>
int launchRes(fe_hip_ctx *ctx, void (*kernel)(Args), int TB, const FeResident &R, const Args &a, size_t lds, bool *fits)
{
  const void *f = (const void *)kernel;
  int perCu = 0, cus = 0;
  std::lock_guard<std::mutex> lock(feResidentGate(ctx->device).launching());
  *fits = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess &&
          hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, f, TB, lds) == hipSuccess &&
          hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) == hipSuccess &&
          perCu * cus >= R.G;
  if(!*fits) {
    (void)hipGetLastError();
    return FE_STATUS_OK;
  }
  hipLaunchKernelGGL(kernel, dim3(R.G), dim3(TB), lds, ctx->stream, a);
  FE_HIP_TRY(ctx, hipGetLastError());
  return FE_STATUS_OK;
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

FeResidentGate &feResidentGate(int device)
{
  static FeResidentGate g[64];
  return g[device & 63];
}

namespace {

// One resident launch over `bufLen` slots, and what it returned.  launch(&fits)
// enqueues the kernel.
template <typename F>
int resRun(fe_hip_ctx *ctx, const fe_hip_solver_opts *o, FeResident &R, unsigned long long *buf, size_t cells,
           FeResidentResult *res, F launch)
{
  bool fits = false;
  {
    const FeResidentPass pass(ctx, R.G);
    if(ctx->profiling)
      if(int rc = feTimerMark(ctx, ctx->spmvTimer)) return rc;
    hipLaunchKernelGGL(resFill, dim3((unsigned)std::min<size_t>(1024, (cells + 255) / 256)), dim3(256), 0, ctx->stream,
                       cells, buf, R.d_out);
    if(int rc = launch(&fits)) return rc;
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
  if(out.gaveUp || !out.ended) {  // a wait ran out: the other kernels take over
    ctx->spmvTimer.used = 0;
    ctx->residentGaveUp = true;
    return FE_STATUS_OK;
  }
  if(resCutShort(ctx, o, out.iters, out.reason)) {
    ctx->spmvTimer.used = 0;
    return FE_STATUS_OK;
  }
  res->ran = ctx->residentRan = true;
  res->reason = out.reason;
  res->iters = out.iters;
  res->outer = out.outer;
  res->relres = out.bn == 0. ? 0. : out.rn / out.bn;  // not a number stays that
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

int resPrepare(fe_hip_ctx *ctx)
{
  if(!ctx->res) ctx->res = new FeResident();
  if(!ctx->res->built) return resBuild(ctx, *ctx->res);
  return FE_STATUS_OK;
}

ResArgs resArgs(const fe_hip_ctx *ctx, const FeResident &R, const fe_hip_solver_opts *o, double *x,
                unsigned long long *buf)
{
  const int hcap = std::min(kResH, kResLds / 16 - R.RW);
  return ResArgs{ctx->n,   R.G,        R.RW, R.H, hcap,    ctx->d_ia, ctx->d_ja,       ctx->d_val, R.d_idx, R.d_hcol,
                 R.d_hcnt, ctx->d_rhs, x,    buf, R.d_out, (double *)(R.d_out + 1), o->rtol, o->atol, o->dtol,
                 std::min(o->max_iter, ctx->residentMaxIter), o->precision == FE_PREC_FP32_IR, resWaitTicks(ctx)};
}

}  // namespace

int feResidentJacobi(fe_hip_ctx *ctx, const fe_hip_solver_opts *o, double *x, FeResidentResult *res)
{
  res->ran = false;
  if(!ctx->resident || ctx->residentGaveUp) return FE_STATUS_OK;
  if(int rc = resPrepare(ctx)) return rc;
  FeResident &R = *ctx->res;
  if(!R.usable) return FE_STATUS_OK;
  const ResArgs a = resArgs(ctx, R, o, x, R.d_buf);
  const size_t lds = 2 * (size_t)(R.RW + R.H) * sizeof(double);
  return resRun(ctx, o, R, R.d_buf, kResBufs * ((size_t)ctx->n + 3 * (size_t)R.G), res, [&](bool *fits) {
    auto *const k = R.TB == 512 ? (R.E == 8 ? resJacobi<512, 8> : R.E == 16 ? resJacobi<512, 16> : resJacobi<512, 24>)
                                : (R.E == 8 ? resJacobi<1024, 8> : R.E == 16 ? resJacobi<1024, 16> : resJacobi<1024, 24>);
    return launchRes(ctx, k, R.TB, R, a, lds, fits);
  });
}

int feResidentSplit(fe_hip_ctx *ctx, const fe_hip_solver_opts *o, double *x, FeResidentResult *res)
{
  res->ran = false;
  if(!ctx->resident || ctx->residentGaveUp || !ctx->pcValues32 || ctx->pcFp32) return FE_STATUS_OK;
  if(int rc = resPrepare(ctx)) return rc;
  FeResident &R = *ctx->res;
  // 1024 threads have no registers for longer rows
  if(!R.usable || R.splitState < 0 || (R.TB == 1024 && R.E > 16)) return FE_STATUS_OK;
  const FePrecond &P = ctx->pc;
  const size_t cells = kSplitSets * 3 * ((size_t)ctx->n + R.G);
  if(R.splitState == 0) {
    int *flag = nullptr, bad = 0;
    if(feAlloc(ctx, &flag, 1) || feAlloc(ctx, &R.d_pos, (size_t)R.G * R.E * R.TB) || feAlloc(ctx, &R.d_splitBuf, cells))
      return FE_STATUS_OUT_OF_MEMORY;
    FE_HIP_TRY(ctx, hipMemsetAsync(flag, 0, sizeof(int), ctx->stream));
    hipLaunchKernelGGL(splitPattern, dim3(R.G), dim3(512), 0, ctx->stream, ctx->n, R.RW, R.E, R.TB, ctx->d_ia, ctx->d_ja,
                       P.d_iaL, P.d_jaL, P.d_iaU, P.d_jaU, R.d_pos, flag);
    FE_HIP_TRY(ctx, hipGetLastError());
    FE_HIP_TRY(ctx, hipMemcpyAsync(&bad, flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    feFree(ctx, flag);
    R.splitState = bad ? -1 : 1;
    if(bad) return FE_STATUS_OK;
  }
  const SplitArgs a{resArgs(ctx, R, o, x, R.d_splitBuf), R.d_pos, P.d_gL32, P.d_gU32, P.d_dinv32};
  const size_t lds = 2 * (size_t)(R.RW + R.H) * sizeof(double);
  return resRun(ctx, o, R, R.d_splitBuf, cells, res, [&](bool *fits) {
    auto *const k = R.TB == 512 ? (R.E == 8 ? resSplit<512, 8> : R.E == 16 ? resSplit<512, 16> : resSplit<512, 24>)
                                : (R.E == 8 ? resSplit<1024, 8> : resSplit<1024, 16>);
    return launchRes(ctx, k, R.TB, R, a, lds, fits);
  });
}

void feResidentRelease(fe_hip_ctx *ctx)
{
  if(ctx->res && ctx->res->h_out) (void)hipHostFree(ctx->res->h_out);
  delete ctx->res;  // device buffers are owned by the context
  ctx->res = nullptr;
}
