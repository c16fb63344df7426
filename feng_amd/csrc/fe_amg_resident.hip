// Multigrid-PCG with all iterations in one launch: the nested-ordered PCG of
// fe_amg_pcg.hip (standard PCG, one symmetric V-cycle of the aggregation
// hierarchy per iteration) as a resident kernel (fe_resident.h).
//
// An iteration of the launch-per-level form is 2 + 2 B + 1 dependent launches
// (B: first level of the single-workgroup part) of 4 to 17 us, most of it the
// launch boundary, loads of row bounds and entries, and for the single
// workgroup the copy of its levels into LDS: 47 us an iteration at 21^3
// tetrahedra (8,000 unknowns), 65 us at 37^3, 92 us at 64^3.  The nested order
// makes the whole cycle local: a workgroup owns a range of level B - 1 rows
// and, with them, the contiguous rows below them on every finer level, so
// restrictions and prolongations stay inside it and only the products need
// boundary values of neighbours.  Per workgroup
//   level 0       one thread a row, FP64 entries and x, r, p, q, A u in registers;
//   1 .. B - 1    matrix rows, b, u, e in LDS, four lanes a row;
//   B .. coarsest in LDS of every workgroup, solved by all of them alike: the
//                 restricted residual is exchanged once and no correction has
//                 to be sent back.
// Exchanges of one iteration: z; w = l1 A z with (r, z), (z, A z), (r, r), the
// only sums over all workgroups (Chronopoulos & Gear's form of CG); u and y of
// each level 1 .. B - 1; the parts of b_B; y of level 0.
//   z:  A z, w = l1 A z
//   w:  beta = rho / rho_old, alpha = rho / ((z, A z) - beta rho / alpha_old);
//       p = z + beta p, q = A z + beta q, a = A w + beta a (= A l1 q);
//       x += alpha p, r -= alpha q, A u -= alpha a for u = l1 r
//   y:  z = y + l1 (r - A y)
// What bounds an iteration is the chain of exchanges (1.3 to 3.3 us for the
// neighbours' values, 3.3 to 6.3 us for the sums) and, on the largest matrices,
// the single-workgroup levels (3.6 us at 190 rows, 11.6 us at 688), not bytes.
// Solve with numeric set-up, launch-per-level -> here: 21^3 1.43 -> 0.62 ms,
// 37^3 2.6 -> 1.15 ms, 64^3 (250,047 unknowns) 4.8 -> 2.38 ms.  Only rows that
// another workgroup gathers are stored to the exchange buffer: the write-through
// stores of all rows and their resets took 3 us an iteration at 64^3.
//
// Exchange slots are used once per iteration and come in three sets: after
// the sums of iteration k every workgroup has left iteration k - 1, whose
// slots are emptied then and are polled again in iteration k + 2; each
// workgroup publishes its sums of iteration k + 1 after its resets are
// complete.
//
// The rule (arBuild): two rows a thread of the device (at most 1024 a
// workgroup, cut at level B - 1 rows: 249,001 P1 triangle unknowns fit, 261,121
// do not), level-0 rows of at most 24 entries, FP64 vectors with FP32 level
// values, and the LDS plan has to fit; otherwise the launch-per-level kernels
// run.  512 threads leave 256 registers to each; 1024
// threads of one row spilled (64 registers more for what does not depend on the
// row): 3.6 instead of 1.3 us for a product with its resets at 21^3.
#include "fe_resident.h"
#include "fe_amg_nested.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

using namespace fe_res;

namespace {

constexpr int kMaxDist = 6;       // distributed levels 0 .. B - 1
constexpr int kMaxBlk = 8;        // levels B .. coarsest - 1
constexpr int kArLds = 156 * 1024;
constexpr int kArRows = 256;      // rows a workgroup below the full device (37^3: 26.8 us an iteration on 182
                                  // workgroups, 30.0 on 92; 150^2 P2: 30.6 on 255, 48.8 on 175 of two rows a thread)
constexpr int kArBlockRows[2] = {512, 1024};  // level B: few rows, or what the LDS holds
constexpr int kTB = 512;
constexpr int kSentBit = 0x8000;
constexpr int kSets = 3;          // sets of exchange slots

struct ArOut {
  int reason, iters, outer, gaveUp, badPivot, ended;
  double bn, rn;
};

// A distributed level; o*: word offsets in an exchange buffer, l*: byte
// offsets in LDS.
struct ArDist {
  const int *rs;       // G + 1: first own row
  const int *ia;       // levels >= 1
  const unsigned short *lidx;  // levels >= 1: LDS position of each entry's column
  const float *val, *l1;
  const int *agg, *aggStart;
  const int *hcol, *hcnt;
  const unsigned char *sent;   // rows that another workgroup gathers
  int n, rows, hcap;   // rows: the most of any workgroup (the gathered values' first position)
  int oU, oY;
  int lReg, lB, lU, lE, lVal, lIdx, lOff, lL1, lAgg, lAs, lHc;
};

struct ArBlock {
  int nLev, bytes;  // levels B .. coarsest - 1; bytes of the image
  int n[kMaxBlk + 1], nc[kMaxBlk], nnz[kMaxBlk];
  int oIa[kMaxBlk], oJa[kMaxBlk], oVal[kMaxBlk], oL1[kMaxBlk], oAgg[kMaxBlk], oAs[kMaxBlk], oCi, oPs;
  int lImg, lB[kMaxBlk + 1], lU[kMaxBlk], lX, lParts;
};

struct ArArgs {
  int n, G, B, parts;
  ArDist lv[kMaxDist];
  ArBlock blk;
  const int2 *sell;
  const double *val0;
  const unsigned *idx0;
  const int *perm, *partBase, *partFirst;  // partBase: G + 1 first slots; partFirst: first level-B row
  const unsigned char *img;
  const int *badPivot;
  const double *b;
  double *x;
  unsigned long long *buf;
  size_t bufLen;
  int oZ, oS, oParts;
  int lReg0;
  ArOut *out;
  double *maxima;
  double rtol, atol, dtol, oc;
  int maxit;
  int wait;  // ticks
};

// LDS positions of the columns of a workgroup's rows (see fe_resident.hip):
// own rows first, the others behind position `rows`, in increasing order.
// SELL: level 0, packed per thread; otherwise one position per CSR entry.
template <bool SELL>
__global__ __launch_bounds__(1024) void arPattern(int n, const int *__restrict__ rs, int rows, int E, int TB, int hcap,
                                                  const int2 *__restrict__ sell, const int *__restrict__ ia,
                                                  const int *__restrict__ ja, unsigned short *__restrict__ idx,
                                                  int *__restrict__ hcol, int *__restrict__ hcnt, int *flag)
{
  __shared__ unsigned bits[8192];
  __shared__ int base[8192];
  __shared__ int sums[1024];
  const int wg = blockIdx.x, t = threadIdx.x, r0 = rs[wg], r1 = rs[wg + 1], nw = (n + 31) / 32;
  for(int q = t; q < nw; q += 1024) bits[q] = 0u;
  __syncthreads();
  auto mark = [&](int j) {
    if(j < r0 || j >= r1) atomicOr(&bits[j >> 5], 1u << (j & 31));
  };
  if(SELL) {
    for(int r = r0 + t; r < r1; r += 1024) {
      const int2 bl = sell[r];
      for(int e = 0; e < bl.y; ++e) mark(ja[bl.x + 64 * e]);
    }
  } else {
    for(int k = ia[r0] + t; k < ia[r1]; k += 1024) mark(ja[k]);
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
    atomicMax(flag, sums[1023]);
  }
  auto position = [&](int j) {
    const int p = j >= r0 && j < r1 ? j - r0 : rows + base[j >> 5] + __popc(bits[j >> 5] & ((1u << (j & 31)) - 1u));
    return (unsigned short)min(p, 65535);
  };
  if(SELL) {
    for(int i = t; i < TB; i += 1024) {  // TB: positions a workgroup has for rows
      const int2 bl = r0 + i < r1 ? sell[r0 + i] : make_int2(0, 0);
      for(int e = 0; e < E; ++e)
        idx[(((size_t)wg * (E / 2) + e / 2) * TB + i) * 2 + (e & 1)] =
            e < bl.y ? position(ja[bl.x + 64 * e]) : (unsigned short)min(i, rows - 1);  // no entry: value 0, own row
    }
  } else {
    for(int k = ia[r0] + t; k < ia[r1]; k += 1024) idx[k] = position(ja[k]);
  }
}

// Marks the rows that a workgroup gathers from another one.
__global__ void arSent(const int *__restrict__ hcol, const int *__restrict__ hcnt, int hcap,
                       unsigned char *__restrict__ sent)
{
  const int cnt = min(hcnt[blockIdx.x], hcap);
  for(int h = threadIdx.x; h < cnt; h += blockDim.x) sent[hcol[(size_t)blockIdx.x * hcap + h]] = 1;
}

struct ArPackLevel {
  int n, nc, nnz, oIa, oJa, oVal, oL1, oAgg, oAs;
  const int *ia, *ja, *agg, *aggStart;
  const float *val, *l1;
};
struct ArPackArgs {
  int nLev, nC, oCi;
  ArPackLevel lv[kMaxBlk];
  const double *cinv;
  unsigned char *img;
};

// The levels B .. coarsest (16-bit offsets, columns and aggregates, FP32
// values, the coarsest inverse) in their LDS layout, once per numeric set-up:
// one level a block, the inverse the last.
__global__ __launch_bounds__(256) void arPack(ArPackArgs a)
{
  const int s = blockIdx.y;
  const int t = blockIdx.x * 256 + threadIdx.x, step = gridDim.x * 256;
  if(s == a.nLev) {
    for(int q = t; q < a.nC * a.nC; q += step) ((double *)(a.img + a.oCi))[q] = a.cinv[q];
    return;
  }
  const ArPackLevel &L = a.lv[s];
  for(int q = t; q <= L.n; q += step) ((unsigned short *)(a.img + L.oIa))[q] = (unsigned short)L.ia[q];
  for(int q = t; q < L.nnz; q += step) {
    ((unsigned short *)(a.img + L.oJa))[q] = (unsigned short)L.ja[q];
    ((float *)(a.img + L.oVal))[q] = L.val[q];
  }
  for(int q = t; q < L.n; q += step) {
    ((float *)(a.img + L.oL1))[q] = L.l1[q];
    ((unsigned short *)(a.img + L.oAgg))[q] = (unsigned short)L.agg[q];
  }
  for(int q = t; q <= L.nc; q += step) ((unsigned short *)(a.img + L.oAs))[q] = (unsigned short)L.aggStart[q];
}

__global__ void arFill(size_t count, unsigned long long *__restrict__ buf, ArOut *out)
{
  for(size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
    buf[i] = kSentinel;
  if(blockIdx.x == 0 && threadIdx.x == 0) *out = ArOut{0, 0, 0, 0, 0, 0, 0., 0.};
}

// sum over [k0, k1) of val[k] x[ja[k]] for a row of an LDS matrix, LPR (1, 2,
// 4, 8) consecutive lanes; every one of them gets the sum.
template <int LPR>
__device__ __forceinline__ double ldsRowSum(int k0, int k1, int sub, const unsigned short *ja, const float *val,
                                            const double *x)
{
  constexpr int U = LPR == 1 ? 8 : 4;
  double acc = 0.;
  for(int k = k0 + sub; k < k1; k += U * LPR) {
    int c[U];
    float v[U];
    double g[U];
#pragma unroll
    for(int u = 0; u < U; ++u) {
      const bool in = k + u * LPR < k1;
      const int kk = in ? k + u * LPR : k0;
      c[u] = ja[kk];
      v[u] = val[kk];
      if(!in) v[u] = 0.f;
    }
#pragma unroll
    for(int u = 0; u < U; ++u) g[u] = x[c[u]];
#pragma unroll
    for(int u = 0; u < U; ++u) acc += (double)v[u] * g[u];
  }
  if constexpr(LPR >= 2) acc += dppMove<0xB1>(acc);
  if constexpr(LPR >= 4) acc += dppMove<0x4E>(acc);
  if constexpr(LPR >= 8) acc += dppMove<0x141>(acc);
  return acc;
}

// f(row, sum_j a_row,j x_j) for all n rows of an LDS matrix, by as many lanes
// a row as the workgroup has.
template <int LPR, typename F>
__device__ __forceinline__ void ldsRowsL(int n, const unsigned short *off, const unsigned short *ja, const float *val,
                                         const double *x, F f)
{
  const int sub = threadIdx.x % LPR;
  for(int i = threadIdx.x / LPR; i < n; i += kTB / LPR) {
    const double s = ldsRowSum<LPR>(off[i], off[i + 1], sub, ja, val, x);
    if(sub == 0) f(i, s);
  }
}
template <typename F>
__device__ __forceinline__ void ldsRows(int n, const unsigned short *off, const unsigned short *ja, const float *val,
                                        const double *x, F f)
{
  if(n * 8 <= kTB) ldsRowsL<8>(n, off, ja, val, x, f);
  else if(n * 4 <= kTB) ldsRowsL<4>(n, off, ja, val, x, f);
  else if(n * 2 <= kTB) ldsRowsL<2>(n, off, ja, val, x, f);
  else ldsRowsL<1>(n, off, ja, val, x, f);
}

// Sum of x over [m0, m1), a few loads in flight together.
__device__ __forceinline__ double ldsRange(const double *x, int m0, int m1)
{
  double s = 0.;
  for(int m = m0; m < m1; m += 4) {
    double g[4];
#pragma unroll
    for(int u = 0; u < 4; ++u) g[u] = x[min(m + u, m1 - 1)];
#pragma unroll
    for(int u = 0; u < 4; ++u) s += m + u < m1 ? g[u] : 0.;
  }
  return s;
}

// The V-cycle of levels B .. coarsest from b and u = l1 b of level B in LDS
// (blk.lB[0], blk.lU[0]); e of every level replaces its b (blk.lX: the
// coarsest); the residuals share one array with the parts of b_B.
__device__ __forceinline__ void arBlockSolve(const ArBlock &k, unsigned char *lds, double oc)
{
  const int t = threadIdx.x;
  const unsigned char *im = lds + k.lImg;
  for(int s = 0; s < k.nLev; ++s) {
    const unsigned short *ia = (const unsigned short *)(im + k.oIa[s]), *ja = (const unsigned short *)(im + k.oJa[s]),
                         *as = (const unsigned short *)(im + k.oAs[s]);
    const float *val = (const float *)(im + k.oVal[s]);
    const double *b = (const double *)(lds + k.lB[s]), *u = (const double *)(lds + k.lU[s]);
    double *r = (double *)(lds + k.lParts), *bn = (double *)(lds + k.lB[s + 1]);
    ldsRows(k.n[s], ia, ja, val, u, [&](int i, double acc) { r[i] = b[i] - acc; });
    resBarrier();
    const bool more = s + 1 < k.nLev;
    const float *l1n = (const float *)(im + k.oL1[more ? s + 1 : s]);
    double *un = (double *)(lds + k.lU[more ? s + 1 : s]);
    for(int I = t; I < k.nc[s]; I += kTB) {
      const double acc = ldsRange(r, as[I], as[I + 1]);
      bn[I] = acc;
      if(more) un[I] = (double)l1n[I] * acc;
    }
    resBarrier();
  }
  {
    const int nC = k.n[k.nLev];
    const double *b = (const double *)(lds + k.lB[k.nLev]), *ci = (const double *)(im + k.oCi);
    double *x = (double *)(lds + k.lX);
    const int i = t / 8, sub = t & 7;  // nC <= 64
    if(i < nC) {
      double acc = 0.;
#pragma unroll 4
      for(int j = sub; j < nC; j += 8) acc += ci[i * nC + j] * b[j];
      acc += dppMove<0xB1>(acc);
      acc += dppMove<0x4E>(acc);
      acc += dppMove<0x141>(acc);
      if(sub == 0) x[i] = acc;
    }
    resBarrier();
  }
  for(int s = k.nLev - 1; s >= 0; --s) {
    const int n = k.n[s];
    const unsigned short *ia = (const unsigned short *)(im + k.oIa[s]), *ja = (const unsigned short *)(im + k.oJa[s]),
                         *agg = (const unsigned short *)(im + k.oAgg[s]);
    const float *val = (const float *)(im + k.oVal[s]), *l1 = (const float *)(im + k.oL1[s]);
    double *be = (double *)(lds + k.lB[s]), *y = (double *)(lds + k.lU[s]);
    const double *en = (const double *)(lds + (s + 1 == k.nLev ? k.lX : k.lB[s + 1]));
    for(int i = t; i < n; i += kTB) y[i] = __builtin_fma(oc, en[agg[i]], y[i]);
    resBarrier();
    ldsRows(n, ia, ja, val, y, [&](int i, double acc) { be[i] = __builtin_fma((double)l1[i], be[i] - acc, y[i]); });
    resBarrier();
  }
}

template <int RPT, int E>
__global__ __launch_bounds__(kTB) void arSolve(ArArgs a)
{
  extern __shared__ __align__(16) unsigned char lds[];
  constexpr int kHeld = RPT == 1 ? 2 : 4;
  __shared__ double wsum[3][4], psum[3][kTB / 64];
  __shared__ int gaveUp, wait;
  __shared__ int4 info[kMaxDist + 1];  // per level: first own row, own rows, gathered rows
  const int wg = blockIdx.x, t = threadIdx.x, G = a.G, B = a.B;
  const ArDist &L0 = a.lv[0];
  const int rs0 = L0.rs[wg], R0 = L0.rs[wg + 1] - rs0;
  const int hc0 = L0.hcnt[wg];
  const int *hcol0 = L0.hcol + (size_t)wg * L0.hcap;
  const int pb = a.partBase[wg], pc = a.partBase[wg + 1] - pb, pf = a.partFirst[wg];
  if(t == 0) {
    gaveUp = 0;
    wait = a.wait;
  }
  // --- what stays for the whole solve
  for(int c = t; c < a.blk.bytes / 16; c += kTB) ((uint4 *)(lds + a.blk.lImg))[c] = ((const uint4 *)a.img)[c];
  for(int l = 0; l < B; ++l) {
    const ArDist &L = a.lv[l];
    const int r0 = L.rs[wg], R = L.rs[wg + 1] - r0, hc = L.hcnt[wg];
    if(t == 0) info[l] = make_int4(r0, R, hc, 0);
    // starts of the own rows' aggregates, and the aggregate of each row: local
    // to the workgroup, or on level B itself
    const int c0 = l + 1 < B ? a.lv[l + 1].rs[wg] : pf, C = l + 1 < B ? a.lv[l + 1].rs[wg + 1] - c0 : pc;
    unsigned short *as = (unsigned short *)(lds + L.lAs);
    for(int c = t; c <= C; c += kTB)
      as[c] = (unsigned short)max(0, min(R, L.aggStart[c0 + c] - r0));
    if(l == 0) continue;
    const int k0 = L.ia[r0], K = L.ia[r0 + R] - k0;
    for(int k = t; k < K; k += kTB) {
      ((float *)(lds + L.lVal))[k] = L.val[k0 + k];
      ((unsigned short *)(lds + L.lIdx))[k] = L.lidx[k0 + k];
    }
    for(int r = t; r <= R; r += kTB) ((unsigned short *)(lds + L.lOff))[r] = (unsigned short)(L.ia[r0 + r] - k0);
    for(int r = t; r < R; r += kTB) {
      ((float *)(lds + L.lL1))[r] = L.l1[r0 + r];
      // the top bit: the row is sent
      ((unsigned short *)(lds + L.lAgg))[r] =
          (unsigned short)((L.agg[r0 + r] - (l + 1 < B ? c0 : 0)) | (L.sent[r0 + r] ? kSentBit : 0));
    }
    for(int h = t; h < hc; h += kTB) ((int *)(lds + L.lHc))[h] = L.hcol[(size_t)wg * L.hcap + h];
  }
  double v[RPT][E];
  unsigned ix[RPT][E / 2];
  bool own[RPT], send[RPT];
  int orig[RPT], ag[RPT];
  float l1[RPT];
  double x[RPT], r[RPT], p[RPT], q[RPT], aq[RPT], au[RPT], z[RPT];
#pragma unroll
  for(int i = 0; i < RPT; ++i) {
    const int lr = t + i * kTB, row = rs0 + lr;
    own[i] = lr < R0;
#pragma unroll
    for(int e = 0; e < E / 2; ++e) ix[i][e] = a.idx0[((size_t)wg * (E / 2) + e) * (RPT * kTB) + lr];
    const int2 bl = own[i] ? a.sell[row] : make_int2(0, 0);
#pragma unroll
    for(int e = 0; e < E; ++e) v[i][e] = e < bl.y ? a.val0[bl.x + 64 * e] : 0.;
    send[i] = own[i] && L0.sent[row];
    orig[i] = own[i] ? a.perm[row] : 0;
    l1[i] = own[i] ? L0.l1[row] : 0.f;
    ag[i] = own[i] ? L0.agg[row] - (B > 1 ? a.lv[1].rs[wg] : 0) : 0;
    x[i] = p[i] = q[i] = aq[i] = au[i] = z[i] = 0.;
    r[i] = own[i] ? a.b[orig[i]] : 0.;
  }
  int hcl[kHeld];
#pragma unroll
  for(int k = 0; k < kHeld; ++k) hcl[k] = t + k * kTB < hc0 ? hcol0[t + k * kTB] : -1;
  // --- uniform state
  double bn = 0., rn = 0., target = 0., tol2 = 0., rhoOld = 1., alphaOld = 1.;
  int it = 0, outer = 0, breakdowns = 0, reason = 0;
  bool iterating = false, started = false, first = true, alive = true;
  unsigned long long *buf = a.buf;
  resBarrier();

  // Own values into the slots o + row and the region, the gathered values of
  // the other rows; with kSum three partial sums, folded into f.  False: gave up.
  auto exchange0 = [&](auto withSums, int o, const double (&m)[RPT], const double (&s)[3], double (&f)[3]) -> bool {
    constexpr bool kSum = decltype(withSums)::value;
    double *reg = (double *)(lds + a.lReg0);
#pragma unroll
    for(int i = 0; i < RPT; ++i)
      if(own[i]) {
        if(send[i]) resStore(buf + o + rs0 + t + i * kTB, m[i]);
        reg[t + i * kTB] = m[i];
      }
    if constexpr(kSum) {
#pragma unroll
      for(int j = 0; j < 3; ++j) {
        const double w = resWaveSum(s[j]);
        if((t & 63) == 0) psum[j][t >> 6] = w;
      }
      resBarrier();
      if(t < 3) {
        double sum = 0.;
#pragma unroll
        for(int k = 0; k < kTB / 64; ++k) sum += psum[t][k];
        resStore(buf + a.oS + t * G + wg, sum);
      }
    }
    constexpr int kS = kSum ? 3 : 0;
    unsigned long long pv[kS + kHeld];
    int at[kS + kHeld];
    if constexpr(kSum) {
#pragma unroll
      for(int j = 0; j < 3; ++j) at[j] = t < G ? a.oS + j * G + t : -1;
    }
#pragma unroll
    for(int k = 0; k < kHeld; ++k) at[kS + k] = hcl[k] >= 0 ? o + hcl[k] : -1;
    bool ok = resPoll<kS + kHeld>(buf, at, pv, wait);
#pragma unroll
    for(int k = 0; k < kHeld; ++k)
      if(hcl[k] >= 0) reg[L0.rows + t + k * kTB] = __longlong_as_double((long long)pv[kS + k]);
    for(int h = t + kHeld * kTB; h < hc0 && ok; h += kTB) {
      const int a1[1] = {o + hcol0[h]};
      unsigned long long v1[1];
      ok = resPoll<1>(buf, a1, v1, wait);
      reg[L0.rows + h] = __longlong_as_double((long long)v1[0]);
    }
    if(!ok) gaveUp = 1;
    if constexpr(kSum) {
      if(t < ((G + 63) & ~63)) {
#pragma unroll
        for(int j = 0; j < 3; ++j) {
          const double w = resWaveSum(t < G ? __longlong_as_double((long long)pv[j]) : 0.);
          if((t & 63) == 0) wsum[j][t >> 6] = w;
        }
      }
    }
    resBarrier();
    if(gaveUp) return false;
    if constexpr(kSum) {
#pragma unroll
      for(int j = 0; j < 3; ++j) {
        double w = 0.;
        for(int k = 0; k < (G + 63) / 64; ++k) w += wsum[j][k];
        f[j] = resUniform(w);
      }
    }
    return true;
  };
  using Yes = std::true_type;
  using No = std::false_type;
  // A times the exchanged vector, own rows; its values may be overwritten then
  auto product = [&](double (&y)[RPT]) {
    const double *reg = (const double *)(lds + a.lReg0);
#pragma unroll
    for(int i = 0; i < RPT; ++i) {
      double s = 0.;
#pragma unroll
      for(int e = 0; e < E / 2; ++e) {
        asm volatile("" : "+v"(ix[i][e]));  // unpacked here, not kept unpacked across the loop
        s += v[i][2 * e] * reg[ix[i][e] & 0xffffu];
        s += v[i][2 * e + 1] * reg[ix[i][e] >> 16];
      }
      y[i] = own[i] ? s : 0.;  // a position without a row reads whatever is there
    }
    resBarrier();
  };
  auto levelInfo = [&](int l) {
    const int4 v4 = info[l];
    return make_int4(__builtin_amdgcn_readfirstlane(v4.x), __builtin_amdgcn_readfirstlane(v4.y),
                     __builtin_amdgcn_readfirstlane(v4.z), 0);
  };
  // the own slots of set `set` are empty again
  auto reset = [&](int set) {
    unsigned long long *o = a.buf + (size_t)set * a.bufLen;
#pragma unroll
    for(int i = 0; i < RPT; ++i)
      if(send[i]) {
        const int row = rs0 + t + i * kTB;
        resStore(o + a.oZ + row, kSentinel);
        resStore(o + L0.oU + row, kSentinel);
        resStore(o + L0.oY + row, kSentinel);
      }
    if(t < 3) resStore(o + a.oS + t * G + wg, kSentinel);
    for(int l = 1; l < B; ++l) {
      const int4 in = levelInfo(l);
      const unsigned short *ags = (const unsigned short *)(lds + a.lv[l].lAgg);
      for(int i = t; i < in.y; i += kTB)
        if(ags[i] & kSentBit) {
          resStore(o + a.lv[l].oU + in.x + i, kSentinel);
          resStore(o + a.lv[l].oY + in.x + i, kSentinel);
        }
    }
    for(int c = t; c < pc; c += kTB) resStore(o + a.oParts + pb + c, kSentinel);
  };
  // a coarse level's region: own values are in it; the others' from slots o
  auto gatherL = [&](const ArDist &L, int o, int hc) -> bool {
    double *reg = (double *)(lds + L.lReg);
    const int *hcol = (const int *)(lds + L.lHc);
    bool ok = true;
    for(int h = t; h < hc && ok; h += kTB) {
      const int a1[1] = {o + hcol[h]};
      unsigned long long v1[1];
      ok = resPoll<1>(buf, a1, v1, wait);
      reg[L.rows + h] = __longlong_as_double((long long)v1[0]);
    }
    if(!ok) gaveUp = 1;
    resBarrier();
    return !gaveUp;
  };
  // sums of res over the own rows of each aggregate: b of the next level, with
  // u = l1 b published, or the parts of b_B
  auto restrictTo = [&](int l, const double *res) {
    const ArDist &L = a.lv[l];
    const unsigned short *as = (const unsigned short *)(lds + L.lAs);
    if(l + 1 < B) {
      const ArDist &N = a.lv[l + 1];
      const int4 in = levelInfo(l + 1);
      const float *l1s = (const float *)(lds + N.lL1);
      const unsigned short *ags = (const unsigned short *)(lds + N.lAgg);
      double *b = (double *)(lds + N.lB), *us = (double *)(lds + N.lU), *reg = (double *)(lds + N.lReg);
      for(int c = t; c < in.y; c += kTB) {
        const double s = ldsRange(res, as[c], as[c + 1]), u = (double)l1s[c] * s;
        if(ags[c] & kSentBit) resStore(buf + N.oU + in.x + c, u);
        b[c] = s;
        us[c] = u;
        reg[c] = u;
      }
    } else {
      for(int c = t; c < pc; c += kTB) resStore(buf + a.oParts + pb + c, ldsRange(res, as[c], as[c + 1]));
    }
  };

  for(int k = 0; alive; ++k) {
    buf = a.buf + (size_t)(k % kSets) * a.bufLen;
    const int nextSet = (k + 2) % kSets;
    double s[3] = {0., 0., 0.}, f[3], w[RPT], az[RPT], aw[RPT];
    if(iterating) {
      if(!(alive = exchange0(No{}, a.oZ, z, s, f))) break;
      product(az);
#pragma unroll
      for(int i = 0; i < RPT; ++i) {
        w[i] = (double)l1[i] * az[i];
        s[0] += own[i] ? r[i] * z[i] : 0.;
        s[1] += own[i] ? z[i] * az[i] : 0.;
        s[2] += r[i] * r[i];
      }
    } else {
      if(started) {
        // a segment has ended: its correction joins the solution, whose true residual this is
#pragma unroll
        for(int i = 0; i < RPT; ++i)
          if(own[i]) {
            x[i] += outer > 0 ? a.x[orig[i]] : 0.;
            a.x[orig[i]] = x[i];
          }
        if(!(alive = exchange0(No{}, a.oZ, x, s, f))) break;
        product(az);
#pragma unroll
        for(int i = 0; i < RPT; ++i) {
          r[i] = own[i] ? a.b[orig[i]] - az[i] : 0.;
          x[i] = 0.;
        }
        ++outer;
      }
#pragma unroll
      for(int i = 0; i < RPT; ++i) {
        w[i] = (double)l1[i] * r[i];
        s[2] += r[i] * r[i];
      }
    }
    resStoresDone();  // the resets of the previous round
    if(!(alive = exchange0(Yes{}, L0.oU, w, s, f))) break;
    product(aw);
    const double rr = f[2];
    bool vcycle = true;
    if(!iterating) {
      rn = resUniform(sqrt(rr));
      if(outer == 0) {
        bn = rn;
        target = resUniform(fmax(a.rtol * bn, a.atol));
        tol2 = resUniform(0.25 * target * target);
        if(bn == 0. || rn <= target) reason = 2;
        else if(a.maxit <= 0) reason = -3;
      } else {
        if(rn <= target) reason = 2;
        else if(!(rn == rn)) reason = -9;
        else if(breakdowns > 20) reason = -3;
        else if(rn / bn > a.dtol) reason = -4;
        else if(outer >= kResOuter) reason = kResLimit;
        else if(it >= a.maxit) reason = -3;
      }
      if(reason) break;
#pragma unroll
      for(int i = 0; i < RPT; ++i) {
        au[i] = aw[i];
        p[i] = q[i] = aq[i] = 0.;
      }
      first = iterating = started = true;
    } else {
      const double rho = f[0];
      bool stop = false;
      double alpha = 0., beta = 0.;
      if(!(rho > 0.) || !(rr == rr)) {
        ++breakdowns;
        stop = true;
      } else if((!first && rr <= tol2) || it >= a.maxit) {
        stop = true;
      } else {
        beta = first ? 0. : resUniform(rho / rhoOld);
        const double den = resUniform(first ? f[1] : f[1] - beta * rho / alphaOld);  // (p, A p)
        if(den > 0.) {
          alpha = resUniform(rho / den);
        } else {
          ++breakdowns;
          stop = true;
        }
      }
      if(stop) {
        iterating = false;
        vcycle = false;
      } else {
        rhoOld = rho;
        alphaOld = alpha;
#pragma unroll
        for(int i = 0; i < RPT; ++i) {
          p[i] = __builtin_fma(beta, p[i], z[i]);
          q[i] = __builtin_fma(beta, q[i], az[i]);
          aq[i] = __builtin_fma(beta, aq[i], aw[i]);
          x[i] = __builtin_fma(alpha, p[i], x[i]);
          r[i] = __builtin_fma(-alpha, q[i], r[i]);
          au[i] = __builtin_fma(-alpha, aq[i], au[i]);
        }
        ++it;
        first = false;
      }
    }
    if(!vcycle) {
      reset(nextSet);
      continue;
    }
    // --- V-cycle: down
    {
      double *res = (double *)(lds + a.lReg0);
#pragma unroll
      for(int i = 0; i < RPT; ++i)
        if(own[i]) res[t + i * kTB] = r[i] - au[i];
      resBarrier();
      restrictTo(0, res);
    }
    reset(nextSet);  // while the published values travel
    for(int l = 1; l < B; ++l) {
      const ArDist &L = a.lv[l];
      const double *b = (const double *)(lds + L.lB);
      double *es = (double *)(lds + L.lE);
      const int4 in = levelInfo(l);
      if(!(alive = gatherL(L, L.oU, in.z))) break;
      ldsRows(in.y, (const unsigned short *)(lds + L.lOff), (const unsigned short *)(lds + L.lIdx),
              (const float *)(lds + L.lVal), (const double *)(lds + L.lReg),
              [&](int i, double acc) { es[i] = b[i] - acc; });
      resBarrier();
      restrictTo(l, es);
    }
    if(!alive) break;
    // --- levels B .. coarsest, in every workgroup
    {
      double *parts = (double *)(lds + a.blk.lParts), *b = (double *)(lds + a.blk.lB[0]);
      double *u = (double *)(lds + (a.blk.nLev > 0 ? a.blk.lU[0] : a.blk.lParts));
      const float *l1s = (const float *)(lds + a.blk.lImg + a.blk.oL1[0]);
      const unsigned short *ps = (const unsigned short *)(lds + a.blk.lImg + a.blk.oPs);
      bool ok = true;
      for(int i = t; i < a.parts && ok; i += 2 * kTB) {
        const int a2[2] = {a.oParts + i, i + kTB < a.parts ? a.oParts + i + kTB : -1};
        unsigned long long v2[2];
        ok = resPoll<2>(buf, a2, v2, wait);
        parts[i] = __longlong_as_double((long long)v2[0]);
        if(i + kTB < a.parts) parts[i + kTB] = __longlong_as_double((long long)v2[1]);
      }
      if(!ok) gaveUp = 1;
      resBarrier();
      if(gaveUp) {
        alive = false;
        break;
      }
      for(int i = t; i < a.blk.n[0]; i += kTB) {
        const double sum = ldsRange(parts, ps[i], ps[i + 1]);
        b[i] = sum;
        if(a.blk.nLev > 0) u[i] = (double)l1s[i] * sum;
      }
      resBarrier();
      arBlockSolve(a.blk, lds, a.oc);
    }
    // --- up
    const double *en = (const double *)(lds + (a.blk.nLev > 0 ? a.blk.lB[0] : a.blk.lX));
    for(int l = B - 1; l >= 1; --l) {
      const ArDist &L = a.lv[l];
      const int4 in = levelInfo(l);
      const float *l1s = (const float *)(lds + L.lL1);
      const unsigned short *ags = (const unsigned short *)(lds + L.lAgg);
      const double *b = (const double *)(lds + L.lB), *us = (const double *)(lds + L.lU);
      double *es = (double *)(lds + L.lE), *reg = (double *)(lds + L.lReg);
      for(int i = t; i < in.y; i += kTB) {
        const int ag1 = ags[i];
        const double y = __builtin_fma(a.oc, en[ag1 & (kSentBit - 1)], us[i]);
        if(ag1 & kSentBit) resStore(buf + L.oY + in.x + i, y);
        reg[i] = y;
      }
      if(!(alive = gatherL(L, L.oY, in.z))) break;
      ldsRows(in.y, (const unsigned short *)(lds + L.lOff), (const unsigned short *)(lds + L.lIdx),
              (const float *)(lds + L.lVal), reg,
              [&](int i, double acc) { es[i] = __builtin_fma((double)l1s[i], b[i] - acc, reg[i]); });
      resBarrier();
      en = es;
    }
    if(!alive) break;
    double y0[RPT];
#pragma unroll
    for(int i = 0; i < RPT; ++i) y0[i] = own[i] ? __builtin_fma(a.oc, en[ag[i]], (double)l1[i] * r[i]) : 0.;
    if(!(alive = exchange0(No{}, L0.oY, y0, s, f))) break;
    product(az);
#pragma unroll
    for(int i = 0; i < RPT; ++i) z[i] = __builtin_fma((double)l1[i], r[i] - az[i], y0[i]);
  }
  if(t == 0) {
    if(gaveUp) __hip_atomic_store(&a.out->gaveUp, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if(wg == 0) {
      a.out->ended = 1;
      a.out->reason = reason == kResLimit ? 0 : reason;
      a.out->iters = it;
      a.out->outer = outer;
      a.out->badPivot = *a.badPivot;
      a.out->bn = bn;
      a.out->rn = rn;
    }
  }
  double mx[3] = {0., 0., 0.};
#pragma unroll
  for(int i = 0; i < RPT; ++i)
    if(own[i]) {
      if(outer == 0) a.x[orig[i]] = 0.;
      mx[0] = fmax(mx[0], fabs(a.x[orig[i]]));
      mx[1] = fmax(mx[1], fabs(a.b[orig[i]]));
      mx[2] = fmax(mx[2], fabs(r[i]));
    }
  resBarrier();
#pragma unroll
  for(int j = 0; j < 3; ++j) {
#pragma unroll
    for(int o = 32; o > 0; o >>= 1) mx[j] = fmax(mx[j], __shfl_xor(mx[j], o, 64));
    if((t & 63) == 0) psum[j][t >> 6] = mx[j];
  }
  resBarrier();
  if(t < 3) {
    double mm = 0.;
    for(int k = 0; k < kTB / 64; ++k) mm = fmax(mm, psum[t][k]);
    a.maxima[3 * wg + t] = mm;
  }
}

template <typename T>
int upload(fe_hip_ctx *ctx, T **d, const std::vector<T> &h)
{
  if(int rc = feAlloc(ctx, d, std::max<size_t>(1, h.size()))) return rc;
  if(!h.empty()) FE_HIP_TRY(ctx, hipMemcpy(*d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice));
  return FE_STATUS_OK;
}

}  // namespace

struct FeAmgResident {
  bool built = false, usable = false;
  int RPT = 0, E = 0, lds = 0;
  ArArgs args{};
  ArPackArgs pack{};
  unsigned char *img = nullptr;
  ArOut *d_out = nullptr, *h_out = nullptr;
};

namespace {

// Cuts the rows of the last distributed level so that no workgroup has more
// than `limit` level-0 rows (start[j]: first level-0 row of level row j).
std::vector<int> arCut(const std::vector<int> &start, int limit)
{
  std::vector<int> cut(1, 0);
  const int m = (int)start.size() - 1;
  for(int j = 0; j < m; ++j)
    if(start[j + 1] - start[cut.back()] > limit) {
      if(cut.back() == j) return {};  // one row is too large
      cut.push_back(j);
      if(start[j + 1] - start[j] > limit) return {};
    }
  cut.push_back(m);
  return cut;
}

int arBuild(fe_hip_ctx *ctx, const FeNestedView &V, FeAmgResident &R)
{
  R.built = true;
  const int Lc = (int)V.lv.size() - 1, n = ctx->n;
  int cus = 0;
  FE_HIP_TRY(ctx, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
  cus = std::min(cus, 256);
  int longest = 0;
  for(int i = 0; i < n; ++i) longest = std::max(longest, ctx->amgHost[0].ia[i + 1] - ctx->amgHost[0].ia[i]);
  if(n > cus * 1024 || longest > 24) return FE_STATUS_OK;
  R.E = longest <= 8 ? 8 : longest <= 16 ? 16 : 24;
  const int maxRows = 2 * kTB;
  std::vector<std::vector<int>> as(Lc);  // first row of each aggregate
  for(int l = 0; l < Lc; ++l) {
    as[l].resize(V.lv[l].nc + 1);
    FE_HIP_TRY(ctx, hipMemcpy(as[l].data(), V.lv[l].aggStart, sizeof(int) * as[l].size(), hipMemcpyDeviceToHost));
  }
  const int Bmax = std::min(Lc, kMaxDist);
  for(int c = 0; c < 2 * Bmax; ++c) {
    const int B = c % Bmax + 1, limit = kArBlockRows[c / Bmax];
    if(V.lv[B].n > limit || Lc - B > kMaxBlk) continue;
    // level-0 start of every row of level B - 1
    std::vector<int> start(V.lv[B - 1].n + 1);
    for(int j = 0; j <= V.lv[B - 1].n; ++j) {
      int i = j;
      for(int l = B - 2; l >= 0; --l) i = as[l][i];
      start[j] = i;
    }
    // workgroups: as few as hold kArRows rows each, all of the device at most;
    // the lowest limit that needs no more
    const int want = std::max(1, std::min(cus, (n + kArRows - 1) / kArRows));
    int lo = (n + want - 1) / want, hi = maxRows;
    std::vector<int> cut = arCut(start, hi);
    if(cut.empty() || (int)cut.size() - 1 > cus) continue;
    const int most = std::max(want, (int)cut.size() - 1);
    while(lo < hi) {
      const int mid = (lo + hi) / 2;
      std::vector<int> c = arCut(start, mid);
      if(!c.empty() && (int)c.size() - 1 <= most) {
        hi = mid;
        cut.swap(c);
      } else {
        lo = mid + 1;
      }
    }
    const int G = (int)cut.size() - 1;
    ArArgs A{};
    A.n = n;
    A.G = G;
    A.B = B;
    // row ranges, parts of b_B
    std::vector<std::vector<int>> rs(B);
    rs[B - 1] = cut;
    for(int l = B - 2; l >= 0; --l) {
      rs[l].resize(G + 1);
      for(int g = 0; g <= G; ++g) rs[l][g] = as[l][rs[l + 1][g]];
    }
    const int nB = V.lv[B].n;
    std::vector<int> partBase(1, 0), partFirst;
    std::vector<unsigned short> ps(nB + 1, 0);
    {
      std::vector<int> cnt(nB + 1, 0);
      for(int g = 0; g < G; ++g) {
        const int f = (int)(std::upper_bound(as[B - 1].begin(), as[B - 1].end(), cut[g]) - as[B - 1].begin()) - 1;
        const int e = (int)(std::upper_bound(as[B - 1].begin(), as[B - 1].end(), cut[g + 1] - 1) - as[B - 1].begin()) - 1;
        partFirst.push_back(f);
        partBase.push_back(partBase.back() + e - f + 1);
        for(int I = f; I <= e; ++I) cnt[I + 1]++;
      }
      for(int I = 0; I < nB; ++I) cnt[I + 1] += cnt[I];
      for(int I = 0; I <= nB; ++I) ps[I] = (unsigned short)cnt[I];
    }
    A.parts = partBase.back();
    if(A.parts > 4096 || G > 256) continue;
    int rows0 = 0;
    for(int g = 0; g < G; ++g) rows0 = std::max(rows0, rs[0][g + 1] - rs[0][g]);
    const int RPT = rows0 <= kTB ? 1 : 2, TB = RPT * kTB;
    // gathered rows per level (device), LDS positions of the columns
    int *d_flag = nullptr;
    if(feAlloc(ctx, &d_flag, kMaxDist)) return FE_STATUS_OUT_OF_MEMORY;
    FE_HIP_TRY(ctx, hipMemsetAsync(d_flag, 0, kMaxDist * sizeof(int), ctx->stream));
    unsigned *idx0 = nullptr;
    std::vector<int> rowsMax(B), entMax(B, 0), hcap(B);
    std::vector<void *> mine;  // freed when this B does not fit
    for(int l = 0; l < B; ++l) {
      ArDist &D = A.lv[l];
      const FeNestedLevel &L = V.lv[l];
      for(int g = 0; g < G; ++g) rowsMax[l] = std::max(rowsMax[l], rs[l][g + 1] - rs[l][g]);
      hcap[l] = std::min(l == 0 ? 8192 : 4096, L.n);
      int *drs = nullptr, *hcol = nullptr, *hcnt = nullptr;
      unsigned short *lidx = nullptr;
      if(upload(ctx, &drs, rs[l]) || feAlloc(ctx, &hcol, (size_t)G * hcap[l]) || feAlloc(ctx, &hcnt, G))
        return FE_STATUS_OUT_OF_MEMORY;
      mine.insert(mine.end(), {drs, hcol, hcnt});
      if(l == 0) {
        if(feAlloc(ctx, &idx0, (size_t)G * (R.E / 2) * TB)) return FE_STATUS_OUT_OF_MEMORY;
        mine.push_back(idx0);
        hipLaunchKernelGGL(arPattern<true>, dim3(G), dim3(1024), 0, ctx->stream, L.n, drs, rowsMax[l], R.E, TB, hcap[l],
                           L.sell, (const int *)nullptr, L.ja, (unsigned short *)idx0, hcol, hcnt, d_flag + l);
      } else {
        if(feAlloc(ctx, &lidx, (size_t)L.nnz)) return FE_STATUS_OUT_OF_MEMORY;
        mine.push_back(lidx);
        hipLaunchKernelGGL(arPattern<false>, dim3(G), dim3(1024), 0, ctx->stream, L.n, drs, rowsMax[l], 0, 0, hcap[l],
                           (const int2 *)nullptr, L.ia, L.ja, lidx, hcol, hcnt, d_flag + l);
        std::vector<int> ia(L.n + 1);
        FE_HIP_TRY(ctx, hipMemcpy(ia.data(), L.ia, sizeof(int) * ia.size(), hipMemcpyDeviceToHost));
        for(int g = 0; g < G; ++g) entMax[l] = std::max(entMax[l], ia[rs[l][g + 1]] - ia[rs[l][g]]);
      }
      unsigned char *sent = nullptr;
      if(feAlloc(ctx, &sent, (size_t)L.n)) return FE_STATUS_OUT_OF_MEMORY;
      mine.push_back(sent);
      FE_HIP_TRY(ctx, hipMemsetAsync(sent, 0, (size_t)L.n, ctx->stream));
      hipLaunchKernelGGL(arSent, dim3(G), dim3(256), 0, ctx->stream, hcol, hcnt, hcap[l], sent);
      D.sent = sent;
      D.rs = drs;
      D.ia = L.ia;
      D.lidx = lidx;
      D.val = L.val32;
      D.l1 = L.l1_32;
      D.agg = L.agg;
      D.aggStart = L.aggStart;
      D.hcol = hcol;
      D.hcnt = hcnt;
      D.n = L.n;
      D.rows = rowsMax[l];
      D.hcap = hcap[l];
    }
    FE_HIP_TRY(ctx, hipGetLastError());
    int hmax[kMaxDist];
    FE_HIP_TRY(ctx, hipMemcpyAsync(hmax, d_flag, sizeof(hmax), hipMemcpyDeviceToHost, ctx->stream));
    FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    feFree(ctx, d_flag);
    bool ok = true;
    for(int l = 0; l < B; ++l) ok = ok && hmax[l] <= hcap[l] && rowsMax[l] + hmax[l] < 65536 && entMax[l] < 65536;
    // LDS plan
    int bytes = 0;
    auto take = [&](size_t b) {
      const int o = bytes;
      bytes += (int)std::min<size_t>((b + 15) & ~(size_t)15, 1 << 20);
      return o;
    };
    ArBlock &K = A.blk;
    ArPackArgs &P = R.pack;
    P = ArPackArgs{};
    K.nLev = Lc - B;
    {
      int ib = 0;
      auto img = [&](size_t b) {
        const int o = ib;
        ib += (int)((b + 15) & ~(size_t)15);
        return o;
      };
      P.nLev = K.nLev;
      for(int s = 0; s < K.nLev; ++s) {
        const FeNestedLevel &L = V.lv[B + s];
        ok = ok && L.nnz < 65536;
        K.n[s] = L.n;
        K.nc[s] = L.nc;
        K.nnz[s] = (int)L.nnz;
        K.oIa[s] = img(2 * (size_t)(L.n + 1));
        K.oJa[s] = img(2 * (size_t)L.nnz);
        K.oVal[s] = img(4 * (size_t)L.nnz);
        K.oL1[s] = img(4 * (size_t)L.n);
        K.oAgg[s] = img(2 * (size_t)L.n);
        K.oAs[s] = img(2 * (size_t)(L.nc + 1));
        P.lv[s] = ArPackLevel{L.n, L.nc, (int)L.nnz, K.oIa[s], K.oJa[s], K.oVal[s], K.oL1[s], K.oAgg[s], K.oAs[s],
                              L.ia, L.ja, L.agg, L.aggStart, L.val32, L.l1_32};
      }
      K.n[K.nLev] = V.lv[Lc].n;
      P.nC = V.lv[Lc].n;
      P.cinv = V.cinv;
      K.oCi = P.oCi = img(8 * (size_t)P.nC * P.nC);
      K.oPs = img(2 * (size_t)(nB + 1));
      K.bytes = ib;
    }
    K.lImg = take(K.bytes);
    for(int s = 0; s < K.nLev; ++s) {
      K.lB[s] = take(8 * (size_t)K.n[s]);
      K.lU[s] = take(8 * (size_t)K.n[s]);
    }
    K.lB[K.nLev] = take(8 * (size_t)K.n[K.nLev]);
    K.lX = take(8 * (size_t)K.n[K.nLev]);
    K.lParts = take(8 * (size_t)std::max(A.parts, nB));
    A.lReg0 = take(8 * (size_t)(rowsMax[0] + hmax[0]));
    for(int l = 0; l < B; ++l) {
      ArDist &D = A.lv[l];
      const int coarse = l + 1 < B ? rowsMax[l + 1] : [&] {
        int c = 0;
        for(int g = 0; g < G; ++g) c = std::max(c, partBase[g + 1] - partBase[g]);
        return c;
      }();
      D.lAs = take(2 * (size_t)(coarse + 1));
      if(l == 0) continue;
      D.lReg = take(8 * (size_t)(rowsMax[l] + hmax[l]));
      D.lHc = take(4 * (size_t)std::max(1, hmax[l]));
      D.lB = take(8 * (size_t)rowsMax[l]);
      D.lU = take(8 * (size_t)rowsMax[l]);
      D.lE = take(8 * (size_t)rowsMax[l]);
      D.lVal = take(4 * (size_t)entMax[l]);
      D.lIdx = take(2 * (size_t)entMax[l]);
      D.lOff = take(2 * (size_t)(rowsMax[l] + 1));
      D.lL1 = take(4 * (size_t)rowsMax[l]);
      D.lAgg = take(2 * (size_t)rowsMax[l]);
    }
    if(!ok || bytes > kArLds) {
      for(void *m : mine) feFree(ctx, m);
      continue;
    }
    // exchange buffer
    size_t w = 0;
    auto words = [&](size_t c) {
      const size_t o = w;
      w += (c + 7) & ~(size_t)7;
      return (int)o;
    };
    A.oZ = words(n);
    A.lv[0].oU = words(n);
    A.lv[0].oY = words(n);
    for(int l = 1; l < B; ++l) {
      A.lv[l].oU = words(V.lv[l].n);
      A.lv[l].oY = words(V.lv[l].n);
    }
    A.oS = words(3 * (size_t)G);
    A.oParts = words(A.parts);
    A.bufLen = w;
    int *dpb = nullptr, *dpf = nullptr;
    if(upload(ctx, &dpb, partBase) || upload(ctx, &dpf, partFirst) || feAlloc(ctx, &A.buf, kSets * w) ||
       feAlloc(ctx, &R.img, std::max(16, K.bytes)) ||
       feAlloc(ctx, (char **)&R.d_out, sizeof(ArOut) + 3 * sizeof(double) * G))
      return FE_STATUS_OUT_OF_MEMORY;
    FE_HIP_TRY(ctx, hipMemcpy(R.img + K.oPs, ps.data(), 2 * ps.size(), hipMemcpyHostToDevice));
    FE_HIP_TRY(ctx, hipHostMalloc((void **)&R.h_out, sizeof(ArOut) + 3 * sizeof(double) * G));
    P.img = R.img;
    A.sell = V.lv[0].sell;
    A.val0 = V.lv[0].valD;
    A.idx0 = idx0;
    A.perm = V.perm;
    A.partBase = dpb;
    A.partFirst = dpf;
    A.img = R.img;
    A.badPivot = V.flag;
    A.out = R.d_out;
    A.maxima = (double *)(R.d_out + 1);
    R.args = A;
    R.RPT = RPT;
    R.lds = bytes;
    R.usable = true;
    return FE_STATUS_OK;
  }
  return FE_STATUS_OK;
}

template <int RPT, int E>
int launchAr(fe_hip_ctx *ctx, const FeAmgResident &R, const ArArgs &a, bool *fits)
{
  const void *f = (const void *)arSolve<RPT, E>;
  int perCu = 0, cus = 0;
  std::lock_guard<std::mutex> lock(feResidentGate(ctx->device).launching());
  *fits = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, R.lds) == hipSuccess &&
          hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, f, kTB, R.lds) == hipSuccess &&
          hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) == hipSuccess &&
          perCu * cus >= a.G;
  if(!*fits) {
    (void)hipGetLastError();
    return FE_STATUS_OK;
  }
  hipLaunchKernelGGL((arSolve<RPT, E>), dim3(a.G), dim3(kTB), R.lds, ctx->stream, a);
  FE_HIP_TRY(ctx, hipGetLastError());
  return FE_STATUS_OK;
}

}  // namespace

int feAmgResidentSolve(fe_hip_ctx *ctx, const fe_hip_solver_opts *o, double *x, FeResidentResult *res)
{
  res->ran = false;
  if(!ctx->resident || ctx->residentGaveUp || !ctx->pcValues32 || ctx->amgWcycle || ctx->amgFuse) return FE_STATUS_OK;
  if(ctx->amgRes && ctx->amgRes->built && !ctx->amgRes->usable) return FE_STATUS_OK;
  FeNestedView V;
  if(int rc = feAmgNestedPrepare(ctx, &V)) return rc;
  if(!ctx->amgRes) ctx->amgRes = new FeAmgResident();
  FeAmgResident &R = *ctx->amgRes;
  if(!R.built)
    if(int rc = arBuild(ctx, V, R)) return rc;
  if(!R.usable) return FE_STATUS_OK;
  hipLaunchKernelGGL(arPack, dim3(8, R.pack.nLev + 1), dim3(256), 0, ctx->stream, R.pack);
  ArArgs a = R.args;
  a.b = ctx->d_rhs;
  a.x = x;
  a.rtol = o->rtol;
  a.atol = o->atol;
  a.dtol = o->dtol;
  a.oc = ctx->amgOverCorrect;
  a.maxit = std::min(o->max_iter, ctx->residentMaxIter);
  a.wait = resWaitTicks(ctx);
  bool fits = false;
  {
    const FeResidentPass pass(ctx, a.G);
    const size_t cells = kSets * a.bufLen;
    hipLaunchKernelGGL(arFill, dim3((unsigned)std::min<size_t>(1024, (cells + 255) / 256)), dim3(256), 0, ctx->stream,
                       cells, a.buf, a.out);
    if(ctx->profiling)
      if(int rc = feTimerMark(ctx, ctx->iterTimer)) return rc;
    int rc = FE_STATUS_OK;
    if(R.RPT == 1) {
      if(R.E == 8) rc = launchAr<1, 8>(ctx, R, a, &fits);
      else if(R.E == 16) rc = launchAr<1, 16>(ctx, R, a, &fits);
      else rc = launchAr<1, 24>(ctx, R, a, &fits);
    } else {
      if(R.E == 8) rc = launchAr<2, 8>(ctx, R, a, &fits);
      else if(R.E == 16) rc = launchAr<2, 16>(ctx, R, a, &fits);
      else rc = launchAr<2, 24>(ctx, R, a, &fits);
    }
    if(rc) return rc;
    if(fits) {
      if(ctx->profiling)
        if(int rc2 = feTimerMark(ctx, ctx->iterTimer)) return rc2;
      FE_HIP_TRY(ctx, hipMemcpyAsync(R.h_out, R.d_out, sizeof(ArOut) + 3 * sizeof(double) * a.G, hipMemcpyDeviceToHost,
                                     ctx->stream));
    }
    FE_HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  }
  if(!fits) {
    ctx->iterTimer.used = 0;
    R.usable = false;
    return FE_STATUS_OK;
  }
  const ArOut &out = *R.h_out;
  if(out.gaveUp || !out.ended) {  // a wait ran out: the other kernels take over
    ctx->iterTimer.used = 0;
    ctx->residentGaveUp = true;
    return FE_STATUS_OK;
  }
  if(resCutShort(ctx, o, out.iters, out.reason)) {
    ctx->iterTimer.used = 0;
    return FE_STATUS_OK;
  }
  FE_REQUIRE(ctx, out.bn == 0. || !out.badPivot, "AMG: the coarsest operator is not positive definite");
  res->ran = ctx->residentRan = true;
  res->reason = out.reason;
  res->iters = out.iters;
  res->outer = out.outer;
  res->relres = out.bn == 0. ? 0. : out.rn / out.bn;  // not a number stays that
  const double *mx = (const double *)(R.h_out + 1);
  for(int k = 0; k < 3; ++k) res->inf[k] = 0.;
  for(int k = 0; k < 3 * a.G; ++k) res->inf[k % 3] = std::max(res->inf[k % 3], mx[k]);
  if(ctx->profiling) {  // the launch's time over its iterations, as the dominant kernel and as the iteration
    float ms = 0.f;
    FeKernelTimer &t = ctx->iterTimer;
    FE_HIP_TRY(ctx, hipEventElapsedTime(&ms, t.ev[t.used - 2], t.ev[t.used - 1]));
    t.used = 0;
    for(FeKernelTimer *q : {&ctx->iterTimer, &ctx->spmvTimer}) {
      q->total_ms += ms;
      q->launches += std::max(1, out.iters);
    }
  }
  return FE_STATUS_OK;
}

void feAmgResidentRelease(fe_hip_ctx *ctx)
{
  if(ctx->amgRes && ctx->amgRes->h_out) (void)hipHostFree(ctx->amgRes->h_out);
  delete ctx->amgRes;  // device buffers are owned by the context
  ctx->amgRes = nullptr;
}
