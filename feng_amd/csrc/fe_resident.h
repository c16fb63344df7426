// Building blocks of the resident Krylov kernels: one launch runs all
// iterations of a solve, every workgroup keeps its rows' matrix entries and
// vectors in registers and LDS, and workgroups exchange only what others need
// (boundary values of the gathered vector, partial sums) through memory.
//
// Exchange.  No grid barrier and no fence: every exchanged 8-byte word is
// stored and loaded with device-scope relaxed atomics (write-through past the
// per-XCD L2), and a word's arrival is the word itself -- a slot holds a
// sentinel (a signalling NaN no arithmetic produces) until its value is
// stored, and readers poll the slot.  So an exchange costs one store-to-load
// trip, without a flag store ordered behind the data.  Exchange q uses buffer
// q mod 4; while workgroups run between exchanges q and q + 1 the owner of a
// slot puts the sentinel back into buffer (q + 2) mod 4: every workgroup has
// left exchange q - 1 by then (its partial sums of exchange q were received),
// and the reset is complete (vmcnt 0) before the owner publishes its part of
// exchange q + 1, which any workgroup receives before it polls exchange q + 2.
//
// Every wait is bounded by wall time (50 ms, tuning key resident_wait_us): a
// workgroup that gives up raises a flag and leaves, later waits of the launch
// give up the same way, and the host repeats the solve with the
// launch-per-iteration kernels.
// All workgroups of a launch must be resident together: the host checks the
// occupancy and admits to a device what fits it together (fe_resident_gate.h).
#pragma once

#include "fe_hip_internal.h"
#include "fe_resident_gate.h"

// Of a device.
FeResidentGate &feResidentGate(int device);

// Held from a resident launch of G workgroups to its end.
class FeResidentPass {
 public:
  FeResidentPass(fe_hip_ctx *ctx, int G) : gate_(feResidentGate(ctx->device))
  {
    int cus = 0;
    if(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device) != hipSuccess) cus = 0;
    need_ = feGateNeed(G, cus);
    // others wait, or are waited for: not inside for this stream's earlier work
    if(gate_.busy()) (void)hipStreamSynchronize(ctx->stream);
    gate_.enter(need_, kGateCus);
  }
  ~FeResidentPass() { gate_.leave(need_); }
  FeResidentPass(const FeResidentPass &) = delete;
  FeResidentPass &operator=(const FeResidentPass &) = delete;

 private:
  FeResidentGate &gate_;
  int need_;
};

namespace fe_res {

constexpr unsigned long long kSentinel = 0x7FF4DEAD5EA7F00Dull;
constexpr int kResBufs = 4;
// Most solves from a true residual (the launch-per-iteration loops of refined,
// split and multigrid solves have the same bound); a target below the floor of
// FP64 would otherwise be tried until the iteration budget ends.  A solve that
// stops there has no reason code (0): kResLimit inside a kernel.
constexpr int kResOuter = 60;
constexpr int kResLimit = 100;

__device__ __forceinline__ unsigned long long resLoad(const unsigned long long *p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void resStore(unsigned long long *p, unsigned long long v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void resStore(unsigned long long *p, double v) { resStore(p, (unsigned long long)__double_as_longlong(v)); }

// Orders the LDS accesses of the workgroup; global accesses stay in flight.
__device__ __forceinline__ void resBarrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// Every global store of this wavefront has reached its coherence point.
__device__ __forceinline__ void resStoresDone() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The longest wait of a launch, in ticks of the 100 MHz counter; 0 us: no wait
// at all, give up on the first value that has not arrived.
inline int resWaitTicks(const fe_hip_ctx *ctx) { return ctx->residentWaitUs > 0 ? 100 * ctx->residentWaitUs : -1; }

// A solve that the iteration limit of a launch has cut short of its own budget:
// the launches per iteration repeat it.
inline bool resCutShort(const fe_hip_ctx *ctx, const fe_hip_solver_opts *o, int iters, int reason)
{
  return o->max_iter > ctx->residentMaxIter && iters >= ctx->residentMaxIter && reason != 2;
}

// Polls the K slots base[idx[k]] (idx < 0: none) until all have arrived; false
// when the time (ticks, in LDS: scalar registers are short) is up.  The loads
// of a round are issued together.
template <int K>
__device__ __forceinline__ bool resPoll(const unsigned long long *base, const int (&idx)[K], unsigned long long (&v)[K],
                                        const int &ticks)
{
#pragma unroll
  for(int k = 0; k < K; ++k) v[k] = idx[k] >= 0 ? resLoad(base + (unsigned)idx[k]) : 0ull;
  bool all = true;
#pragma unroll
  for(int k = 0; k < K; ++k) all = all && v[k] != kSentinel;
  if(all) return true;
  const long long t0 = wall_clock64();
  for(;;) {
    all = true;
#pragma unroll
    for(int k = 0; k < K; ++k)
      if(v[k] == kSentinel) {
        v[k] = resLoad(base + (unsigned)idx[k]);
        all = all && v[k] != kSentinel;
      }
    if(all) return true;
    if(wall_clock64() - t0 > ticks) return false;
  }
}

// Sum of one value per lane of a wavefront, in every lane, in a fixed order
// (data-parallel primitives, no LDS): quads, halves of a row of 16, rows, then
// the row sums passed on to the next row and the upper half.
template <int CTRL>
__device__ __forceinline__ double dppMove(double v)
{
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffull), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)((unsigned long long)(unsigned)lo | (unsigned long long)(unsigned)hi << 32));
}
__device__ __forceinline__ double resReadLane(double v, int lane)
{
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffull), lane);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double((long long)((unsigned long long)(unsigned)lo | (unsigned long long)(unsigned)hi << 32));
}
// A value that all lanes hold, in scalar registers.
__device__ __forceinline__ double resUniform(double v) { return resReadLane(v, 0); }
__device__ __forceinline__ double resWaveSum(double v)
{
  v += dppMove<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v += dppMove<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v += dppMove<0x141>(v);  // row_half_mirror
  v += dppMove<0x140>(v);  // row_mirror: every lane has its row's sum
  return (resReadLane(v, 0) + resReadLane(v, 16)) + (resReadLane(v, 32) + resReadLane(v, 48));
}

}  // namespace fe_res
