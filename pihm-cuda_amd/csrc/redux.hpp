// redux.hpp - element-wise operation fused with NV deterministic sums.
//
// Each workgroup accumulates NV partial sums over a fixed strided set of
// entries (wavefront butterfly, then the four waves in order) and writes
// them; the second pass adds each slot's partials (per thread in workgroup
// order, wavefront butterfly, waves in order) and writes the NV results to
// pinned host memory.  The summation tree depends only on the length, so every
// result is reproducible bit for bit.
//
// The second pass is a launch of its own, or, where a reduction has at most
// kTicketBlocks workgroups, the work of the workgroup that finishes last: each
// stores its partials as agent-scope atomics (coherent across the XCDs), waits
// for the stores and takes a ticket.  No fence writes back an L2: the results
// go to coherent host memory, ordered by waiting for the stores.
//
// Both passes are bound by latency.  The second pass took 5.7 us a launch in
// the 200,000-triangle run with one slot's butterfly after the other through
// the LDS, 2.8-3.7 us with the slots in step and lane moves (lanes.hpp).
//
// The line at 64 workgroups (32,768 entries) is on the safe side.  A dot product
// and the Arnoldi step's six sums, from the call to the result (us, two launches
// / one), by workgroups:
//     36: 11.3 / 9.3, 13.9 / 12.3     64: 11.3 / 9.5, 14.1 / 12.4
//    119: 11.4 / 10.0, 14.0 / 12.9   160: 11.3 / 10.5, 14.1 / 13.4
//    256: 11.4 / 11.6, 14.2 / 14.6   512: 11.3 / 14.7, 14.7 / 17.5
//   1024: 11.4 / 20.7, 16.4 / 24.2
// Every further workgroup's ticket waits its turn at one address, about 10 ns
// each: the single launch is ahead up to some 200 workgroups, and whole runs say
// the same (20,011 triangles, 119 workgroups: 25.5 / 23.1 ms for 12 minutes;
// 60,000, 355: 21.6 / 21.7 for 8; 200,000, 1,024: 10.1 / 11.9 for 4).
#pragma once
#include <hip/hip_runtime.h>
#include <cfloat>
#include "common.hpp"
#include "lanes.hpp"
#include "nvector_impl.hpp"

namespace pihm {

constexpr int kRedThreads = 256;

inline int fused_blocks(long n) {
  long b = (n + 2L * kRedThreads - 1) / (2L * kRedThreads);
  if (b < 1) b = 1;
  if (b > PIHM_RED_MAXBLOCKS) b = PIHM_RED_MAXBLOCKS;
  return (int)b;
}

// How the second pass combines the partials of slot k: 2 bits per slot.
enum : unsigned { COMB_SUM = 0u, COMB_MIN = 1u, COMB_MAX = 2u };

__device__ __forceinline__ double comb_ident(unsigned c) {
  return c == COMB_MIN ? DBL_MAX : 0.0;
}
__device__ __forceinline__ double comb(unsigned c, double a, double b) {
  return c == COMB_MIN ? fmin(a, b) : (c == COMB_MAX ? fmax(a, b) : a + b);
}
__device__ __forceinline__ double wave_comb(unsigned c, double v) {
  return c == COMB_MIN ? wave_min(v) : (c == COMB_MAX ? wave_max(v) : wave_sum(v));
}

// Workgroups up to which a reduction ends in its own launch (the last
// workgroup's second pass).
constexpr int kTicketBlocks = PIHM_RED_TICKETS;

// Waits for this wavefront's outstanding stores (and loads).
__device__ __forceinline__ void wait_memory() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ void store_partial(double *p, double v, bool shared) {
  if (shared) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

// True in every thread of the workgroup that takes the last of nb tickets.
// Called by all threads after wavefront 0 stored the workgroup's partials.
__device__ __forceinline__ bool last_workgroup(unsigned *ticket, int nb) {
  __shared__ int last;
  if (threadIdx.x == 0) {
    wait_memory();
    const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = t == (unsigned)(nb - 1);
    if (last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next reduction
  }
  __syncthreads();
  return last;
}

// Second pass by one workgroup: every thread loads its partials of all NV
// slots (workgroups t, t+256, t+512, t+768) before combining any, so it waits
// for one round of memory latency; the slots' butterflies then run in step.
// Each slot is combined in the fixed order thread (ascending workgroup),
// wavefront butterfly, waves in order.  Optionally stores one extra scalar
// (xstore) for kernels that follow on the stream.
template <int NV, unsigned COMBS, bool SHARED>
__device__ __forceinline__ void second_pass(int nb, const double *partials, double *result, double *devcopy,
                                            unsigned *ctr, volatile unsigned *flag, double *xstore, double xval) {
  constexpr int kPer = PIHM_RED_MAXBLOCKS / kRedThreads;
  static_assert(PIHM_RED_MAXBLOCKS % kRedThreads == 0, "whole rounds of partials per thread");
  __shared__ double lds[(kRedThreads / 64) * NV];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned count = *ctr + 1u;
  double v[NV][kPer];
#pragma unroll
  for (int k = 0; k < NV; k++) {
    constexpr unsigned m = 3u;
    const unsigned c = (COMBS >> (2 * k)) & m;
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      const int b = (int)threadIdx.x + j * kRedThreads;
      const double *p = partials + (long)k * PIHM_RED_MAXBLOCKS + b;
      v[k][j] = comb_ident(c);
      if (b < nb) v[k][j] = SHARED ? __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *p;
    }
  }
  double x[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const unsigned c = (COMBS >> (2 * k)) & 3u;
    x[k] = v[k][0];
#pragma unroll
    for (int j = 1; j < kPer; j++) x[k] = comb(c, x[k], v[k][j]);
    x[k] = wave_comb(c, x[k]);
  }
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) lds[wave * NV + k] = x[k];
  }
  __syncthreads();
  if (wave == 0) {
    if (lane < NV) {
      double r = lds[lane];
#pragma unroll
      for (int w2 = 1; w2 < kRedThreads / 64; w2++) {
        const double o = lds[w2 * NV + lane];
        r = comb((COMBS >> (2 * lane)) & 3u, r, o);
      }
      __hip_atomic_store(&result[lane], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      if (devcopy) devcopy[lane] = r;
    }
    if (lane == 0) {
      if (xstore) *xstore = xval;
      *ctr = count;
    }
    // the results have reached host memory before the count that announces them
    wait_memory();
    if (lane == 0) *flag = count;
  }
}

template <int NV, class F>
__global__ __launch_bounds__(kRedThreads) void k_fused_sum(long n, F f, double *partials, pihm_redwork w,
                                                           double *devcopy, double *xstore, double xval) {
  __shared__ double lds[4 * NV];
  double acc[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) acc[k] = 0.0;
  const long stride = (long)gridDim.x * blockDim.x;
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if constexpr (requires(const F &g, long j) { g.load(j); }) {
    // two entries' loads before either entry's stores; the sums keep the
    // order of the entries
    for (; i + stride < n; i += 2 * stride) {
      const auto a = f.load(i);
      const auto b = f.load(i + stride);
      f.apply(i, a, acc);
      f.apply(i + stride, b, acc);
    }
    if (i < n) f.apply(i, f.load(i), acc);
  } else {
    for (; i < n; i += stride) f(i, acc);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool ends = (int)gridDim.x <= kTicketBlocks;    // this launch has the second pass too
#pragma unroll
  for (int k = 0; k < NV; k++) acc[k] = wave_sum(acc[k]);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) lds[wave * NV + k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    const int k = threadIdx.x;
    const double v = ((lds[k] + lds[NV + k]) + lds[2 * NV + k]) + lds[3 * NV + k];
    store_partial(&partials[(long)k * PIHM_RED_MAXBLOCKS + blockIdx.x], v, ends);
  }
  if (ends && last_workgroup(w.ticket, gridDim.x))
    second_pass<NV, 0u, true>(gridDim.x, partials, w.result, devcopy, w.ctr, w.flag, xstore, xval);
}

namespace {
template <int NV, unsigned COMBS>
__global__ __launch_bounds__(kRedThreads) void k_partials_final(int nb, const double *partials, double *result,
                                                                double *devcopy, unsigned *ctr,
                                                                volatile unsigned *flag, double *xstore,
                                                                double xval) {
  second_pass<NV, COMBS, false>(nb, partials, result, devcopy, ctr, flag, xstore, xval);
}
}  // namespace

// Launch the second pass of a reduction whose first pass wrote nb partials,
// unless the first pass ended in it.
template <int NV, unsigned COMBS>
inline void launch_final(int nb, pihm_redwork w, hipStream_t st, double *devcopy, double *xstore = nullptr,
                         double xval = 0.0) {
  if (nb <= kTicketBlocks && w.ticket) return;
  hipLaunchKernelGGL((k_partials_final<NV, COMBS>), dim3(1), dim3(kRedThreads), 0, st, nb, w.partials, w.result,
                     devcopy, w.ctr, w.flag, xstore, xval);
}

// Launch both passes without waiting (devcopy: optional device copy of the
// results; xstore: optional scalar store made by the second pass).
template <int NV, class F>
void fused_sum_launch(long n, const F &f, pihm_redwork w, hipStream_t st, double *devcopy,
                      double *xstore = nullptr, double xval = 0.0) {
  const int nb = fused_blocks(n);
  hipLaunchKernelGGL((k_fused_sum<NV, F>), dim3(nb), dim3(kRedThreads), 0, st, n, f, w.partials, w, devcopy, xstore,
                     xval);
  launch_final<NV, 0u>(nb, w, st, devcopy, xstore, xval);
}

// Launch both passes and wait; results in out[0..NV).
template <int NV, class F>
int fused_sum(long n, const F &f, pihm_redwork w, hipStream_t st, double *out, double *devcopy = nullptr,
              double *xstore = nullptr, double xval = 0.0) {
  fused_sum_launch<NV>(n, f, w, st, devcopy, xstore, xval);
  if (hipGetLastError() != hipSuccess) return -2;
  if (pihm_red_wait(w, st)) return -2;
  for (int k = 0; k < NV; k++) out[k] = w.result[k];
  return 0;
}

}  // namespace pihm
