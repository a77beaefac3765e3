// basic_dev.hpp -- device helpers shared by the formation and pass kernels: a
// workgroup's system, its buffers, and deterministic sums.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace hykkt {
namespace dev {
namespace {

constexpr int TPB = 256;

inline unsigned nblocks(int64_t n, int b = TPB)
{
  int64_t g = (n + b - 1) / b;
  if (g > 65536) g = 65536;
  return static_cast<unsigned>(g > 0 ? g : 1);
}

// This workgroup's system, or -1 when the mask skips it.
__device__ __forceinline__ int sys_of(const Batch& b)
{
  const int s = blockIdx.y;
  return (b.mask && !b.mask[s]) ? -1 : s;
}
template <class T>
__device__ __forceinline__ T* at(T* p, int s, const Batch& b)
{
  return p ? p + static_cast<int64_t>(s) * b.vs : p;
}

// Sum of a wave's 64 values, lane 0 has it (a fixed tree).
__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
  for (int k = 32; k > 0; k >>= 1) v += __shfl_down(v, k);
  return v;
}

// Deterministic tree sum of one value per thread (TPB threads); all threads
// get the result.  Thread t adds t + k's value for k = 128, 64, .., 1, the first
// two levels through LDS, the rest within the first wave.
__device__ __forceinline__ double block_sum(double v)
{
  static_assert(TPB == 256, "two levels across four waves");
  __shared__ double sh[TPB];
  const int t = threadIdx.x;
  __syncthreads();   // sh may still be read by a previous call
  sh[t] = v;
  __syncthreads();
  if (t < 64) {
    const double x = wave_sum((sh[t] + sh[t + 128]) + (sh[t + 64] + sh[t + 192]));
    if (t == 0) sh[0] = x;
  }
  __syncthreads();
  return sh[0];
}

// The sum of np partials as one workgroup forms it (all threads get it).
__device__ __forceinline__ double sum_partials(const double* part, int np)
{
  double t = 0.0;
  for (int i = threadIdx.x; i < np; i += TPB) t += part[i];
  return block_sum(t);
}

// The sentinel the sweeps wait on (see kernels_trsv.hip) into the buffers of f,
// shared by `of` workgroups of which this is number `blk`.
__device__ __forceinline__ void fill_sweep(const SweepFill& f, int s, const Batch& b, int blk,
                                           int of)
{
#pragma unroll
  for (int j = 0; j < 4; j++) {
    uint64_t* p = reinterpret_cast<uint64_t*>(at(f.p[j], s, b));
    for (int64_t i = blk * static_cast<int64_t>(TPB) + threadIdx.x; i < f.n[j];
         i += static_cast<int64_t>(of) * TPB)
      p[i] = SWEEP_SENTINEL;
  }
}

// The sweeps' item counters (once per launch, whatever the masks).
__device__ __forceinline__ void clear_tickets(int* ticket)
{
  if (ticket && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 4)
    __hip_atomic_store(ticket + threadIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace
}  // namespace dev
}  // namespace hykkt
