// sweep_dev.hpp -- device helpers of the triangular-solve sweeps (gfx950): the
// exchanged values and their waits, work items, buffer loads, and cross-lane
// sums.  See kernels_trsv.hip for how the sweeps synchronise.
#pragma once

#include <hip/hip_runtime.h>

#include "batch_dev.hpp"
#include "kernels.hpp"

namespace hykkt {
namespace dev {
namespace {

constexpr int SPIN_LIMIT = 1 << 22;      // polls; each sleeps >= 128 clocks and waits one
                                         // device-scope load: seconds per wait at most

// Wave-uniform copies (scalar registers) of values every lane loaded alike.
// Buffer descriptors built from them stay scalar; a descriptor the compiler
// cannot prove uniform turns every buffer load into a serialising loop.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uni64(int64_t v)
{
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(static_cast<uint64_t>(v) >> 32));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// One system's buffers in a sweep (wave-uniform pointers).
struct SysBufs {
  const double* L;
  const double* dinv;
  double* ubuf;
  double* exch;
  const double* in;    // right-hand side (forward) or y (backward)
  double* out;         // y (forward) or x (backward)
};

__device__ __forceinline__ SysBufs sys_bufs(const CholDev& c, const SolveDev& sd, int sy,
                                            const Batch& bt, const double* in, double* out)
{
  const int64_t o = static_cast<int64_t>(sy) * bt.vs;
  return SysBufs{c.L + o, c.dinv + o, sd.ubuf + o, sd.exch + o, in + o, out + o};
}

__device__ __forceinline__ double xload(const double* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void xstore(double* p, double v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ bool pending(double v)
{
  return __builtin_bit_cast(uint64_t, v) == SWEEP_SENTINEL;
}

// The value at p once its producer has written it.  Gives up (sets *err,
// returns 0) after SPIN_LIMIT polls, or soon after another wait gave up.
__device__ double spin_load(const double* p, int* err)
{
  double v = xload(p);
  int it = 0;
  while (pending(v)) {
    __builtin_amdgcn_s_sleep(2);
    ++it;
    if (it > SPIN_LIMIT ||
        ((it & 1023) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
      __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return 0.0;
    }
    v = xload(p);
  }
  return v;
}

// acc + (minus, NEG) the values at(0), .., at(n - 1), in that order, each once
// its producer has written it.  U loads are in flight at a time: one after the
// other they cost a round trip to the coherent level each (0.7 us).
template <bool NEG, int U = 8, class AT>
__device__ __forceinline__ double spin_sum(double acc, int n, AT at, int* err)
{
  for (int p0 = 0; p0 < n; p0 += U) {
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = xload(at(min(p0 + u, n - 1)));
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (p0 + u >= n) break;
      const double x = pending(v[u]) ? spin_load(at(p0 + u), err) : v[u];
      acc = NEG ? acc - x : acc + x;
    }
  }
  return acc;
}

// The launch's next item, in the order workgroups start running.  Item i
// goes to a workgroup only after items 0..i-1 went to workgroups that were
// already running, so the smallest unfinished item is always held by a
// running workgroup whose producers have all finished: the sweep progresses
// whatever else shares the device (kernels of other streams may hold the
// compute units, and workgroup dispatch order alone would not guarantee it).
__device__ __forceinline__ int take_item(int* ticket)
{
  __shared__ int item;
  if (threadIdx.x == 0)
    item = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  return uni(item);
}

// Buffer loads: a uniform base in a buffer descriptor (SGPRs), a per-lane
// byte offset and a uniform byte offset, so a stretch of strided loads costs
// scalar arithmetic and one offset register instead of one address pair per
// load.  Word 3 of the descriptor is the gfx9-family raw-buffer setting.
using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr int RSRC_W3 = 0x00020000;

__device__ __forceinline__ rsrc_t view(const double* base, uint32_t bytes)
{
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(base), 0, bytes, RSRC_W3);
}

__device__ __forceinline__ double ld(rsrc_t r, uint32_t voff, uint32_t soff)
{
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}

// Two consecutive values (any multiple of 8 bytes).
typedef double d2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ d2v ld2(rsrc_t r, uint32_t voff, uint32_t soff)
{
  return __builtin_bit_cast(d2v, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// Cross-lane sums of several values per lane.  Each exchange halves the values a
// lane keeps: the lanes with bit M of the lane index set keep the upper half,
// the others the lower half, and each adds its partner's (lane l ^ M).  The
// exchanges run on the VALU: the lane-half swaps of gfx950
// (v_permlane32_swap, v_permlane16_swap) for M = 32 and 16, DPP row rotations
// and shifts for M = 8 and 4, DPP quad permutations for 2 and 1.
__device__ __forceinline__ uint32_t lo32(double v)
{
  return static_cast<uint32_t>(__builtin_bit_cast(uint64_t, v));
}
__device__ __forceinline__ uint32_t hi32(double v)
{
  return static_cast<uint32_t>(__builtin_bit_cast(uint64_t, v) >> 32);
}
__device__ __forceinline__ double mk64(uint32_t lo, uint32_t hi)
{
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

// One exchange for M = 32 (W32) or 16 over the pairs (acc[i], acc[i + N/2]):
// the swap puts a lane's kept value and its partner's sent value in the
// two registers, whose sum is keep + partner's value (addition commutes).
template <int N, bool W32, int W>
__device__ __forceinline__ void halve_swap(double (&acc)[W])
{
#pragma unroll
  for (int i = 0; i < N / 2; i++) {
    const double x = acc[i], y = acc[i + N / 2];
    const auto lo = W32 ? __builtin_amdgcn_permlane32_swap(lo32(x), lo32(y), false, false)
                        : __builtin_amdgcn_permlane16_swap(lo32(x), lo32(y), false, false);
    const auto hi = W32 ? __builtin_amdgcn_permlane32_swap(hi32(x), hi32(y), false, false)
                        : __builtin_amdgcn_permlane16_swap(hi32(x), hi32(y), false, false);
    acc[i] = mk64(lo[0], hi[0]) + mk64(lo[1], hi[1]);
  }
}

// The value of lane l ^ M (M = 8, 4, 2 or 1) by DPP: row_ror:8 for 8;
// row_shr:4 / row_shl:4 by the lane's bit 2 for 4; quad_perm for 2 and 1.
template <int M>
__device__ __forceinline__ double xor_dpp(double v, int lane)
{
  const uint32_t a = lo32(v), b = hi32(v);
  if constexpr (M == 8) {
    return mk64(__builtin_amdgcn_update_dpp(0u, a, 0x128, 0xf, 0xf, false),
                __builtin_amdgcn_update_dpp(0u, b, 0x128, 0xf, 0xf, false));
  } else if constexpr (M == 4) {
    const uint32_t dl = __builtin_amdgcn_update_dpp(0u, a, 0x114, 0xf, 0xf, false);
    const uint32_t dh = __builtin_amdgcn_update_dpp(0u, b, 0x114, 0xf, 0xf, false);
    const uint32_t ul = __builtin_amdgcn_update_dpp(0u, a, 0x104, 0xf, 0xf, false);
    const uint32_t uh = __builtin_amdgcn_update_dpp(0u, b, 0x104, 0xf, 0xf, false);
    return (lane & 4) ? mk64(dl, dh) : mk64(ul, uh);
  } else {
    constexpr int QP = M == 2 ? 0x4E : 0xB1;   // quad_perm [2,3,0,1] / [1,0,3,2]
    return mk64(__builtin_amdgcn_update_dpp(0u, a, QP, 0xf, 0xf, false),
                __builtin_amdgcn_update_dpp(0u, b, QP, 0xf, 0xf, false));
  }
}

// One exchange for M = 8, 4 or 2 over the pairs (acc[i], acc[i + N/2]).
template <int N, int M, int W>
__device__ __forceinline__ void halve(double (&acc)[W], int lane)
{
  const bool hi = (lane & M) != 0;
#pragma unroll
  for (int i = 0; i < N / 2; i++) {
    const double send = hi ? acc[i] : acc[i + N / 2];
    const double keep = hi ? acc[i + N / 2] : acc[i];
    acc[i] = keep + xor_dpp<M>(send, lane);
  }
}

}  // namespace
}  // namespace dev
}  // namespace hykkt
