// kernels_basic.hip -- gfx950 kernels for the formation, Ruiz, SpMV, CG and
// recovery steps of the HyKKT solve, over a batch of same-pattern systems
// (system blockIdx.y; see Batch in kernels.hpp).
//
// Built with -ffp-contract=off: every fused multiply-add here is an explicit
// fma(), so the SpGEMM/Ruiz/rhs values are bit-identical to the CPU oracle,
// which uses the same operation order.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdio>
#include <string>

#include "basic_dev.hpp"
#include "common.hpp"

namespace hykkt {
namespace dev {

void check(hipError_t e, const char* what)
{
  if (e != hipSuccess) {
    int code = (e == hipErrorOutOfMemory) ? HYKKT_E_NOMEM : HYKKT_E_HIP;
    throw Error(code, std::string("HIP error ") + hipGetErrorString(e) + " in " + what);
  }
}

namespace {

constexpr int SPMV_E = 1024;    // entries of a row block staged in LDS

inline dim3 grid2(int64_t n, const Batch& b) { return dim3(nblocks(n), b.count); }

// ------------------------------------------------------------- vectors
__global__ void k_fill(double* __restrict__ p, double v, int64_t n, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  p = at(p, s, b);
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_fill_i(int* __restrict__ p, int v, int64_t n)
{
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_copy(double* __restrict__ d, const double* __restrict__ src, int64_t n, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  d = at(d, s, b);
  src = at(src, s, b);
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    d[i] = src[i];
}

struct CopyDesc {
  double* dst[COPY_ARRAYS];
  int64_t len[COPY_ARRAYS];
  bool zero_null[COPY_ARRAYS];
  const double* src[COPY_SYSTEMS][COPY_ARRAYS];
  double* dst_scalar;
  double scalar[COPY_SYSTEMS];
  int s0;   // first system of the launch
};
static_assert(sizeof(CopyDesc) <= 4000, "kernel argument space");

// grid (blocks, systems of the launch, arrays)
__global__ void k_copy_in(CopyDesc c, Batch b)
{
  const int j = blockIdx.z, k = blockIdx.y, s = c.s0 + k;
  if (j == 0 && blockIdx.x == 0 && threadIdx.x == 0) at(c.dst_scalar, s, b)[0] = c.scalar[k];
  const double* src = c.src[k][j];
  double* d = at(c.dst[j], s, b);
  const int64_t n = c.len[j];
  if (!src && !c.zero_null[j]) return;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    d[i] = src ? src[i] : 0.0;
}

__global__ void k_gather64(double* __restrict__ d, const double* __restrict__ s,
                           const int64_t* __restrict__ map, int64_t n)
{
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    d[i] = s[map[i]];
}

__global__ void k_vec_scale(double* __restrict__ y, const double* __restrict__ sv, int n, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  y = at(y, s, b);
  sv = at(sv, s, b);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    y[i] *= sv[i];
}

// ------------------------------------------------------------- sparse
__global__ void k_row_scale(int d, const int* __restrict__ rp, const double* __restrict__ v,
                            const double* __restrict__ ds, const double* __restrict__ ryd,
                            const double* __restrict__ rs, double* __restrict__ vs,
                            double* __restrict__ ryd_s, int* __restrict__ word0,
                            int* __restrict__ word1, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (word0) word0[s] = INT_MAX;
    if (word1) word1[s] = INT_MAX;
  }
  v = at(v, s, b);
  ds = at(ds, s, b);
  ryd = at(ryd, s, b);
  rs = at(rs, s, b);
  vs = at(vs, s, b);
  ryd_s = at(ryd_s, s, b);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < d; i += gridDim.x * blockDim.x) {
    double di = ds[i];
    if (vs)
      for (int p = rp[i]; p < rp[i + 1]; p++) vs[p] = v[p] * di;
    double t = ryd[i] * di;
    ryd_s[i] = t + 1.0 * rs[i];
  }
}

// CSR-stream SpMV (Greathouse & Daga, SC'14): one workgroup per row block;
// the block's values and the x entries they multiply are staged through LDS
// with coalesced loads, then each row is summed by one thread in column
// order, so the result equals the sequential fma chain bit for bit.
__global__ void __launch_bounds__(TPB) k_spmv(const int* __restrict__ rp,
                                              const int* __restrict__ ci,
                                              const int* __restrict__ map,
                                              const double* __restrict__ v, double alpha,
                                              const double* __restrict__ alpha_ps,
                                              const double* __restrict__ x, double beta,
                                              const double* __restrict__ y_in,
                                              double* __restrict__ y_out,
                                              const int* __restrict__ blocks,
                                              const double* __restrict__ dot_w,
                                              double* __restrict__ dot_part,
                                              const int* __restrict__ y_map, SweepFill fill,
                                              Batch b)
{
  __shared__ double lv[SPMV_E];
  __shared__ double lx[SPMV_E];
  clear_tickets(fill.ticket);
  const int s = sys_of(b);
  if (s < 0) return;
  fill_sweep(fill, s, b, blockIdx.x, gridDim.x);
  v = at(v, s, b);
  x = at(x, s, b);
  y_in = at(y_in, s, b);
  y_out = at(y_out, s, b);
  if (alpha_ps) alpha = *at(alpha_ps, s, b);
  const int r0 = blocks[blockIdx.x], r1 = blocks[blockIdx.x + 1];
  const int e0 = rp[r0], e1 = rp[r1];
  const int tid = threadIdx.x;
  double yi = 0.0;
  const int r = r0 + tid;
  if (e1 - e0 <= SPMV_E) {
    for (int k = tid; k < e1 - e0; k += TPB) {
      const int q = e0 + k;
      lv[k] = v[map ? map[q] : q];
      lx[k] = x[ci[q]];
    }
    __syncthreads();
    if (r < r1) {
      double t = 0.0;
      for (int q = rp[r] - e0; q < rp[r + 1] - e0; q++) t = fma(lv[q], lx[q], t);
      yi = (beta == 0.0) ? alpha * t : fma(alpha, t, beta * y_in[y_map ? y_map[r] : r]);
      y_out[r] = yi;
    }
  } else {
    // one long row (the block has only this row): staged in chunks, summed
    // by thread 0 in order
    double t = 0.0;
    for (int c0 = e0; c0 < e1; c0 += SPMV_E) {
      const int cn = min(SPMV_E, e1 - c0);
      __syncthreads();
      for (int k = tid; k < cn; k += TPB) {
        const int q = c0 + k;
        lv[k] = v[map ? map[q] : q];
        lx[k] = x[ci[q]];
      }
      __syncthreads();
      if (tid == 0)
        for (int k = 0; k < cn; k++) t = fma(lv[k], lx[k], t);
    }
    if (tid == 0) {
      yi = (beta == 0.0) ? alpha * t : fma(alpha, t, beta * y_in[y_map ? y_map[r0] : r0]);
      y_out[r0] = yi;
    }
  }
  if (dot_part) {
    const double w = (r < r1) ? yi * at(dot_w, s, b)[r] : 0.0;
    const double tot = block_sum(w);
    if (tid == 0) at(dot_part, s, b)[blockIdx.x] = tot;
  }
}

__device__ __forceinline__ double spgemm_entry(int p, const int* __restrict__ d_src,
                                               const double* __restrict__ d_v,
                                               const int* __restrict__ tp,
                                               const int* __restrict__ ta,
                                               const int* __restrict__ tb,
                                               const double* __restrict__ av,
                                               const double* __restrict__ bv, double alpha_p)
{
  double acc = 0.0;
  for (int t = tp[p]; t < tp[p + 1]; t++) acc = fma(av[ta[t]], bv[tb[t]], acc);
  int s = d_src[p];
  double d = (s >= 0) ? d_v[s] : 0.0;
  double c = alpha_p * acc;
  return 1.0 * d + 1.0 * c;
}

__global__ void k_spgemm_values(int nnz, const int* __restrict__ d_src,
                                const double* __restrict__ d_v, const int* __restrict__ tp,
                                const int* __restrict__ ta, const int* __restrict__ tb,
                                const double* __restrict__ av, const double* __restrict__ bv,
                                double alpha_p, double* __restrict__ out, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  d_v = at(d_v, s, b);
  av = at(av, s, b);
  bv = at(bv, s, b);
  out = at(out, s, b);
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nnz; p += gridDim.x * blockDim.x)
    out[p] = spgemm_entry(p, d_src, d_v, tp, ta, tb, av, bv, alpha_p);
}

__global__ void k_spgemm_scatter(int nent, const int* __restrict__ src,
                                 const int64_t* __restrict__ dst,
                                 const int* __restrict__ d_src, const double* __restrict__ d_v,
                                 const int* __restrict__ tp, const int* __restrict__ ta,
                                 const int* __restrict__ tb, const double* __restrict__ av,
                                 const double* __restrict__ bv,
                                 const double* __restrict__ alpha_ps, double* __restrict__ out,
                                 Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  d_v = at(d_v, s, b);
  av = at(av, s, b);
  bv = at(bv, s, b);
  out = at(out, s, b);
  const double alpha_p = *at(alpha_ps, s, b);
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nent; e += gridDim.x * blockDim.x)
    out[dst[e]] = spgemm_entry(src[e], d_src, d_v, tp, ta, tb, av, bv, alpha_p);
}

__global__ void k_scatter(double* __restrict__ out, const int64_t* __restrict__ dst,
                          const double* __restrict__ vals, const int* __restrict__ src, int n,
                          Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  out = at(out, s, b);
  vals = at(vals, s, b);
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x)
    out[dst[e]] = vals[src[e]];
}

__global__ void k_add_at(double* __restrict__ out, const int64_t* __restrict__ pos, int n,
                         double delta, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  out = at(out, s, b);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    out[pos[i]] += delta;
}

// ------------------------------------------------------------- Ruiz
__global__ void k_ruiz_rowmax(int n, int totn, const int* __restrict__ h_rp,
                              const double* __restrict__ h_v, const int* __restrict__ jt_rp,
                              const int* __restrict__ jt_map, const double* __restrict__ jt_v,
                              const int* __restrict__ j_rp, const double* __restrict__ j_v,
                              double* __restrict__ scale, int* __restrict__ zero_row, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  h_v = at(h_v, s, b);
  jt_v = at(jt_v, s, b);
  j_v = at(j_v, s, b);
  scale = at(scale, s, b);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < totn; i += gridDim.x * blockDim.x) {
    double max_l = 0.0, max_u = 0.0;
    if (i < n) {
      for (int p = h_rp[i]; p < h_rp[i + 1]; p++) {
        double e = fabs(h_v[p]);
        if (e > max_l) max_l = e;
      }
      for (int q = jt_rp[i]; q < jt_rp[i + 1]; q++) {
        double e = fabs(jt_v[jt_map ? jt_map[q] : q]);
        if (e > max_u) max_u = e;
      }
      scale[i] = (max_l > max_u) ? 1.0 / sqrt(max_l) : 1.0 / sqrt(max_u);
    } else {
      for (int p = j_rp[i - n]; p < j_rp[i - n + 1]; p++) {
        double e = fabs(j_v[p]);
        if (e > max_l) max_l = e;
      }
      scale[i] = 1.0 / sqrt(max_l);
    }
    // a row without a nonzero value (or with a NaN) gets the scale 1/sqrt(0)
    if (zero_row && !(max_l > 0.0 || max_u > 0.0)) atomicMin(zero_row + s, i);
  }
}

__global__ void k_ruiz_scale(int n, int totn, const int* __restrict__ h_rp,
                             const int* __restrict__ h_ci, double* __restrict__ h_v,
                             const int* __restrict__ jt_rp, const int* __restrict__ jt_ci,
                             double* __restrict__ jt_v, const int* __restrict__ j_rp,
                             const int* __restrict__ j_ci, double* __restrict__ j_v,
                             const double* __restrict__ scale, double* __restrict__ rhs1,
                             double* __restrict__ rhs2, double* __restrict__ max_d, int first,
                             Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  h_v = at(h_v, s, b);
  jt_v = at(jt_v, s, b);
  j_v = at(j_v, s, b);
  scale = at(scale, s, b);
  rhs1 = at(rhs1, s, b);
  rhs2 = at(rhs2, s, b);
  max_d = at(max_d, s, b);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < totn; i += gridDim.x * blockDim.x) {
    double si = scale[i];
    if (i < n) {
      for (int p = h_rp[i]; p < h_rp[i + 1]; p++) h_v[p] *= si * scale[h_ci[p]];
      rhs1[i] *= si;
      max_d[i] = first ? 1.0 * si : max_d[i] * si;
      if (jt_v)
        for (int q = jt_rp[i]; q < jt_rp[i + 1]; q++) jt_v[q] *= si * scale[n + jt_ci[q]];
    } else {
      for (int p = j_rp[i - n]; p < j_rp[i - n + 1]; p++) j_v[p] *= si * scale[j_ci[p]];
      rhs2[i - n] *= si;
      max_d[i] = first ? 1.0 * si : max_d[i] * si;
    }
  }
}

// One sweep of the solver's equilibration over the rows of [H~ Jc^T; Jc], RL
// lanes per row: apply the last scale (c.scale_in: h, j_src -> j_dst, the
// right-hand sides, max_d) and form the next one from the scaled rows
// (c.scale_out), so `its` sweeps take its + 1 passes over the values instead of
// 2 its.  Jc^T's values are Jc's, scaled here by the same product as in Jc's own
// row (multiplication commutes), read from j_src, which the pass leaves alone.
// The maxima are exact in any order and every other value is the rounding of
// k_ruiz_rowmax / k_ruiz_scale, so all results are the same bits.  Bound by the
// latency of a row's chain of loads with a thread per row (four launches of 22
// us at 1,000 buses); with 16 lanes the three passes take 15 us
// together (10,000 buses: 112 -> 35 us).
constexpr int RL = 16;

__global__ void __launch_bounds__(TPB) k_ruiz_pass(RuizPass c, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  double* const h_v = at(c.h_v, s, b);
  const double* const j_src = at(c.j_src, s, b);
  double* const j_dst = at(c.j_dst, s, b);
  const double* const sin = at(c.scale_in, s, b);
  double* const sout = at(c.scale_out, s, b);
  const int n = c.n, l = threadIdx.x & (RL - 1);
  const int rows = gridDim.x * (TPB / RL);
  for (int i = blockIdx.x * (TPB / RL) + threadIdx.x / RL; i < n + c.m; i += rows) {
    const double si = sin ? sin[i] : 1.0;
    double max_l = 0.0, max_u = 0.0;
    if (i < n) {
      for (int p = c.h_rp[i] + l; p < c.h_rp[i + 1]; p += RL) {
        double v = h_v[p];
        if (sin) {
          v *= si * sin[c.h_ci[p]];
          h_v[p] = v;
        }
        const double e = fabs(v);
        if (e > max_l) max_l = e;
      }
      if (sout)
        for (int q = c.jt_rp[i] + l; q < c.jt_rp[i + 1]; q += RL) {
          double v = j_src[c.jt_map[q]];
          if (sin) v *= sin[n + c.jt_ci[q]] * si;
          const double e = fabs(v);
          if (e > max_u) max_u = e;
        }
    } else {
      for (int p = c.j_rp[i - n] + l; p < c.j_rp[i - n + 1]; p += RL) {
        double v = j_src[p];
        if (sin) {
          v *= si * sin[c.j_ci[p]];
          j_dst[p] = v;
        }
        const double e = fabs(v);
        if (e > max_l) max_l = e;
      }
    }
    if (sin && l == 0) {
      if (i < n) {
        double* r = at(c.rhs1, s, b);
        r[i] *= si;
      } else {
        at(c.rhs2, s, b)[i - n] = at(c.rhs2_src, s, b)[i - n] * si;
      }
      double* md = at(c.max_d, s, b);
      md[i] = c.first ? 1.0 * si : md[i] * si;
    }
    if (sout) {
#pragma unroll
      for (int k = RL / 2; k > 0; k >>= 1) {
        const double ol = __shfl_xor(max_l, k, RL), ou = __shfl_xor(max_u, k, RL);
        if (ol > max_l) max_l = ol;
        if (ou > max_u) max_u = ou;
      }
      if (l == 0) {
        if (i < n) sout[i] = (max_l > max_u) ? 1.0 / sqrt(max_l) : 1.0 / sqrt(max_u);
        else sout[i] = 1.0 / sqrt(max_l);
        // a row without a nonzero value (or with a NaN) gets the scale 1/sqrt(0)
        if (!(max_l > 0.0 || max_u > 0.0)) atomicMin(c.zero_row + s, i);
      }
    }
  }
}

// ------------------------------------------------------------- reductions
// grid (reduce_blocks(n), systems): block j sums i = j*TPB + t + k*(blocks*TPB)
__global__ void k_dot_partial(int n, const double* __restrict__ a, const double* __restrict__ bv,
                              double* __restrict__ part, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  a = at(a, s, b);
  bv = at(bv, s, b);
  double t = 0.0;
  for (int i = blockIdx.x * TPB + threadIdx.x; i < n; i += gridDim.x * TPB)
    t = bv ? fma(a[i], bv[i], t) : t + a[i];
  const double tot = block_sum(t);
  if (threadIdx.x == 0) at(part, s, b)[blockIdx.x] = tot;
}

// words[0]: set by k_set_word; words[1]: what k_wait_word saw of it in at most
// `polls` polls (about a microsecond each).
__global__ void k_wait_word(int* words, int polls)
{
  int v = 0;
  for (int i = 0; i < polls && v == 0; i++) {
    v = __hip_atomic_load(words, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_sleep(16);
  }
  __hip_atomic_store(words + 1, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void k_set_word(int* word, int v)
{
  __hip_atomic_store(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

// =================================================================== launchers
#define LAUNCH_CHECK() HIPCHK(hipGetLastError())

bool streams_overlap(hipStream_t a, hipStream_t b, int* words)
{
  constexpr int POLLS = 400;
  // both kernels once before, so their code is loaded and the words are clear
  k_set_word<<<1, 1, 0, b>>>(words, 0);
  LAUNCH_CHECK();
  HIPCHK(hipStreamSynchronize(b));
  k_wait_word<<<1, 1, 0, a>>>(words, 1);
  LAUNCH_CHECK();
  HIPCHK(hipStreamSynchronize(a));
  k_wait_word<<<1, 1, 0, a>>>(words, POLLS);
  LAUNCH_CHECK();
  k_set_word<<<1, 1, 0, b>>>(words, 1);
  LAUNCH_CHECK();
  HIPCHK(hipStreamSynchronize(a));
  HIPCHK(hipStreamSynchronize(b));
  int saw = 0;
  HIPCHK(hipMemcpy(&saw, words + 1, sizeof(int), hipMemcpyDeviceToHost));
  return saw != 0;
}

void fill(double* p, double v, int64_t n, const Batch& b, hipStream_t st)
{
  if (n <= 0 || b.count <= 0) return;
  k_fill<<<grid2(n, b), TPB, 0, st>>>(p, v, n, b);
  LAUNCH_CHECK();
}

void fill_i(int* p, int v, int64_t n, hipStream_t st)
{
  if (n <= 0) return;
  k_fill_i<<<nblocks(n), TPB, 0, st>>>(p, v, n);
  LAUNCH_CHECK();
}

void copy(double* d, const double* s, int64_t n, const Batch& b, hipStream_t st)
{
  if (n <= 0 || b.count <= 0) return;
  k_copy<<<grid2(n, b), TPB, 0, st>>>(d, s, n, b);
  LAUNCH_CHECK();
}

void copy_in(double* const* dst, const int64_t* len, const bool* zero_null,
             const double* const* src, double* dst_scalar, const double* scalar, const Batch& b,
             hipStream_t st, hipEvent_t start)
{
  CopyDesc c{};
  int64_t mx = 1;
  for (int j = 0; j < COPY_ARRAYS; j++) {
    c.dst[j] = dst[j];
    c.len[j] = len[j];
    c.zero_null[j] = zero_null[j];
    mx = std::max(mx, len[j]);
  }
  c.dst_scalar = dst_scalar;
  for (c.s0 = 0; c.s0 < b.count; c.s0 += COPY_SYSTEMS) {
    const int ns = std::min(COPY_SYSTEMS, b.count - c.s0);
    for (int k = 0; k < ns; k++) {
      for (int j = 0; j < COPY_ARRAYS; j++) c.src[k][j] = src[(c.s0 + k) * COPY_ARRAYS + j];
      c.scalar[k] = scalar[c.s0 + k];
    }
    hipExtLaunchKernelGGL(k_copy_in, dim3(nblocks(mx), ns, COPY_ARRAYS), dim3(TPB), 0, st,
                          c.s0 == 0 ? start : nullptr, nullptr, 0, c, b);
    LAUNCH_CHECK();
  }
}

void gather64(double* d, const double* s, const int64_t* map, int64_t n, hipStream_t st)
{
  if (n <= 0) return;
  k_gather64<<<nblocks(n), TPB, 0, st>>>(d, s, map, n);
  LAUNCH_CHECK();
}

void vec_scale(double* y, const double* s, int n, const Batch& b, hipStream_t st)
{
  if (n <= 0 || b.count <= 0) return;
  k_vec_scale<<<grid2(n, b), TPB, 0, st>>>(y, s, n, b);
  LAUNCH_CHECK();
}

void row_scale(int d, const int* rp, const double* v, const double* ds, const double* ryd,
               const double* rs, double* vs, double* ryd_s, const Batch& b, hipStream_t st,
               int* word0, int* word1)
{
  if (d <= 0 || b.count <= 0) return;
  k_row_scale<<<grid2(d, b), TPB, 0, st>>>(d, rp, v, ds, ryd, rs, vs, ryd_s, word0, word1, b);
  LAUNCH_CHECK();
}

int spmv_lds_entries() { return SPMV_E; }

void spmv(int nrows, const int* rp, const int* ci, const int* map, const double* v, double alpha,
          const double* alpha_ps, const double* x, double beta, const double* y_in,
          double* y_out, const int* blocks, int nblk, const Batch& b, hipStream_t st,
          const double* dot_w, double* dot_part, const int* y_map, const SweepFill& fill)
{
  if (nrows <= 0 || nblk <= 0 || b.count <= 0) return;
  k_spmv<<<dim3(nblk, b.count), TPB, 0, st>>>(rp, ci, map, v, alpha, alpha_ps, x, beta, y_in,
                                               y_out, blocks, dot_w, dot_part, y_map, fill, b);
  LAUNCH_CHECK();
}

void spgemm_values(int nnz, const int* d_src, const double* d_v, const int* tp, const int* ta,
                   const int* tb, const double* av, const double* bv, double alpha_p,
                   double* out, const Batch& b, hipStream_t st)
{
  if (nnz <= 0 || b.count <= 0) return;
  k_spgemm_values<<<grid2(nnz, b), TPB, 0, st>>>(nnz, d_src, d_v, tp, ta, tb, av, bv, alpha_p,
                                                 out, b);
  LAUNCH_CHECK();
}

void spgemm_scatter(int nent, const int* src, const int64_t* dst, const int* d_src,
                    const double* d_v, const int* tp, const int* ta, const int* tb,
                    const double* av, const double* bv, const double* alpha_ps, double* out,
                    const Batch& b, hipStream_t st)
{
  if (nent <= 0 || b.count <= 0) return;
  k_spgemm_scatter<<<grid2(nent, b), TPB, 0, st>>>(nent, src, dst, d_src, d_v, tp, ta, tb, av,
                                                   bv, alpha_ps, out, b);
  LAUNCH_CHECK();
}

void scatter(double* out, const int64_t* dst, const double* vals, const int* src, int n,
             const Batch& b, hipStream_t st)
{
  if (n <= 0 || b.count <= 0) return;
  k_scatter<<<grid2(n, b), TPB, 0, st>>>(out, dst, vals, src, n, b);
  LAUNCH_CHECK();
}

void add_at(double* out, const int64_t* pos, int n, double delta, const Batch& b,
            hipStream_t st)
{
  if (n <= 0 || b.count <= 0) return;
  k_add_at<<<grid2(n, b), TPB, 0, st>>>(out, pos, n, delta, b);
  LAUNCH_CHECK();
}

void ruiz_rowmax(int n, int totn, const int* h_rp, const double* h_v, const int* jt_rp,
                 const int* jt_map, const double* jt_v, const int* j_rp, const double* j_v,
                 double* scale, int* zero_row, const Batch& b, hipStream_t st)
{
  if (totn <= 0 || b.count <= 0) return;
  k_ruiz_rowmax<<<grid2(totn, b), TPB, 0, st>>>(n, totn, h_rp, h_v, jt_rp, jt_map, jt_v, j_rp,
                                                j_v, scale, zero_row, b);
  LAUNCH_CHECK();
}

void ruiz_scale(int n, int totn, const int* h_rp, const int* h_ci, double* h_v,
                const int* jt_rp, const int* jt_ci, double* jt_v, const int* j_rp,
                const int* j_ci, double* j_v, const double* scale, double* rhs1, double* rhs2,
                double* max_d, int first, const Batch& b, hipStream_t st)
{
  if (totn <= 0 || b.count <= 0) return;
  k_ruiz_scale<<<grid2(totn, b), TPB, 0, st>>>(n, totn, h_rp, h_ci, h_v, jt_rp, jt_ci, jt_v,
                                               j_rp, j_ci, j_v, scale, rhs1, rhs2, max_d, first,
                                               b);
  LAUNCH_CHECK();
}

void ruiz_pass(const RuizPass& c, const Batch& b, hipStream_t st)
{
  if (c.n + c.m <= 0 || b.count <= 0) return;
  k_ruiz_pass<<<dim3(nblocks(c.n + c.m, TPB / RL), b.count), TPB, 0, st>>>(c, b);
  LAUNCH_CHECK();
}

void dot_partial(int n, const double* a, const double* bv, double* part, const Batch& b,
                 hipStream_t st)
{
  if (b.count <= 0) return;
  k_dot_partial<<<dim3(reduce_blocks(n), b.count), TPB, 0, st>>>(n, a, bv, part, b);
  LAUNCH_CHECK();
}

}  // namespace dev
}  // namespace hykkt
