// kernels_pass.hip -- the kernels of a solve pass around the triangular solves
// (gfx950): Schur CG, recovery, residual check, over a batch of same-pattern
// systems (system blockIdx.y; see Batch in kernels.hpp).
//
// These steps move little data, so they are bound by launches (4.5 us each,
// back to back, whatever they do) and by a row's chain of dependent loads.  So
// one kernel does what can be done together, reductions are finished by the
// kernels that use them (every workgroup adds the partials itself, in one
// order), and row sums stage their entries through LDS: a 1,000-bus solve takes
// 25 launches around its factorization and triangular solves instead of 85 (1,000
// buses 1623 -> 1435 us, 203 buses 1059 -> 868).
//
// Built with -ffp-contract=off like kernels_basic.hip: every fused multiply-add
// is an explicit fma().
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "basic_dev.hpp"

namespace hykkt {
namespace dev {

namespace {

constexpr int ROWS = 64;    // rows of a workgroup in the row-sum kernels
constexpr int STAGE = 1024; // entries staged through LDS at a time

// Row sums of rows r0 .. r0 + ROWS - 1 of a CSR matrix: thread t < ROWS returns
// t0 extended by fma(v, x, t) over its row's entries in column order, the pair
// (v, x) of entry q being vx(q).  The entries are fetched by all threads, so a
// row's loads do not wait for each other.  All threads of the workgroup.
template <class VX>
__device__ __forceinline__ double row_sums(const int* rp, int r0, int nrows, double t, VX vx,
                                           double* lv, double* lx)
{
  const int r1 = min(r0 + ROWS, nrows), tid = threadIdx.x;
  const int e0 = rp[r0], e1 = rp[r1];
  const bool mine = tid < r1 - r0;
  const int qa = mine ? rp[r0 + tid] : 0, qb = mine ? rp[r0 + tid + 1] : 0;
  constexpr int PER = STAGE / TPB;
  for (int c0 = e0; c0 < e1; c0 += STAGE) {
    const int c1 = min(c0 + STAGE, e1);
    double v[PER], x[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) vx(min(c0 + tid + u * TPB, c1 - 1), v[u], x[u]);
    __syncthreads();   // the last chunk's reads
#pragma unroll
    for (int u = 0; u < PER; u++) {
      lv[tid + u * TPB] = v[u];
      lx[tid + u * TPB] = x[u];
    }
    __syncthreads();
    int q = max(qa, c0) - c0;
    const int qe = min(qb, c1) - c0;
    for (; q + 4 <= qe; q += 4) {   // four entries' LDS reads at a time
      double a[4], y[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        a[u] = lv[q + u];
        y[u] = lx[q + u];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) t = fma(a[u], y[u], t);
    }
    for (; q < qe; q++) t = fma(lv[q], lx[q], t);
  }
  return t;
}

// After the factorization: Jc's and Jc^T's values in the factor's order (maps
// into jcs); ok[s] = 1 when system s's factorization met no failing pivot, else 0,
// and then its solution (dx, dsv, dyc, dyd) is zero: such a system takes no part
// in the solve phase.
__global__ void k_after_factor(AfterFactor c, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  const bool failed = c.pivot[s] != INT_MAX;
  if (blockIdx.x == 0 && threadIdx.x == 0) c.ok[s] = failed ? 0 : 1;
  const double* jcs = at(c.jcs, s, b);
  double *jh = at(c.jh_v, s, b), *jth = at(c.jth_v, s, b);
  const int len = failed ? max(c.nnz, max(c.n, max(c.m, c.d))) : c.nnz;
  for (int i = blockIdx.x * TPB + threadIdx.x; i < len; i += gridDim.x * TPB) {
    if (i < c.nnz) {
      jh[i] = jcs[c.jh_map[i]];
      jth[i] = jcs[c.jth_map[i]];
    }
    if (failed) {
      if (i < c.n) at(c.dx, s, b)[i] = 0.0;
      if (i < c.m) at(c.dyc, s, b)[i] = 0.0;
      if (i < c.d) {
        at(c.dsv, s, b)[i] = 0.0;
        at(c.dyd, s, b)[i] = 0.0;
      }
    }
  }
}

// ------------------------------------------------------------------- CG
// setup() (SchurComplementConjugateGradient.cpp:89-100): p = s = b and, with a
// zero start, x = 0, r = b (r = b - S 0: the product is exactly zero and
// fma(-1, 0, b) = b) and the partials of r.r; q = z = 0; the flags of every
// system, live for those of the mask.
__global__ void __launch_bounds__(TPB) k_cg_start(CgVecs c, const double* __restrict__ rhs,
                                                  int x0_zero, CgFlags f, Batch b)
{
  const int s = blockIdx.y;
  const bool in = !b.mask || b.mask[s];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    f.live[s] = in ? 1 : 0;
    f.iters[s] = 0;
    f.status[s] = 0;
    // a system that takes no part reports ||r|| = 0, not a previous pass's
    at(c.sc, s, b)[CG_RR] = 0.0;
  }
  if (!in) return;
  rhs = at(rhs, s, b);
  double *p = at(c.p, s, b), *sv = at(c.s, s, b), *x = at(c.x, s, b), *r = at(c.r, s, b);
  double t = 0.0;
  for (int i = blockIdx.x * TPB + threadIdx.x; i < c.m; i += gridDim.x * TPB) {
    const double v = rhs[i];
    p[i] = v;
    sv[i] = v;
    if (x0_zero) {
      x[i] = 0.0;
      r[i] = v;
      t = fma(v, v, t);
    }
  }
  if (c.q) {
    double *q = at(c.q, s, b), *z = at(c.z, s, b);
    for (int i = blockIdx.x * TPB + threadIdx.x; i < c.n; i += gridDim.x * TPB) {
      q[i] = 0.0;
      z[i] = 0.0;
    }
  }
  if (!x0_zero) return;
  const double tot = block_sum(t);
  if (threadIdx.x == 0) at(c.part, s, b)[blockIdx.x] = tot;
}

// The stopping test after k updates (SchurComplementConjugateGradient.cpp:
// 164-170), rr = r.r: at the start r.r == 0 ends the system (x0 already solves
// it; the reference would divide 0/0), later sqrt(r.r) < tol (status 0) or the
// iteration limit (status 1).  `write`: the one thread per system that records
// it.  Returns whether the system has stopped.
__device__ __forceinline__ bool cg_stop(double rr, int k, double tol, int itmax, double* sc,
                                        const CgFlags& f, int s, bool write)
{
  const bool zero = k == 0 && rr == 0.0, conv = k > 0 && sqrt(rr) < tol;
  const bool limit = k > 0 && !conv && k >= itmax;
  if (write) {
    sc[CG_GAM + (k & 1)] = rr;
    sc[CG_RR] = rr;
    if (zero || conv || limit) {
      f.live[s] = 0;
      f.iters[s] = zero ? 0 : k;
      f.status[s] = limit ? 1 : 0;
    }
  }
  return zero || conv || limit;
}

// The start of S r after k updates: the stopping test on the partials of r.r (a
// system that stops does nothing more), the sweeps' buffers filled, t1 = Jh^T r.
// A workgroup may see `live` already cleared by its system's first one: both
// ways it stops.
__global__ void __launch_bounds__(TPB) k_cg_apply(CgVecs c, int k, double tol, int itmax,
                                                  const int* __restrict__ rp,
                                                  const int* __restrict__ ci,
                                                  const double* __restrict__ v, SweepFill fill,
                                                  CgFlags f, Batch b)
{
  __shared__ double lv[STAGE], lx[STAGE];
  __shared__ int alive;
  clear_tickets(fill.ticket);
  const int s = blockIdx.y;
  if (threadIdx.x == 0)   // one look for the whole workgroup
    alive = __hip_atomic_load(f.live + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (!alive) return;
  const double rr = sum_partials(at(c.part, s, b), reduce_blocks_of(c.m));
  if (cg_stop(rr, k, tol, itmax, at(c.sc, s, b), f, s, blockIdx.x == 0 && threadIdx.x == 0)) return;
  fill_sweep(fill, s, b, blockIdx.x, gridDim.x);
  v = at(v, s, b);
  const double* r = at(c.r, s, b);
  const int r0 = blockIdx.x * ROWS;
  const double t = row_sums(rp, r0, c.n, 0.0,
                            [&](int q, double& a, double& x) {
                              a = v[q];
                              x = r[ci[q]];
                            },
                            lv, lx);
  if (threadIdx.x < ROWS && r0 + threadIdx.x < c.n) at(c.t1, s, b)[r0 + threadIdx.x] = t;
}

// y = A x, ROWS rows per workgroup.
__global__ void __launch_bounds__(TPB) k_spmv_rows(int nrows, const int* __restrict__ rp,
                                                   const int* __restrict__ ci,
                                                   const double* __restrict__ v,
                                                   const double* __restrict__ xv,
                                                   double* __restrict__ y, Batch b)
{
  __shared__ double lv[STAGE], lx[STAGE];
  const int s = sys_of(b);
  if (s < 0) return;
  v = at(v, s, b);
  xv = at(xv, s, b);
  const int r0 = blockIdx.x * ROWS;
  const double t = row_sums(rp, r0, nrows, 0.0,
                            [&](int q, double& a, double& x) {
                              a = v[q];
                              x = xv[ci[q]];
                            },
                            lv, lx);
  if (threadIdx.x < ROWS && r0 + threadIdx.x < nrows) at(y, s, b)[r0 + threadIdx.x] = t;
}

// Iteration k's update once w = S r and the partials of w.r are there: delta =
// w.r, beta = gam1/gam, alpha = gam1/(delta - beta gam1/alpha) (:181-183; k = 0:
// alpha = gam/delta, beta = 0, :143), p = beta p + r, s = beta s + w, x += alpha
// p, r -= alpha s and the partials of r.r; and the image of the iterate under
// A^{-1} Jh^T carried along with it: q = beta q + t (t = A^{-1} Jh^T r, from this
// iteration's S r), z += alpha q, the same coefficients in the same forms, so z
// = A^{-1} Jh^T x without a solve.  gam and alpha of iteration k live in the slot
// of k's parity: no workgroup reads what another one writes.
__global__ void __launch_bounds__(TPB) k_cg_update(CgVecs c, int k, CgFlags f, Batch b)
{
  const int s = blockIdx.y;
  if (!f.live[s]) return;
  double* sc = at(c.sc, s, b);
  const double delta = sum_partials(at(c.part2, s, b), c.np2);
  const double gam = sc[CG_GAM + (k & 1)];
  double alpha, beta;
  if (k == 0) {
    alpha = gam / delta;
    beta = 0.0;
  } else {
    beta = gam / sc[CG_GAM + ((k - 1) & 1)];
    alpha = gam / (delta - beta * gam / sc[CG_ALPHA + ((k - 1) & 1)]);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) sc[CG_ALPHA + (k & 1)] = alpha;
  double *p = at(c.p, s, b), *sv = at(c.s, s, b), *x = at(c.x, s, b), *r = at(c.r, s, b);
  const double* w = at(c.w, s, b);
  double t = 0.0;
  for (int i = blockIdx.x * TPB + threadIdx.x; i < c.m; i += gridDim.x * TPB) {
    const double pi = beta * p[i] + r[i];
    const double si = beta * sv[i] + w[i];
    p[i] = pi;
    sv[i] = si;
    x[i] = fma(alpha, pi, x[i]);
    const double ri = fma(-alpha, si, r[i]);
    r[i] = ri;
    t = fma(ri, ri, t);
  }
  if (c.q) {
    double *q = at(c.q, s, b), *z = at(c.z, s, b);
    const double* tt = at(c.t2, s, b);
    for (int i = blockIdx.x * TPB + threadIdx.x; i < c.n; i += gridDim.x * TPB) {
      const double qi = beta * q[i] + tt[i];
      q[i] = qi;
      z[i] = fma(alpha, qi, z[i]);
    }
  }
  const double tot = block_sum(t);
  if (threadIdx.x == 0) at(c.part, s, b)[blockIdx.x] = tot;
}

// ------------------------------------------------------------- recovery
// recover_solution (HykktSolver.cpp:410-457): dx = (h0 - z) in natural order times
// max_d, dyc = x times max_d; s = Jd dx - ryd (Jd empty: -ryd), yd = s Ds - rs, the
// rows of Jd taking dx's values as this kernel forms them.  With base_*: each
// result is a correction, added to base's after it is rounded.
__global__ void __launch_bounds__(TPB) k_recover(Recover c, Batch b)
{
  __shared__ double lv[STAGE], lx[STAGE];
  const int s = sys_of(b);
  if (s < 0) return;
  const double *h0 = at(c.h0, s, b), *z = at(c.z, s, b), *md = at(c.max_d, s, b);
  auto dx_of = [&](int i) {
    const int j = c.ipos[i];
    const double t = h0[j] - z[j];
    return t * md[i];
  };
  const int tid = threadIdx.x, nx = static_cast<int>(gridDim.x) - c.nbd;
  const int blk = static_cast<int>(blockIdx.x) - nx;
  if (blk < 0) {
    double *dx = at(c.dx, s, b), *dyc = at(c.dyc, s, b);
    const double* cx = at(c.x, s, b);
    for (int i = blockIdx.x * TPB + tid; i < c.n || i < c.m; i += nx * TPB) {
      if (i < c.n) {
        const double t = dx_of(i);
        dx[i] = c.base_dx ? t + at(c.base_dx, s, b)[i] : t;
      }
      if (i < c.m) {
        const double t = cx[i] * md[c.n + i];
        dyc[i] = c.base_dyc ? t + at(c.base_dyc, s, b)[i] : t;
      }
    }
    return;
  }
  const int r0 = blk * ROWS, k = r0 + tid;
  const double* v = at(c.jd_v, s, b);
  double t = 0.0;
  if (c.has_jd)
    t = row_sums(c.jd_rp, r0, c.d, 0.0,
                 [&](int q, double& a, double& x) {
                   a = v[q];
                   x = dx_of(c.jd_ci[q]);
                 },
                 lv, lx);
  if (tid >= ROWS || k >= c.d) return;
  const double ryd = at(c.ryd, s, b)[k];
  // Jd*dx - ryd (HykktSolver.cpp:429-440); mult_const(-1) (:443)
  const double sv = c.has_jd ? fma(1.0, t, -1.0 * ryd) : ryd * -1.0;
  const double y = sv * at(c.ds, s, b)[k];                 // vec_scale (:447)
  const double yd = y + -1.0 * at(c.rs, s, b)[k];          // add_vecs(-1) (:448)
  at(c.dsv, s, b)[k] = c.base_dsv ? sv + at(c.base_dsv, s, b)[k] : sv;
  at(c.dyd, s, b)[k] = c.base_dyd ? yd + at(c.base_dyd, s, b)[k] : yd;
}

// ------------------------------------------------------------- residual
// check_error (HykktSolver.cpp:846-930) and rows 2 and 4: the signed residual
// rows, and per workgroup of ROWS rows the partial sums of their squares and of
// the right-hand side's: part[slot * stride + workgroup], slots 0..3 rows 1, 3,
// 2, 4, slots 4..7 rx, rs, ry, ryd.
__global__ void __launch_bounds__(TPB) k_residual(Residual c, Batch b)
{
  __shared__ double lv[STAGE], lx[STAGE];
  const int s = sys_of(b);
  if (s < 0) return;
  const double *dx = at(c.dx, s, b), *dyd = at(c.dyd, s, b);
  double* part = at(c.part, s, b);
  const int tid = threadIdx.x;
  const bool lead = tid < ROWS;
  auto put = [&](int slot, int blk, double v) {   // the first wave
    const double t = wave_sum(v);
    if (tid == 0) part[slot * c.stride + blk] = t;
  };
  int blk = blockIdx.x;
  if (blk < c.nbn) {
    // rx - H dx - Jc^T dyc - Jd^T dyd (the transposes through their maps)
    const int r0 = blk * ROWS, r = r0 + tid;
    const bool mine = lead && r < c.n;
    const double rx = mine ? at(c.rx, s, b)[r] : 0.0;
    const double *hv = at(c.h_v, s, b), *jcv = at(c.jc_v, s, b), *jdv = at(c.jd_v, s, b);
    const double* dyc = at(c.dyc, s, b);
    double t = row_sums(c.h_rp, r0, c.n, rx,
                        [&](int q, double& a, double& x) {
                          a = -hv[q];
                          x = dx[c.h_ci[q]];
                        },
                        lv, lx);
    t = row_sums(c.ct_rp, r0, c.n, t,
                 [&](int q, double& a, double& x) {
                   a = -jcv[c.ct_map[q]];
                   x = dyc[c.ct_ci[q]];
                 },
                 lv, lx);
    if (c.has_jd)
      t = row_sums(c.dt_rp, r0, c.n, t,
                   [&](int q, double& a, double& x) {
                     a = -jdv[c.dt_map[q]];
                     x = dyd[c.dt_ci[q]];
                   },
                   lv, lx);
    if (!lead) return;
    if (mine) at(c.e_x, s, b)[r] = t;
    put(0, blk, mine ? t * t : 0.0);
    put(4, blk, rx * rx);
    return;
  }
  blk -= c.nbn;
  if (blk < c.nbm) {
    // ry - Jc dx
    const int r0 = blk * ROWS, r = r0 + tid;
    const bool mine = lead && r < c.m;
    const double ry = mine ? at(c.ry, s, b)[r] : 0.0;
    const double* jcv = at(c.jc_v, s, b);
    const double t = row_sums(c.jc_rp, r0, c.m, ry,
                              [&](int q, double& a, double& x) {
                                a = -jcv[q];
                                x = dx[c.jc_ci[q]];
                              },
                              lv, lx);
    if (!lead) return;
    if (mine) at(c.e_y, s, b)[r] = t;
    put(1, blk, mine ? t * t : 0.0);
    put(6, blk, ry * ry);
    return;
  }
  blk -= c.nbm;
  // rs - (Ds ds - dyd), ryd - (Jd dx - ds)
  const int r0 = blk * ROWS, r = r0 + tid;
  const bool mine = lead && r < c.d;
  double jx = 0.0;
  if (c.has_jd) {
    const double* jdv = at(c.jd_v, s, b);
    jx = row_sums(c.jd_rp, r0, c.d, 0.0,
                  [&](int q, double& a, double& x) {
                    a = jdv[q];
                    x = dx[c.jd_ci[q]];
                  },
                  lv, lx);
  }
  if (!lead) return;
  double rs = 0.0, ryd = 0.0, a2 = 0.0, a4 = 0.0;
  if (mine) {
    const double dsv = at(c.dsv, s, b)[r];
    rs = at(c.rs, s, b)[r];
    ryd = at(c.ryd, s, b)[r];
    a2 = rs - (at(c.ds, s, b)[r] * dsv - dyd[r]);
    a4 = ryd - (jx - dsv);
    at(c.e_s, s, b)[r] = a2;
    at(c.e_d, s, b)[r] = a4;
  }
  put(2, blk, a2 * a2);
  put(3, blk, a4 * a4);
  put(5, blk, rs * rs);
  put(7, blk, ryd * ryd);
}

// ------------------------------------------------------------- results
// One workgroup per system: the CG's stopping test (k updates done), the
// residual's sums, and everything the host reads of a pass in `out` (FIN_SLOTS
// doubles per system; memory the host can read).
__global__ void __launch_bounds__(TPB) k_finish(Finish c, CgVecs v, int k, double tol, int itmax,
                                                CgFlags f, Batch b)
{
  const int s = sys_of(b);
  if (s < 0) return;
  double* sc = at(v.sc, s, b);
  double* out = c.out + static_cast<int64_t>(s) * FIN_SLOTS;
  if (f.live[s]) {
    const double rr = sum_partials(at(v.part, s, b), reduce_blocks_of(v.m));
    cg_stop(rr, k, tol, itmax, sc, f, s, threadIdx.x == 0);
  }
  if (c.part) {
    const double* part = at(c.part, s, b);
    const int lane = threadIdx.x & 63;
    for (int j = threadIdx.x >> 6; j < 8; j += TPB / 64) {
      const int np = c.np[j];
      const double* pj = part + j * c.stride;
      double t = 0.0;
      for (int i = lane; i < np; i += 64 * 8) {   // eight loads in flight
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = i + 64 * u < np ? pj[i + 64 * u] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++) t += v[u];
      }
      t = wave_sum(t);
      if (lane == 0) out[FIN_RES + j] = t;
    }
  }
  if (threadIdx.x == 0) {   // the thread that cg_stop wrote with
    out[FIN_RR] = sc[CG_RR];
    out[FIN_ITERS] = f.iters[s];
    out[FIN_STATUS] = f.status[s];
    out[FIN_LIVE] = f.live[s];
    out[FIN_ZERO_ROW] = c.zero_row ? c.zero_row[s] : INT_MAX;
    out[FIN_PIVOT] = c.pivot ? c.pivot[s] : INT_MAX;
    out[FIN_SWEEP_ERR] = c.sweep_err ? *c.sweep_err : 0;
  }
}

// dst[j] <- src[j] for the systems with keep[s] (null: all of them)
__global__ void k_keep(Keep c, const int* __restrict__ keep, Batch b)
{
  const int s = sys_of(b);
  if (s < 0 || (keep && !keep[s])) return;
  for (int j = 0; j < 4; j++) {
    const double* src = at(c.src[j], s, b);
    double* dst = at(c.dst[j], s, b);
    for (int i = blockIdx.x * TPB + threadIdx.x; i < c.n[j]; i += gridDim.x * TPB) dst[i] = src[i];
  }
}

inline int row_blocks(int rows) { return (rows + ROWS - 1) / ROWS; }

}  // namespace

#define LAUNCH_CHECK() HIPCHK(hipGetLastError())

void after_factor(const AfterFactor& c, const Batch& b, hipStream_t st, hipEvent_t start)
{
  if (b.count <= 0) return;
  const int len = std::max({c.nnz, c.n, c.m, c.d, 1});
  hipExtLaunchKernelGGL(k_after_factor, dim3(nblocks(len), b.count), dim3(TPB), 0, st, start,
                        nullptr, 0, c, b);
  LAUNCH_CHECK();
}

void cg_start(const CgVecs& c, const double* rhs, bool x0_zero, const CgFlags& f, const Batch& b,
              hipStream_t st)
{
  if (b.count <= 0) return;
  k_cg_start<<<dim3(reduce_blocks(c.m), b.count), TPB, 0, st>>>(c, rhs, x0_zero ? 1 : 0, f, b);
  LAUNCH_CHECK();
}

void cg_apply(const CgVecs& c, int k, double tol, int itmax, const int* jth_rp, const int* jth_ci,
              const double* jth_v, const SweepFill& fill, const CgFlags& f, const Batch& b,
              hipStream_t st)
{
  if (b.count <= 0) return;
  const int g = std::max(row_blocks(c.n), 1);
  k_cg_apply<<<dim3(g, b.count), TPB, 0, st>>>(c, k, tol, itmax, jth_rp, jth_ci, jth_v, fill, f, b);
  LAUNCH_CHECK();
}

void spmv_rows(int nrows, const int* rp, const int* ci, const double* v, const double* x, double* y,
               const Batch& b, hipStream_t st)
{
  if (b.count <= 0 || nrows <= 0) return;
  k_spmv_rows<<<dim3(row_blocks(nrows), b.count), TPB, 0, st>>>(nrows, rp, ci, v, x, y, b);
  LAUNCH_CHECK();
}

void cg_update(const CgVecs& c, int k, const CgFlags& f, const Batch& b, hipStream_t st)
{
  if (b.count <= 0) return;
  k_cg_update<<<dim3(reduce_blocks(c.m), b.count), TPB, 0, st>>>(c, k, f, b);
  LAUNCH_CHECK();
}

void recover(Recover c, const Batch& b, hipStream_t st, hipEvent_t start)
{
  if (b.count <= 0) return;
  c.nbd = row_blocks(c.d);
  const int nx = static_cast<int>(nblocks(std::max({c.n, c.m, 1})));
  hipExtLaunchKernelGGL(k_recover, dim3(nx + c.nbd, b.count), dim3(TPB), 0, st, start, nullptr, 0,
                        c, b);
  LAUNCH_CHECK();
}

int residual_partials(int n, int m, int d)
{
  return 8 * std::max({row_blocks(n), row_blocks(m), row_blocks(d), 1});
}

void residual(Residual& c, const Batch& b, hipStream_t st)
{
  c.nbn = row_blocks(c.n);
  c.nbm = row_blocks(c.m);
  c.nbd = row_blocks(c.d);
  c.stride = residual_partials(c.n, c.m, c.d) / 8;
  if (b.count <= 0 || c.nbn + c.nbm + c.nbd <= 0) return;
  k_residual<<<dim3(c.nbn + c.nbm + c.nbd, b.count), TPB, 0, st>>>(c, b);
  LAUNCH_CHECK();
}

void finish(Finish c, const Residual* r, const CgVecs& v, int k, double tol, int itmax,
            const CgFlags& f, const Batch& b, hipStream_t st, hipEvent_t stop)
{
  if (b.count <= 0) return;
  c.part = r ? r->part : nullptr;
  if (r) {
    const int np[8] = {r->nbn, r->nbm, r->nbd, r->nbd, r->nbn, r->nbd, r->nbm, r->nbd};
    std::copy(np, np + 8, c.np);
    c.stride = r->stride;
  }
  hipExtLaunchKernelGGL(k_finish, dim3(1, b.count), dim3(TPB), 0, st, nullptr, stop, 0, c, v, k,
                        tol, itmax, f, b);
  LAUNCH_CHECK();
}

void keep_where(const Keep& c, const int* keep, const Batch& b, hipStream_t st)
{
  if (b.count <= 0) return;
  const int len = std::max({c.n[0], c.n[1], c.n[2], c.n[3], 1});
  k_keep<<<dim3(nblocks(len), b.count), TPB, 0, st>>>(c, keep, b);
  LAUNCH_CHECK();
}

}  // namespace dev
}  // namespace hykkt
