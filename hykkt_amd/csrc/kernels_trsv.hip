// kernels_trsv.hip -- supernodal triangular solves L y = b and L^T x = y as
// two single-launch sweeps over the whole elimination tree (gfx950).
//
// This file has the top of the tree (supernodes wider than the forest's, with
// tall fronts, and all their ancestors); kernels_forest.hip the forest of small
// supernodes below it.  Work items here are 1024 threads; the columns of a
// supernode go in groups of up to 512 (INV_GROUP), whose whole inverses the
// factorization leaves.
//
// Forward sweep, per supernode s in postorder:
//   pivot values of a group, 64 rows an item: y = X v with X the group's inverse and
//     v = b + the children's update vectors - the chunks of the groups before,
//     formed where it is read;
//   chunks, 64 rows an item: L y of one group, for each later group's rows;
//   rows below the columns, 128 to 1024 rows an item: the children's update vectors
//     - L y over all the groups, to s's update vector, which the parent pulls.
// Backward sweep, per supernode from the root down and per group from the last,
// items of 16 columns against 1024 rows at a time (a lane per row; for fewer rows
// more columns):
//   right-hand sides: t = y - L^T x over the rows below the group, the nearest
//     ancestor's last, as each becomes ready;
//   pivot values: x = X^T t.
// The entries a step needs are loaded into registers before the item waits, so a
// link of the dependency chain is the exchange's round trip (about 2 us between
// XCDs) and one product: two links for up to 512 columns, where 128-column blocks
// took one of 4 to 6 us each.  Top of the tree, forward / backward sweep: 1,000
// buses 25 / 41 -> 16 / 16 us, 5,000 107 / 151 -> 53 / 51, 10,000 304 / 319 -> 135 /
// 118, 20,000 748 / 694 -> 371 / 385 (its factor entries take 320 us at the rate of a
// large copy).  Chunks rather than items that follow all the groups before their
// rows, since those hold compute units while they wait (20,000, forward: 628 us);
// rows below in items of up to 1024 rows, since narrow supernodes on long fronts
// are most of the top's (64 rows each, with the chunks: 470).
//
// Items are numbered so that every item depends only on items with a
// smaller number, and a workgroup takes its item from a counter when it
// starts running (take_item), so the smallest unfinished item is always
// held by a running workgroup: the sweep cannot deadlock, also while other
// streams' kernels share the device.  Every wait is additionally bounded
// (SPIN_LIMIT); on expiry the item sets an error word the host reports, and
// carries on, so the kernel always terminates.
//
// Several systems of one pattern share a launch: launch item i*count + k is
// item i of system k, whose buffers (factor, right-hand side, exchanged
// values) sit k*vs doubles from system 0's.  The order property above holds
// for the combined numbering, and a system the mask skips returns at once.
//
// Synchronisation is by the data itself.  Every value passed between items
// (forward right-hand sides and y, update vectors, backward right-hand sides
// and x) lives in a buffer that is filled with a sentinel NaN bit pattern
// before the sweep -- a pattern arithmetic never produces -- and is written
// once, with a device-scope atomic store.  A consumer spins on each value it
// needs with device-scope atomic loads until the sentinel is gone.  Each
// value is thus published and observed on its own location, with no flags,
// no fences and no cross-location ordering (the eight XCDs' L2 caches are
// not coherent with each other; device-scope atomics go to the coherent
// level).  Factor values are plain loads: earlier kernels wrote them.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "basic_dev.hpp"
#include "sweep_dev.hpp"

namespace hykkt {
namespace dev {

namespace {

constexpr int NT = 1024;        // threads per item
constexpr int NW = NT / 64;     // waves
constexpr int CW = INV_GROUP / NW;   // most columns of a wave of a pivot or chunk item
constexpr int RW = 128, FC = 16;     // rows and columns of a wave of an item of rows below
constexpr int BC = 16;          // columns of a wave of a backward item

struct SnInfo {
  int a, nc, nr, f;
  const double* Ls;
};

// Supernode s (wave-uniform) of the factor L.
__device__ __forceinline__ SnInfo sninfo(const CholDev& c, const double* L, int s)
{
  SnInfo i;
  i.a = uni(c.sn_first[s]);
  i.nc = uni(c.sn_first[s + 1]) - i.a;
  i.nr = uni(c.rows_ptr[s + 1]) - uni(c.rows_ptr[s]);
  i.f = i.nc + i.nr;
  i.Ls = L + uni64(c.l_off[s]);
  return i;
}

__global__ void k_fill_sentinel(SweepFill f, Batch bt)
{
  clear_tickets(f.ticket);
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  fill_sweep(f, sy, bt, blockIdx.x, gridDim.x);
}

// l[k] = M(row, k) of a column-major matrix with leading dimension ld8 bytes, lane's
// byte offset vo, for the wave's columns c0 + k, k < cw (cw uniform, a multiple of 8;
// columns from n on repeat the last).
__device__ __forceinline__ void load_slice(double (&l)[CW], rsrc_t m, uint32_t vo, uint32_t ld8,
                                           int c0, int cw, int n)
{
#pragma unroll
  for (int k0 = 0; k0 < CW; k0 += 8) {
    if (k0 >= cw) break;
#pragma unroll
    for (int k = k0; k < k0 + 8; k++)
      l[k] = ld(m, vo, static_cast<uint32_t>(min(c0 + k, n - 1)) * ld8);
  }
}

// l . v, v's element k in lane k (0 past the wave's columns)
__device__ __forceinline__ double slice_dot(const double (&l)[CW], double v, int cw)
{
  double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k0 = 0; k0 < CW; k0 += 8) {
    if (k0 >= cw) break;
#pragma unroll
    for (int k = k0; k < k0 + 8; k++)
      s[k & 3] += l[k] * mk64(__builtin_amdgcn_readlane(lo32(v), k),
                              __builtin_amdgcn_readlane(hi32(v), k));
  }
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// Columns of each wave for a product with n columns.
__device__ __forceinline__ int wave_cols(int n) { return (n + 8 * NW - 1) / (8 * NW) * 8; }

// ---------------------------------------------------------------- forward
// v + the children's update-vector entries in front row q of supernode s, each waited
// for as it is read.
__device__ __forceinline__ double pulled(const SolveDev& sd, const SysBufs& B, int s, double v,
                                         int q)
{
  const int64_t fr = sd.front_off[s] + q;
  const int p0 = sd.pull_ptr[fr];
  return spin_sum<false, 4>(v, sd.pull_ptr[fr + 1] - p0,
                            [&](int p) { return B.ubuf + sd.pull_src[p0 + p]; }, sd.err);
}

// Pivot values and chunks: rows r0 .. r0 + 63 of the pivot block, a lane each, against
// up to 512 columns, spread over the waves.
__device__ __forceinline__ void fwd_pivot(const CholDev& c, const SolveDev& sd, const SysBufs& B,
                                          int s, int kind, int idx, int grp, double (*part)[RW])
{
  const SnInfo si = sninfo(c, B.L, s);
  const int lane = threadIdx.x & 63, w = uni(threadIdx.x >> 6);
  const int r0 = idx * TOP_ROWS, r = r0 + lane;
  const int g = kind == TOP_PIVOT ? r0 / INV_GROUP : grp, g0 = g * INV_GROUP;
  // columns: of the inverse those the rows reach
  const int n = kind == TOP_PIVOT ? min(si.nc, r0 + TOP_ROWS) - g0 : INV_GROUP;
  const int cw = wave_cols(n), c0 = w * cw, kv = min(n - c0, cw);
  double* ex = B.exch + uni64(sd.exch_off[s]);
  double l[CW], acc = 0.0;
  if (kv > 0) {
    if (kind == TOP_PIVOT) {
      const uint32_t ld8 = static_cast<uint32_t>(inv_ld(si.nc, g)) * 8u;
      load_slice(l, view(B.dinv + uni64(c.dinv_off[s]) +
                             static_cast<int64_t>(g) * INV_GROUP * INV_GROUP,
                         ld8 * static_cast<uint32_t>(n)),
                 static_cast<uint32_t>(min(r, si.nc - 1) - g0) * 8u, ld8, c0, cw, n);
    } else {
      const uint32_t f8 = static_cast<uint32_t>(si.f) * 8u;
      load_slice(l, view(si.Ls + static_cast<int64_t>(g0) * si.f, f8 * static_cast<uint32_t>(n)),
                 static_cast<uint32_t>(min(r, si.nc - 1)) * 8u, f8, c0, cw, n);
    }
    double v = 0.0;
    if (lane < kv) {
      const int q = g0 + c0 + lane;
      if (kind == TOP_PIVOT) {
        v = pulled(sd, B, s, B.in[si.a + q], q);
        v = spin_sum<true, 4>(
            v, g, [&](int j) { return ex + static_cast<int64_t>(j) * si.nc + q; }, sd.err);
      } else {
        v = spin_load(B.out + si.a + q, sd.err);
      }
    }
    acc = slice_dot(l, v, cw);
  }
  part[w][lane] = acc;
  __syncthreads();
  if (w == 0 && r < si.nc) {
    double t = part[0][lane];
#pragma unroll
    for (int k = 1; k < NW; k++) t += part[k][lane];
    xstore(kind == TOP_PIVOT ? B.out + si.a + r : ex + static_cast<int64_t>(g) * si.nc + r, t);
  }
}

// Rows below the columns: sets of 128 rows, two to a lane, against 16 columns of each
// of the set's waves at a time.  The last lane's pair ends at the last row, whichever
// of the two is its own.
__device__ __forceinline__ void fwd_below(const CholDev& c, const SolveDev& sd, const SysBufs& B,
                                          int s, int idx, double (*part)[RW], double* pull)
{
  const SnInfo si = sninfo(c, B.L, s);
  const int lane = threadIdx.x & 63, w = uni(threadIdx.x >> 6);
  const int wc = top_waves(si.nc), wk = w & (wc - 1);
  const int i0 = si.nc + idx * (NW / wc * RW), r0 = i0 + w / wc * RW;
  const int own = r0 + 2 * lane, r = min(own, si.f - 2);   // rows r and r + 1
  const uint32_t f8 = static_cast<uint32_t>(si.f) * 8u;
  d2v l[FC], acc = {0.0, 0.0};
  if (r0 < si.f) {
    auto load = [&](int c0) {   // columns from c0 + 16 wk on; past nc the last one again
      const int at = c0 + wk * FC;
      const rsrc_t L = view(si.Ls + static_cast<int64_t>(c0) * si.f,
                            static_cast<uint32_t>(min(wc * FC, si.nc - c0)) * f8);
#pragma unroll
      for (int k = 0; k < FC; k++)
        l[k] = ld2(L, static_cast<uint32_t>(r) * 8u,
                   static_cast<uint32_t>(min(at + k, si.nc - 1) - c0) * f8);
    };
    load(0);
    // the children's entries in the item's rows, a row a thread (from this set's first on)
    const int t = threadIdx.x;
    if (t < NW / wc * RW && i0 + t < si.f) pull[t] = pulled(sd, B, s, 0.0, i0 + t);
    for (int c0 = 0, at = wk * FC; at < si.nc;) {
      const int kv = min(si.nc - at, FC);
      const double yv = lane < kv ? spin_load(B.out + si.a + at + lane, sd.err) : 0.0;
#pragma unroll
      for (int k = 0; k < FC; k++) {
        const double yk = mk64(__builtin_amdgcn_readlane(lo32(yv), k),
                               __builtin_amdgcn_readlane(hi32(yv), k));
        acc[0] += l[k][0] * yk;
        acc[1] += l[k][1] * yk;
      }
      // the sums before the next slice's loads: after them they would keep both slices
      // in registers (and 84 bytes a lane in scratch)
      asm volatile("" : "+v"(acc[0]), "+v"(acc[1]) : : "memory");
      c0 += wc * FC;
      at += wc * FC;
      if (at >= si.nc) break;
      load(c0);
    }
  }
  *reinterpret_cast<d2v*>(&part[w][2 * lane]) = acc;
  __syncthreads();
  if (wk == 0 && r0 < si.f) {
    d2v t = *reinterpret_cast<const d2v*>(&part[w][2 * lane]);
    for (int k = 1; k < wc; k++) t += *reinterpret_cast<const d2v*>(&part[w + k][2 * lane]);
    double* u = B.ubuf + sd.uvec_off[s] - si.nc;
    if (r == own) xstore(u + r, pull[r - i0] - t[0]);
    if (r + 1 >= own) xstore(u + r + 1, pull[r + 1 - i0] - t[1]);
  }
}

__device__ __forceinline__ void fwd_item(const CholDev& c, const SolveDev& sd,
                                         const int* __restrict__ items,
                                         const double* __restrict__ rhs,
                                         double* __restrict__ yout, const Batch& bt, int itc,
                                         double (*part)[RW], double* pull)
{
  const int sy = itc % bt.count, it = itc / bt.count;
  if (bt.mask && !bt.mask[sy]) return;
  const SysBufs B = sys_bufs(c, sd, sy, bt, rhs, yout);
  const int s = uni(items[4 * it]), kind = uni(items[4 * it + 1]), idx = uni(items[4 * it + 2]);
  if (kind == TOP_BELOW) fwd_below(c, sd, B, s, idx, part, pull);
  else fwd_pivot(c, sd, B, s, kind, idx, uni(items[4 * it + 3]), part);
}

// LOOP: persistent; a workgroup takes items from the sweep's counter until
// they run out, so the grid may be smaller than the item list (fewer resident
// workgroups leave compute units to other streams); the order argument above
// holds for any grid size.  Otherwise one item per workgroup, one workgroup
// per item (fewer registers on the item's path).
template <bool LOOP>
__global__ void __launch_bounds__(NT) k_solve_fwd(CholDev c, SolveDev sd,
                                                  const int* __restrict__ items,
                                                  const double* __restrict__ rhs,
                                                  double* __restrict__ yout, Batch bt, int total)
{
  __shared__ __attribute__((aligned(16))) double part[NW][RW];
  __shared__ double pull[NT];
  if constexpr (!LOOP) {
    fwd_item(c, sd, items, rhs, yout, bt, take_item(sd.ticket + 1), part, pull);
    return;
  }
  for (;;) {
    const int itc = take_item(sd.ticket + 1);
    if (itc >= total) break;
    fwd_item(c, sd, items, rhs, yout, bt, itc, part, pull);
    __syncthreads();   // the item's last reads of part and pull
  }
}

// ---------------------------------------------------------------- backward
// A lane holds a row's terms of 16 columns over all the rows it takes; the sums over
// the lanes are formed once, at the end, by exchanges that halve the values a lane
// holds, then over the waves through LDS.
__device__ __forceinline__ void bwd_item(const CholDev& c, const SolveDev& sd,
                                         const int* __restrict__ items,
                                         const double* __restrict__ yin,
                                         double* __restrict__ xout, const Batch& bt, int itc,
                                         double (*red)[BC])
{
  const int sy = itc % bt.count, it = itc / bt.count;
  if (bt.mask && !bt.mask[sy]) return;
  const SysBufs B = sys_bufs(c, sd, sy, bt, yin, xout);
  const double* y = B.in;
  double* x = B.out;
  double* rh = B.exch;   // right-hand sides of the groups
  const int s = uni(items[4 * it]), kind = uni(items[4 * it + 1]), q0 = uni(items[4 * it + 2]);
  const SnInfo si = sninfo(c, B.L, s);
  const int lane = threadIdx.x & 63, w = uni(threadIdx.x >> 6);
  const int g = q0 / INV_GROUP, g0 = g * INV_GROUP, g1 = min(si.nc, g0 + INV_GROUP);
  const int shape = top_shape(kind == TOP_RHS ? si.f - g1 : g1 - g0);
  const int rows = NT >> shape, wps = NW >> shape;   // of a step; waves of a set of columns
  const int row = threadIdx.x & (rows - 1);
  const int q = q0 + w / wps * BC;                   // the wave's columns
  const int kv = min(g1 - q, BC);
  double l[BC], acc[BC], yq = 0.0;
#pragma unroll
  for (int k = 0; k < BC; k++) acc[k] = 0.0;
  const int mine = q0 + static_cast<int>(threadIdx.x);   // the column this thread finishes
  const bool fin = threadIdx.x < (BC << shape) && mine < g1;
  if (kind == TOP_RHS) {
    if (fin) yq = y[si.a + mine];
    if (kv > 0) {
      const uint32_t f8 = static_cast<uint32_t>(si.f) * 8u;
      const rsrc_t L = view(si.Ls + static_cast<int64_t>(q) * si.f, static_cast<uint32_t>(kv) * f8);
      const int* below = c.rows + uni(c.rows_ptr[s]);
      int at = 0;   // x of the step's row
      auto load = [&](int step) {
        const int r = min(g1 + step * rows + row, si.f - 1);
        at = r < si.nc ? si.a + r : below[r - si.nc];
#pragma unroll
        for (int k = 0; k < BC; k++)
          l[k] = ld(L, static_cast<uint32_t>(r) * 8u, static_cast<uint32_t>(min(k, kv - 1)) * f8);
      };
      int step = (si.f - g1 + rows - 1) / rows - 1;
      load(step);
      for (; step >= 0; step--) {
        const double xr = g1 + step * rows + row < si.f ? spin_load(x + at, sd.err) : 0.0;
#pragma unroll
        for (int k = 0; k < BC; k++) acc[k] += l[k] * xr;
        if (step > 0) load(step - 1);
      }
    }
  } else if (kv > 0) {
    // rows above the wave's first column hold zeros
    const bool in = g0 + row >= q && g0 + row < g1;
    const uint32_t ld8 = static_cast<uint32_t>(inv_ld(si.nc, g)) * 8u;
    const rsrc_t X = view(B.dinv + uni64(c.dinv_off[s]) +
                              static_cast<int64_t>(g) * INV_GROUP * INV_GROUP,
                          ld8 * static_cast<uint32_t>(g1 - g0));
#pragma unroll
    for (int k = 0; k < BC; k++)
      l[k] = ld(X, in ? static_cast<uint32_t>(row) * 8u : 0u,
                static_cast<uint32_t>(q - g0 + min(k, kv - 1)) * ld8);
    // the last rows' right-hand side is y itself
    const double t = !in ? 0.0 : g1 == si.f ? y[si.a + g0 + row]
                                            : spin_load(rh + si.a + g0 + row, sd.err);
#pragma unroll
    for (int k = 0; k < BC; k++) acc[k] = in ? l[k] * t : 0.0;
  }
  halve_swap<16, true>(acc);
  halve_swap<8, false>(acc);
  halve<4, 8>(acc, lane);
  halve<2, 4>(acc, lane);
  acc[0] += xor_dpp<2>(acc[0], lane);
  acc[0] += xor_dpp<1>(acc[0], lane);
  // lane l now holds column 8 b5 + 4 b4 + 2 b3 + b2
  if ((lane & 3) == 0)
    red[w][((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 +
           ((lane >> 2) & 1)] = acc[0];
  __syncthreads();
  if (fin) {
    const int w0 = static_cast<int>(threadIdx.x) / BC * wps, k = threadIdx.x & (BC - 1);
    double t = red[w0][k];
    for (int j = 1; j < wps; j++) t += red[w0 + j][k];
    if (kind == TOP_RHS) xstore(rh + si.a + mine, yq - t);
    else xstore(x + si.a + mine, t);
  }
}

template <bool LOOP>
__global__ void __launch_bounds__(NT) k_solve_bwd(CholDev c, SolveDev sd,
                                                  const int* __restrict__ items,
                                                  const double* __restrict__ yin,
                                                  double* __restrict__ xout, Batch bt, int total)
{
  __shared__ double red[NW][BC];
  if constexpr (!LOOP) {
    bwd_item(c, sd, items, yin, xout, bt, take_item(sd.ticket + 2), red);
    return;
  }
  for (;;) {
    const int itc = take_item(sd.ticket + 2);
    if (itc >= total) break;
    bwd_item(c, sd, items, yin, xout, bt, itc, red);
    __syncthreads();   // the item's last reads of red
  }
}

}  // namespace

void fill_sentinel(const SweepFill& f, const Batch& b, hipStream_t st)
{
  if (b.count <= 0) return;
  int64_t n = 1;
  for (int j = 0; j < 4; j++) n = std::max(n, f.n[j]);
  k_fill_sentinel<<<dim3(nblocks(n), b.count), TPB, 0, st>>>(f, b);
  HIPCHK(hipGetLastError());
}

// Workgroups of a persistent sweep launch: one per item, at most `cap` (0:
// no bound).
static unsigned sweep_grid(int items, int cap)
{
  const int g = cap > 0 ? std::min(items, cap) : items;
  return static_cast<unsigned>(std::max(g, 1));
}

void solve_forward_top(const CholDev& c, const SolveDev& sd, const double* b, double* y,
                       const Batch& bt, hipStream_t st)
{
  if (bt.count <= 0 || sd.n_fwd_top <= 0) return;
  const int total = sd.n_fwd_top * bt.count;
  if (sd.cap_top > 0)
    k_solve_fwd<true><<<sweep_grid(total, sd.cap_top), NT, 0, st>>>(c, sd, sd.fwd_items_top, b, y,
                                                                    bt, total);
  else
    k_solve_fwd<false><<<total, NT, 0, st>>>(c, sd, sd.fwd_items_top, b, y, bt, total);
  HIPCHK(hipGetLastError());
}

void solve_backward_top(const CholDev& c, const SolveDev& sd, const double* y, double* x,
                        const Batch& bt, hipStream_t st)
{
  if (bt.count <= 0 || sd.n_bwd_top <= 0) return;
  const int total = sd.n_bwd_top * bt.count;
  if (sd.cap_top > 0)
    k_solve_bwd<true><<<sweep_grid(total, sd.cap_top), NT, 0, st>>>(c, sd, sd.bwd_items_top, y, x,
                                                                    bt, total);
  else
    k_solve_bwd<false><<<total, NT, 0, st>>>(c, sd, sd.bwd_items_top, y, x, bt, total);
  HIPCHK(hipGetLastError());
}

}  // namespace dev
}  // namespace hykkt
