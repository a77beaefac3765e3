// kernels_trsv.hip -- supernodal triangular solves L y = b and L^T x = y as
// two single-launch sweeps over the whole elimination tree (gfx950).
//
// This file has the top of the tree (supernodes wider than the forest's, with
// tall fronts, and all their ancestors); kernels_forest.hip the forest of small
// supernodes below it.  Work items here are 128-row blocks of the supernodal
// fronts, 1024 threads each: thread (row = tid % 128, slice q = tid / 128) owns
// one row (forward) or one column (backward) of a 128 x 128 block and a 16-wide
// slice of the other index, so a whole block and an inverted diagonal block fit
// in registers.
//
// Forward sweep, per supernode s in postorder:
//   pivot item (s, b): waits for s's children's update vectors and for the
//     earlier pivot blocks of s, accumulates L(b, j) y_j as each y_j becomes
//     ready, and finishes with the inverted diagonal block:
//     y_b = Dinv_b (v - acc);
//   update item (s, u): the same products for 128 rows below s's columns,
//     written to s's update vector, which the parent pulls.
// Backward sweep, per supernode from the root down:
//   chunk item (s, u, b): the rows of chunk u of s are ancestors' columns, so
//     their x is final once computed there; the item computes
//     L(rows of chunk u, column block b)^T x(rows) into a partial-sum buffer
//     (all chunks of all column blocks run in parallel);
//   pivot item (s, b): sums the chunk partials in a fixed order, then
//     L(j, b)^T x_j over the later pivot blocks j > b as they finish, and
//     x_b = Dinv_b^T (t - acc);
// The L block of the next step, and the inverted diagonal block before the
// last wait, are loaded into registers before the item waits, so a link of
// the dependency chain costs the flag round trip and arithmetic only.
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
// (the forward y blocks, update vectors, backward chunk partials, backward x
// blocks) lives in a buffer that is filled with a sentinel NaN bit pattern
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

constexpr int SB = 128;                  // item rows / diagonal block size
constexpr int NT = 1024;                 // threads per item
constexpr int NQ = NT / SB, QW = SB / NQ;   // slices of a block, their width

struct SnInfo {
  int a, nc, nr, f, np, nu;
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
  i.np = (i.nc + SB - 1) / SB;
  i.nu = (i.nr + SB - 1) / SB;
  i.Ls = L + uni64(c.l_off[s]);
  return i;
}

// Fixed-order sum of the NQ slice partials of one row (column).
template <int NQ>
__device__ __forceinline__ double sum_slices(const double (*part)[SB], int i)
{
  double a = 0.0, b = 0.0;
#pragma unroll
  for (int k = 0; k < NQ; k += 2) {
    a += part[k][i];
    b += part[k + 1][i];
  }
  return a + b;
}

__global__ void k_fill_sentinel(SweepFill f, Batch bt)
{
  clear_tickets(f.ticket);
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  fill_sweep(f, sy, bt, blockIdx.x, gridDim.x);
}

// A slice of QW values, value k at byte offset vo + so0 + k*sstride of the
// view rs, for k < kvalid (uniform); other values and dead lanes read 0.
template <int QW>
__device__ __forceinline__ void slice_load(double (&v)[QW], rsrc_t rs, uint32_t vo, uint32_t so0,
                                           uint32_t sstride, int kvalid, bool live)
{
  const uint32_t vl = live ? vo : 0u;
#pragma unroll
  for (int k = 0; k < QW; k++) {
    const bool in = k < kvalid;
    const double t = ld(rs, vl, in ? so0 + static_cast<uint32_t>(k) * sstride : 0u);
    v[k] = (live && in) ? t : 0.0;
  }
}

template <int QW>
__device__ __forceinline__ double slice_dot(const double (&v)[QW], const double* vec)
{
  double a = 0.0;
#pragma unroll
  for (int k = 0; k < QW; k++) a += v[k] * vec[k];
  return a;
}

// ---------------------------------------------------------------- forward
// The L slice of the next step and the inverted diagonal block are prefetched
// into registers before the waits.
__device__ __forceinline__ void fwd_item(const CholDev& c, const SolveDev& sd,
                                         const int* __restrict__ items,
                                         const double* __restrict__ rhs,
                                         double* __restrict__ yout, const Batch& bt, int itc,
                                         double* yv, double (*part)[SB])
{
  const int sy = itc % bt.count, it = itc / bt.count;
  if (bt.mask && !bt.mask[sy]) return;
  const SysBufs B = sys_bufs(c, sd, sy, bt, rhs, yout);
  const double* b = B.in;
  double* y = B.out;
  const int s = uni(items[3 * it]);
  const int kind = uni(items[3 * it + 1]);
  const int blk = uni(items[3 * it + 2]);
  const SnInfo si = sninfo(c, B.L, s);
  const int r0 = (kind == 0) ? blk * SB : si.nc + blk * SB;
  const int rend = (kind == 0) ? min(si.nc, r0 + SB) : min(si.f, r0 + SB);
  const int nrows = rend - r0;
  const int row = threadIdx.x & (SB - 1);
  const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 7);   // whole waves per slice
  const bool live = row < nrows;
  const int r = r0 + row;
  const int jmax = (kind == 0) ? blk : si.np;
  const uint32_t f8 = static_cast<uint32_t>(si.f) * 8u;

  // row r of column block j: L(r, j*128 + q*QW + k)
  auto lview = [&](int j) {
    return view(si.Ls + static_cast<int64_t>(j) * SB * si.f,
                static_cast<uint32_t>(min(SB, si.nc - j * SB)) * f8);
  };
  auto lvalid = [&](int j) { return min(SB, si.nc - j * SB) - q * QW; };
  const uint32_t vo = static_cast<uint32_t>(r) * 8u;
  const uint32_t so = static_cast<uint32_t>(q * QW) * f8;
  // row `row` of the inverted diagonal block (upper part stored as zeros)
  const rsrc_t wv = view(B.dinv + uni64(c.dinv_off[s]) + static_cast<int64_t>(blk) * SB * SB,
                         SB * SB * 8u);
  const uint32_t wvo = static_cast<uint32_t>(row) * 8u, wso = static_cast<uint32_t>(q * QW) * SB * 8u;

  // Both slices are loaded up front: a load still in flight when the wave
  // polls for a value delays the poll (loads complete in order).
  double l[QW], w[QW];
  if (jmax > 0) slice_load<QW>(l, lview(0), vo, so, f8, lvalid(0), live);
  if (kind == 0) slice_load<QW>(w, wv, wvo, wso, SB * 8u, nrows - q * QW, live);

  // right-hand side plus the children's update-vector entries for this row
  // (each waited for as it is read)
  double v = 0.0;
  if (q == 0 && live) {
    v = (kind == 0) ? b[si.a + r] : 0.0;
    const int64_t fr = sd.front_off[s] + r;
    const int p0 = sd.pull_ptr[fr];
    v = spin_sum<false>(v, sd.pull_ptr[fr + 1] - p0,
                        [&](int p) { return B.ubuf + sd.pull_src[p0 + p]; }, sd.err);
  }
  // v -= L(r, B_j) y_j over the earlier pivot blocks, as each y_j is ready.
  // Step j's slice products go to part[j & 1]: it is written again two steps
  // on, after the next step's barriers, so a step needs two barriers.
  for (int j = 0; j < jmax; j++) {
    const int bj = min(SB, si.nc - j * SB);
    double (*pj)[SB] = part + (j & 1) * NQ;
    if (threadIdx.x < SB)
      yv[threadIdx.x] = (threadIdx.x < bj) ? spin_load(y + si.a + j * SB + threadIdx.x, sd.err) : 0.0;
    __syncthreads();
    pj[q][row] = slice_dot<QW>(l, yv + q * QW);
    __syncthreads();
    // the barrier keeps the next block's loads after the last use of l
    if (j + 1 < jmax) slice_load<QW>(l, lview(j + 1), vo, so, f8, lvalid(j + 1), live);
    if (q == 0) v -= sum_slices<NQ>(pj, row);
  }
  __syncthreads();   // part and yv are written again below
  if (kind == 0) {
    // y = Dinv_blk v
    if (q == 0) yv[row] = live ? v : 0.0;
    __syncthreads();
    part[q][row] = slice_dot<QW>(w, yv + q * QW);
    __syncthreads();
    if (q == 0 && live) xstore(y + si.a + r, sum_slices<NQ>(part, row));
  } else {
    if (q == 0 && live) xstore(B.ubuf + sd.uvec_off[s] + (r - si.nc), v);
  }
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
  __shared__ double yv[SB];
  __shared__ double part[2 * NQ][SB];
  if constexpr (!LOOP) {
    fwd_item(c, sd, items, rhs, yout, bt, take_item(sd.ticket + 1), yv, part);
    return;
  }
  for (;;) {
    const int itc = take_item(sd.ticket + 1);
    if (itc >= total) break;
    fwd_item(c, sd, items, rhs, yout, bt, itc, yv, part);
    __syncthreads();   // the item's last reads of yv and part
  }
}

// ---------------------------------------------------------------- backward
// Column sums of a 128 x 128 block product over 1024 threads: thread
// (row r = tid % 128, column slice q = tid / 128) holds acc[k], its row's
// term for column 16 q + k.  Within each wave the 16 values are
// transpose-reduced over the 64 lanes, then the two row halves of a slice meet
// in LDS.
// The two halves of the column sums: half[h][c] for the rows of wave
// parity h; all threads past a barrier.
__device__ __forceinline__ void column_halves(double (&acc)[16], double (*half)[SB])
{
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  halve_swap<16, true>(acc);
  halve_swap<8, false>(acc);
  halve<4, 8>(acc, lane);
  halve<2, 4>(acc, lane);
  acc[0] += xor_dpp<2>(acc[0], lane);
  acc[0] += xor_dpp<1>(acc[0], lane);
  // lane l now holds column k(l) = 8 b5 + 4 b4 + 2 b3 + b2 of its slice
  if ((lane & 3) == 0) {
    const int k = ((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 +
                  ((lane >> 2) & 1);
    half[wave & 1][(wave >> 1) * 16 + k] = acc[0];
  }
  __syncthreads();
}

// out[c] = the sum over the 128 rows for column c (all threads past a barrier).
__device__ __forceinline__ void column_sums(double (&acc)[16], double (*half)[SB], double* out)
{
  column_halves(acc, half);
  if (threadIdx.x < SB) out[threadIdx.x] = half[0][threadIdx.x] + half[1][threadIdx.x];
  __syncthreads();
}

// Top of the tree (1024 threads).  Loads run along rows (lanes = rows of L,
// coalesced); a thread keeps its row's terms for 16 columns across all the
// blocks it consumes and the column sums are formed once at the end.
//   chunk item (u, b): rows [nc + 128u, ...) of s against column block b:
//     bpart = L(rows, b-block)^T x(rows)
//   pivot item: columns [128 blk, ...): x = Dinv^T (y - sum of its chunks'
//     partials - L(later blocks, blk-block)^T x(later blocks))
__device__ __forceinline__ void solve_bwd_top(const CholDev& c, const SolveDev& sd,
                                              const SysBufs& B, int s, int kind, int idx,
                                              double* wl)
{
  static_assert(QW == 16, "column_halves sums 16 columns per thread");
  __shared__ double xs[2][SB];
  __shared__ double half[2][SB];
  __shared__ double cs[SB];
  __shared__ double ts[SB];
  __shared__ double part[8][SB];
  const double* __restrict__ y = B.in;
  double* __restrict__ x = B.out;
  const SnInfo si = sninfo(c, B.L, s);
  const int r = threadIdx.x & (SB - 1);
  const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 7);
  const uint32_t f8 = static_cast<uint32_t>(si.f) * 8u;
  double acc[QW];
#pragma unroll
  for (int k = 0; k < QW; k++) acc[k] = 0.0;
  // row r of the block of rows starting at r0 (nrows valid) and columns
  // starting at c0 (ncols valid): L(r0 + r, c0 + 16 q + k)
  auto row_slice = [&](double (&l)[QW], int r0, int nrows, int c0, int ncols) {
    const rsrc_t lv = view(si.Ls + static_cast<int64_t>(c0) * si.f,
                           static_cast<uint32_t>(ncols) * f8);
    slice_load<QW>(l, lv, static_cast<uint32_t>(r0 + r) * 8u, static_cast<uint32_t>(q * QW) * f8,
                   f8, ncols - q * QW, r < nrows);
  };

  if (kind == 0) {
    const int u = idx / si.np, b = idx - u * si.np;
    const int rr0 = u * SB;
    const int nrows = min(SB, si.nr - rr0);
    const int bb = min(SB, si.nc - b * SB);
    double l[QW];
    row_slice(l, si.nc + rr0, nrows, b * SB, bb);
    // x of these rows belongs to ancestors: waited for as it is read
    if (threadIdx.x < SB) {
      const int* rows = c.rows + c.rows_ptr[s] + rr0;
      xs[0][threadIdx.x] = (threadIdx.x < nrows) ? spin_load(x + rows[threadIdx.x], sd.err) : 0.0;
    }
    __syncthreads();
    const double xr = xs[0][r];
#pragma unroll
    for (int k = 0; k < QW; k++) acc[k] = l[k] * xr;
    column_sums(acc, half, cs);
    double* out = B.bpart + sd.bpart_off[s] + static_cast<int64_t>(u) * si.nc + b * SB;
    if (threadIdx.x < bb) xstore(out + threadIdx.x, cs[threadIdx.x]);
    return;
  }

  const int blk = idx;
  const int c0 = blk * SB;
  const int nb = min(SB, si.nc - c0);
  const int jtop = si.np - 1;   // later pivot blocks j = jtop .. blk+1
  // x = Dinv^T t: x(i) = sum_j Dinv(j, i) t(j), thread (i = r, slice q of j)
  const rsrc_t wv = view(B.dinv + uni64(c.dinv_off[s]) + static_cast<int64_t>(blk) * SB * SB,
                         SB * SB * 8u);
  // The inverse goes to LDS up front (wl[j * 128 + i] = Dinv(j, i), read
  // along Dinv's column i), so the last link reads no global memory before
  // its result.
  {
    double wt[QW];
    slice_load<QW>(wt, wv, static_cast<uint32_t>(r) * SB * 8u, static_cast<uint32_t>(q * QW) * 8u,
                   8u, nb - q * QW, r < nb);
#pragma unroll
    for (int k = 0; k < QW; k++) wl[(q * QW + k) * SB + r] = wt[k];
  }
  auto rows_of = [&](int j) { return min(SB, si.nc - j * SB); };
  double l[QW];
  if (jtop > blk) row_slice(l, jtop * SB, rows_of(jtop), c0, nb);

  if (threadIdx.x < SB) {
    double t = 0.0;
    if (threadIdx.x < nb) {
      t = y[si.a + c0 + threadIdx.x];
      const double* bp = B.bpart + sd.bpart_off[s] + c0 + threadIdx.x;
      t = spin_sum<true>(t, si.nu, [&](int u) { return bp + static_cast<int64_t>(u) * si.nc; },
                         sd.err);
    }
    ts[threadIdx.x] = t;
  }
  for (int j = jtop; j > blk; j--) {
    double* xb = xs[j & 1];
    if (threadIdx.x < SB)
      xb[threadIdx.x] = (threadIdx.x < rows_of(j)) ? spin_load(x + si.a + j * SB + threadIdx.x, sd.err) : 0.0;
    __syncthreads();   // xs[j & 1] is written again two blocks on, after the next barrier
    const double xr = xb[r];
#pragma unroll
    for (int k = 0; k < QW; k++) acc[k] += l[k] * xr;
    if (j - 1 > blk) row_slice(l, (j - 1) * SB, rows_of(j - 1), c0, nb);
  }
  // x = Dinv^T (t - column sums), the subtraction formed where it is used
  column_halves(acc, half);
  {
    double res = 0.0;
#pragma unroll
    for (int k = 0; k < QW; k++) {
      const int cc = q * QW + k;
      res += wl[cc * SB + r] * (ts[cc] - (half[0][cc] + half[1][cc]));
    }
    part[q][r] = res;
  }
  __syncthreads();
  if (threadIdx.x < nb) xstore(x + si.a + c0 + threadIdx.x, sum_slices<8>(part, threadIdx.x));
}

__device__ __forceinline__ void bwd_item(const CholDev& c, const SolveDev& sd,
                                         const int* __restrict__ items,
                                         const double* __restrict__ yin,
                                         double* __restrict__ xout, const Batch& bt, int itc,
                                         double* wl)
{
  const int sy = itc % bt.count, it = itc / bt.count;
  if (bt.mask && !bt.mask[sy]) return;
  solve_bwd_top(c, sd, sys_bufs(c, sd, sy, bt, yin, xout), uni(items[3 * it]),
                uni(items[3 * it + 1]), uni(items[3 * it + 2]), wl);
}

template <bool LOOP>
__global__ void __launch_bounds__(NT) k_solve_bwd(CholDev c, SolveDev sd,
                                                  const int* __restrict__ items,
                                                  const double* __restrict__ yin,
                                                  double* __restrict__ xout, Batch bt, int total)
{
  extern __shared__ double wl[];   // 128 x 128 inverse block (dynamic LDS)
  if constexpr (!LOOP) {
    bwd_item(c, sd, items, yin, xout, bt, take_item(sd.ticket + 2), wl);
    return;
  }
  for (;;) {
    const int itc = take_item(sd.ticket + 2);
    if (itc >= total) break;
    bwd_item(c, sd, items, yin, xout, bt, itc, wl);
    __syncthreads();   // the item's last reads of the shared arrays
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

// The top backward sweep stages one 128 x 128 inverse block in dynamic LDS.
constexpr size_t WL = static_cast<size_t>(SB) * SB * sizeof(double);

// Raise kernel K's dynamic LDS limit to WL, once per process and kernel (a
// function-local static initialises thread-safely).
template <auto K>
static void allow_top_lds()
{
  static const bool done = [] {
    HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(K),
                               hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(WL)));
    return true;
  }();
  (void)done;
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
  if (sd.cap_top > 0) {
    allow_top_lds<k_solve_bwd<true>>();
    k_solve_bwd<true><<<sweep_grid(total, sd.cap_top), NT, WL, st>>>(c, sd, sd.bwd_items_top, y, x,
                                                                     bt, total);
  } else {
    allow_top_lds<k_solve_bwd<false>>();
    k_solve_bwd<false><<<total, NT, WL, st>>>(c, sd, sd.bwd_items_top, y, x, bt, total);
  }
  HIPCHK(hipGetLastError());
}

}  // namespace dev
}  // namespace hykkt
