// kernels_forest.hip -- the triangular-solve sweeps over the forest of small
// supernodes (gfx950): at most FOREST_NC columns and FOREST_F front rows each.
// See kernels_trsv.hip for the sweeps and how their items synchronise.
//
// One item per supernode and sweep, so the dependency chain has one link per
// tree level.  A lane owns a front row: everything it needs of the factor (its
// row of L, of the inverted diagonal block, its pull list) is loaded into
// registers before the first wait, and a link is the round trip of the awaited
// values, 2 nc (forward) or nc (backward) fused multiply-adds with broadcasts
// through v_readlane, and, backward, the column sums over the rows.
//
// These supernodes are tiny (median 12 columns on 36 rows), and a sweep is
// bound by latency: the depth of the tree on small systems, the number of
// resident items times an item's own loads on large ones and on batches.  So
// fronts of at most 64 rows (four of five) take one wave each, four supernodes
// of a level to a workgroup, with no barrier and no LDS; taller ones a
// workgroup, 256 rows at a time.  Against items of 128-row blocks, 256 threads
// each, forward pivots and updates apart: 1,000 buses 29 -> 15 us forward and
// 41 -> 12 backward, 10,000 buses 105 -> 28 and 127 -> 23, sixteen 1,000-bus
// systems 144 -> 34 and 165 -> 30.
#include <algorithm>

#include "sweep_dev.hpp"

namespace hykkt {
namespace dev {

namespace {

constexpr int NT = 256;
constexpr int SB = FRONT_NC;     // edge of an inverted diagonal block's slot
constexpr int NC = FOREST_NC;
constexpr int G = 8;             // columns per step of the unrolled loops

typedef double d2 __attribute__((ext_vector_type(2)));

// Lane j's value of v, wave-uniform.
__device__ __forceinline__ double rl(double v, int j)
{
  return mk64(__builtin_amdgcn_readlane(lo32(v), j), __builtin_amdgcn_readlane(hi32(v), j));
}

// One supernode (wave-uniform) of one system.
struct Sn {
  int a, nc, nr, f;
  const double* L;   // panel, column-major, f rows
  const double* W;   // inverted diagonal block, SB rows
  double* u;         // its forward update vector
  const int* pull_ptr;
  const int* rows;
};

__device__ __forceinline__ Sn load_sn(const CholDev& c, const SolveDev& sd, const SysBufs& B,
                                      int idx)
{
  const ForestSn& d = sd.forest[idx];
  Sn s;
  s.a = uni(d.a);
  s.nc = uni(d.nc);
  s.nr = uni(d.nr);
  s.f = s.nc + s.nr;
  s.L = B.L + uni64(d.l_off);
  s.W = B.dinv + uni64(d.dinv_off);
  s.u = B.ubuf + uni64(d.uvec_off);
  s.pull_ptr = sd.pull_ptr + uni64(d.front_off);
  s.rows = c.rows + uni64(d.rows_off);
  return s;
}

// m[j] = p[j * stride] for j < nc (j up to the next multiple of G repeats the
// last column).
__device__ __forceinline__ void load_cols(double (&m)[NC], const double* p, int64_t stride, int nc)
{
#pragma unroll
  for (int g = 0; g < NC; g += G) {
    if (g >= nc) break;
#pragma unroll
    for (int j = g; j < g + G; j++) m[j] = p[min(j, nc - 1) * stride];
  }
}

// sum_j m[j] v(j), j ascending, v(j) zero past nc (adds an exact zero).
template <class V>
__device__ __forceinline__ double dot_cols(const double (&m)[NC], int nc, V v)
{
  double t = 0.0;
#pragma unroll
  for (int g = 0; g < NC; g += G) {
    if (g >= nc) break;
#pragma unroll
    for (int j = g; j < g + G; j++) t = fma(m[j], j < nc ? v(j) : 0.0, t);
  }
  return t;
}

// The children's contributions to front row r, onto v.
__device__ __forceinline__ double pulls(const Sn& s, const SolveDev& sd, const double* ubuf, int r,
                                        double v)
{
  const int p0 = s.pull_ptr[r], n = s.pull_ptr[r + 1] - p0;
  return spin_sum<false>(v, n, [&](int p) { return ubuf + sd.pull_src[p0 + p]; }, sd.err);
}

// ---------------------------------------------------------------- forward
// y = Dinv (b + pulls) on the pivot rows, u = pulls - L y below.

// One wave, f <= 64: lane = front row.
__device__ __forceinline__ void fwd_small(const Sn& s, const SolveDev& sd, const SysBufs& B,
                                          int lane)
{
  const bool live = lane < s.f, piv = lane < s.nc;
  double m[NC];   // pivot lanes: a row of Dinv; the others: a row of L
  load_cols(m, piv ? s.W + lane : s.L + (live ? lane : 0), piv ? SB : s.f, s.nc);
  double v = piv ? B.in[s.a + lane] : 0.0;
  if (live) v = pulls(s, sd, B.ubuf, lane, v);
  const double y = dot_cols(m, s.nc, [&](int j) { return rl(v, j); });
  const double t = dot_cols(m, s.nc, [&](int j) { return rl(y, j); });
  if (piv) xstore(B.out + s.a + lane, y);
  else if (live) xstore(s.u + lane - s.nc, v - t);
}

// A workgroup: thread = front row, 256 rows at a time.
__device__ __forceinline__ void fwd_tall(const Sn& s, const SolveDev& sd, const SysBufs& B,
                                         double* ys)
{
  const int t = threadIdx.x;
  for (int r0 = 0; r0 < s.f; r0 += NT) {
    const int r = r0 + t;
    const bool live = r < s.f, piv = r < s.nc;
    double m[NC];
    load_cols(m, piv ? s.W + r : s.L + (live ? r : 0), piv ? SB : s.f, s.nc);
    double v = piv ? B.in[s.a + r] : 0.0;
    if (live) v = pulls(s, sd, B.ubuf, r, v);
    if (r0 == 0) {   // the pivot rows are in the first wave
      if (t < 64) {
        const double y = dot_cols(m, s.nc, [&](int j) { return rl(v, j); });
        if (piv) {
          ys[t] = y;
          xstore(B.out + s.a + t, y);
        }
      }
      __syncthreads();
    }
    if (live && !piv) {
      const double d = dot_cols(m, s.nc, [&](int j) { return ys[j]; });
      xstore(s.u + r - s.nc, v - d);
    }
  }
}

// --------------------------------------------------------------- backward
// x = Dinv^T (y - L^T x(rows)) on the pivot columns.

// The lane's value of column lane / 2 summed over the wave's 64 rows, from its
// row's terms acc[0..31] of all columns (fixed order).
__device__ __forceinline__ double col_sum32(double (&acc)[NC], int lane)
{
  static_assert(NC == 32, "one exchange level per bit of the lane index");
  halve_swap<32, true>(acc);
  halve_swap<16, false>(acc);
  halve<8, 8>(acc, lane);
  halve<4, 4>(acc, lane);
  halve<2, 2>(acc, lane);
  return acc[0] + xor_dpp<1>(acc[0], lane);
}

// Row r's entries of L (zero for rows outside [nc, f)); column j at stride f.
__device__ __forceinline__ void row_of_L(double (&l)[NC], const Sn& s, int r)
{
  const bool live = r >= s.nc && r < s.f;
  const uint32_t f8 = static_cast<uint32_t>(s.f) * 8u;
  const rsrc_t v = view(s.L, static_cast<uint32_t>(s.nc) * f8);
  const uint32_t vo = live ? static_cast<uint32_t>(r) * 8u : 0x80000000u;   // past the view: 0
#pragma unroll
  for (int g = 0; g < NC; g += G) {
    if (g < s.nc) {
#pragma unroll
      for (int j = g; j < g + G; j++)
        l[j] = ld(v, vo, static_cast<uint32_t>(min(j, s.nc - 1)) * f8);
    } else {
#pragma unroll
      for (int j = g; j < g + G; j++) l[j] = 0.0;
    }
  }
}

// Column i of the inverted diagonal block, rows j < nc (lane i; past nc the
// last one).
__device__ __forceinline__ void col_of_W(double (&w)[NC], const Sn& s, int lane)
{
  const double* p = s.W + static_cast<int64_t>(min(lane, s.nc - 1)) * SB;
#pragma unroll
  for (int g = 0; g < NC; g += G) {
    if (g >= s.nc) break;
#pragma unroll
    for (int j = g; j < g + G; j += 2) {
      const d2 t = *reinterpret_cast<const d2*>(p + j);
      w[j] = t[0];
      w[j + 1] = t[1];
    }
  }
}

__device__ __forceinline__ void bwd_small(const Sn& s, const SolveDev& sd, const SysBufs& B,
                                          int lane)
{
  double l[NC], w[NC];
  row_of_L(l, s, lane);
  col_of_W(w, s, lane);
  const int c = lane >> 1;
  const double y = c < s.nc ? B.in[s.a + c] : 0.0;
  double x = 0.0;
  if (lane >= s.nc && lane < s.f) x = spin_load(B.out + s.rows[lane - s.nc], sd.err);
#pragma unroll
  for (int j = 0; j < NC; j++) l[j] *= x;
  const double t = y - col_sum32(l, lane);   // lane 2 c: column c
  x = dot_cols(w, s.nc, [&](int j) { return rl(t, 2 * j); });
  if (lane < s.nc) xstore(B.out + s.a + lane, x);
}

__device__ __forceinline__ void bwd_tall(const Sn& s, const SolveDev& sd, const SysBufs& B,
                                         double (*part)[NC], double (*wl)[NC + 1])
{
  const int t = threadIdx.x, lane = t & 63, wave = uni(t >> 6);
  double l[NC], acc[NC];
  row_of_L(l, s, t);
  for (int e = t; e < s.nc * NC; e += NT) {   // Dinv(j, i) at wl[i][j], rows past nc zero
    const int i = e / NC, j = e % NC;
    wl[i][j] = s.W[i * SB + j];
  }
  const int c = lane >> 1;
  const double y = c < s.nc ? B.in[s.a + c] : 0.0;
#pragma unroll
  for (int j = 0; j < NC; j++) acc[j] = 0.0;
  for (int r0 = 0; r0 < s.f; r0 += NT) {
    const int r = r0 + t;
    if (r0 > 0) row_of_L(l, s, r);
    double x = 0.0;
    if (r >= s.nc && r < s.f) x = spin_load(B.out + s.rows[r - s.nc], sd.err);
#pragma unroll
    for (int j = 0; j < NC; j++) acc[j] = fma(l[j], x, acc[j]);
  }
  const double p = col_sum32(acc, lane);
  if ((lane & 1) == 0) part[wave][c] = p;
  __syncthreads();
  if (wave == 0) {
    const double tc = y - ((part[0][c] + part[1][c]) + (part[2][c] + part[3][c]));
    double w[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) w[j] = wl[min(lane, s.nc - 1)][j];
    const double x = dot_cols(w, s.nc, [&](int j) { return rl(tc, 2 * j); });
    if (lane < s.nc) xstore(B.out + s.a + lane, x);
  }
}

// ------------------------------------------------------------------ items
// An item is four words: four supernodes of one level, one wave each (-1:
// none), or (s, -2, ..): one tall supernode.
template <bool FWD>
__device__ __forceinline__ void forest_item(const CholDev& c, const SolveDev& sd,
                                            const double* __restrict__ in, double* __restrict__ out,
                                            const Batch& bt, int itc, double (*sh)[NC],
                                            double (*wl)[NC + 1])
{
  const int sy = itc % bt.count, it = itc / bt.count;
  if (bt.mask && !bt.mask[sy]) return;
  const SysBufs B = sys_bufs(c, sd, sy, bt, in, out);
  const int* w = (FWD ? sd.fwd_items : sd.bwd_items) + 4 * it;
  const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);
  if (uni(w[1]) == -2) {
    const Sn s = load_sn(c, sd, B, uni(w[0]));
    if constexpr (FWD) fwd_tall(s, sd, B, sh[0]);
    else bwd_tall(s, sd, B, sh, wl);
    return;
  }
  const int idx = uni(w[wave]);
  if (idx < 0) return;
  const Sn s = load_sn(c, sd, B, idx);
  if constexpr (FWD) fwd_small(s, sd, B, lane);
  else bwd_small(s, sd, B, lane);
}

// LOOP: a bounded grid whose workgroups take items until they run out (see
// k_solve_fwd); otherwise one item per workgroup.
template <bool FWD, bool LOOP>
__global__ void __launch_bounds__(NT) k_forest(CholDev c, SolveDev sd,
                                               const double* __restrict__ in,
                                               double* __restrict__ out, Batch bt, int total)
{
  __shared__ double sh[NT / 64][NC];
  __shared__ double wl[FWD ? 1 : NC][NC + 1];
  int* const ticket = sd.ticket + (FWD ? 0 : 3);
  if constexpr (!LOOP) {
    forest_item<FWD>(c, sd, in, out, bt, take_item(ticket), sh, wl);
    return;
  }
  for (;;) {
    const int itc = take_item(ticket);
    if (itc >= total) break;
    forest_item<FWD>(c, sd, in, out, bt, itc, sh, wl);
    __syncthreads();   // the item's last reads of sh and wl, and of take_item's word
  }
}

}  // namespace

int forest_blocks_per_cu()
{
  int nb = 0;
  HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_forest<true, true>, NT, 0));
  return std::max(nb, 1);
}

template <bool FWD>
static void launch_forest(const CholDev& c, const SolveDev& sd, const double* in, double* out,
                          const Batch& bt, hipStream_t st)
{
  const int items = FWD ? sd.n_fwd : sd.n_bwd;
  if (bt.count <= 0 || items <= 0) return;
  const int total = items * bt.count;
  if (sd.cap_forest > 0 && sd.cap_forest < total)
    k_forest<FWD, true><<<sd.cap_forest, NT, 0, st>>>(c, sd, in, out, bt, total);
  else
    k_forest<FWD, false><<<total, NT, 0, st>>>(c, sd, in, out, bt, total);
  HIPCHK(hipGetLastError());
}

void solve_forward_forest(const CholDev& c, const SolveDev& sd, const double* b, double* y,
                          const Batch& bt, hipStream_t st)
{
  launch_forest<true>(c, sd, b, y, bt, st);
}

void solve_backward_forest(const CholDev& c, const SolveDev& sd, const double* y, double* x,
                           const Batch& bt, hipStream_t st)
{
  launch_forest<false>(c, sd, y, x, bt, st);
}

}  // namespace dev
}  // namespace hykkt
