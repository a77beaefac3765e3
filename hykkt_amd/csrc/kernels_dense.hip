// kernels_dense.hip -- dense FP64 kernels of the supernodal Cholesky on
// gfx950: NT-GEMM updates on the matrix cores (v_mfma_f64_16x16x4f64), and the
// factorization + inversion of 128x128 diagonal blocks.
//
// MFMA f64 16x16x4 operand layout on gfx950 (lane l, 64 lanes):
//   A operand: A[i = l%16][k = l/16];  B operand: B[k = l/16][j = l%16];
//   result element v (0..3): D[i = 4v + l/16][j = l%16].
// The GEMM computes C(r, c) = beta*C(r, c) + alpha * sum_k A(r, k) * B(c, k)
// with A, B, C column-major.  It feeds the MFMA with B's rows as the A
// operand and A's rows as the B operand, so each result register holds 16
// consecutive rows of one C column (coalesced column-major stores).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "batch_dev.hpp"
#include "kernels.hpp"

namespace hykkt {
namespace dev {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int BT = 128;        // tile edge (rows and columns of C)
constexpr int KC = 16;         // K chunk staged in LDS
constexpr int LDA_S = BT + 2;  // LDS row length (doubles)

struct GemmArgs {
  const double* A;
  int64_t lda;
  const double* B;
  int64_t ldb;
  double* C;
  int64_t ldc;
  int M, N, K;   // C is M x N (tile-local bounds), K inner
};

// One TM x TN tile of C = A*B^T.  256 threads: 4 waves in a WM x WN
// arrangement (2x2 for 128x128 tiles, 1x4 for 32x128), each owning a QM x QN
// block of IM x JN MFMA tiles, stored once at the end.  K is staged through
// LDS in chunks of KC, the next chunk's global loads overlapping the current
// chunk's MFMAs.
template <int TM, int TN>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, double* smem)
{
  constexpr int WN = TM == TN ? 2 : 4, WM = 4 / WN;
  constexpr int QM = TM / WM, QN = TN / WN, IM = QM / 16, JN = QN / 16;
  constexpr int LA = TM + 2, LB = TN + 2;          // LDS row lengths (doubles)
  constexpr int EA = TM / 16, EB = TN / 16;        // staged elements per thread
  double* As = smem;                               // [KC][LA]
  double* Bs = smem + KC * LA;                     // [KC][LB]
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int wr = (wave / WN) * QM, wc = (wave % WN) * QN;
  d4 acc[IM][JN];
  // acc[i][j][v]: C row = wr + 16 i + lane%16, C col = wc + 16 j + 4 v + lane/16
#pragma unroll
  for (int i = 0; i < IM; i++)
#pragma unroll
    for (int j = 0; j < JN; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

  // staging assignment: thread t loads k = t/16, rows t%16 + 16 q (q < E): the
  // 16 lanes of a k write 16 consecutive LDS words (no bank conflicts)
  const int sk = t >> 4, sa = t & 15, sb = t & 15;
  double ra[EA], rb[EB];
  auto gload = [&](int k0) {
    const int kk = k0 + sk;
#pragma unroll
    for (int q = 0; q < EA; q++) {
      const int r = sa + 16 * q;
      ra[q] = (kk < g.K && r < g.M) ? g.A[kk * g.lda + r] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < EB; q++) {
      const int r = sb + 16 * q;
      rb[q] = (kk < g.K && r < g.N) ? g.B[kk * g.ldb + r] : 0.0;
    }
  };
  gload(0);
  for (int k0 = 0; k0 < g.K; k0 += KC) {
    __syncthreads();   // the previous chunk's fragments have been read
#pragma unroll
    for (int q = 0; q < EA; q++) As[sk * LA + sa + 16 * q] = ra[q];
#pragma unroll
    for (int q = 0; q < EB; q++) Bs[sk * LB + sb + 16 * q] = rb[q];
    __syncthreads();
    if (k0 + KC < g.K) gload(k0 + KC);
#pragma unroll
    for (int ks = 0; ks < KC / 4; ks++) {
      const int kr = ks * 4 + (lane >> 4);
      double fa[IM], fb[JN];
#pragma unroll
      for (int i = 0; i < IM; i++) fa[i] = As[kr * LA + wr + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < JN; j++) fb[j] = Bs[kr * LB + wc + j * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < IM; i++)
#pragma unroll
        for (int j = 0; j < JN; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < IM; i++) {
    const int r = wr + i * 16 + (lane & 15);
#pragma unroll
    for (int j = 0; j < JN; j++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int c = wc + j * 16 + 4 * v + (lane >> 4);
        if (r < g.M && c < g.N) g.C[c * g.ldc + r] = acc[i][j][v];
      }
  }
}

struct SnInfo {
  int a, nc, nr, f;
  double* Ls;
};

__device__ __forceinline__ SnInfo sninfo(const CholDev& c, double* L, int s)
{
  SnInfo i;
  i.a = c.sn_first[s];
  i.nc = c.sn_first[s + 1] - i.a;
  i.nr = c.rows_ptr[s + 1] - c.rows_ptr[s];
  i.f = i.nc + i.nr;
  i.Ls = L + c.l_off[s];
  return i;
}

// ------------------------------------------------------------- updates
// Buffer descriptors over factor data: a uniform base, so a load costs one
// 32-bit offset register, and a byte limit past which loads return 0 (word 3:
// the gfx9-family raw-buffer setting).
using rsrc_t = __amdgpu_buffer_rsrc_t;
typedef double d2 __attribute__((ext_vector_type(2)));
constexpr uint32_t VIEW_MAX = 0x7fffffffu;
constexpr uint32_t OFF_NONE = 0x80000000u;   // past every view: the load returns 0

__device__ __forceinline__ int64_t uni64(int64_t v)
{
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi =
      __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(static_cast<uint64_t>(v) >> 32));
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ rsrc_t view(const double* base, int64_t bytes)
{
  const int64_t n = bytes < 0 ? 0 : (bytes > VIEW_MAX ? VIEW_MAX : bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(base), 0, static_cast<uint32_t>(n),
                                           0x00020000);
}

// Row (column) of group g's element m (0..15) within a wave's block of CNT
// groups of 16: with an even CNT the groups come in pairs of interleaved rows,
// so the two groups' values of a lane are adjacent in memory (one 16-byte
// load or store instead of two of 8 bytes).
template <int CNT>
__device__ __forceinline__ constexpr int grow16(int g, int m)
{
  return CNT % 2 == 0 ? (g / 2) * 32 + 2 * m + (g & 1) : 16 * g + m;
}

// A lane's values of CNT groups of 16 rows of one matrix column (k), from the
// view whose element (0, k) is at byte offset vo (the lane's row included).
template <int CNT>
__device__ __forceinline__ void frag_load(double (&v)[CNT], rsrc_t r, uint32_t vo)
{
  if constexpr (CNT % 2 == 0) {
#pragma unroll
    for (int g = 0; g < CNT; g += 2) {
      const d2 t = __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, vo, g * 128, 0));
      v[g] = t[0];
      v[g + 1] = t[1];
    }
  } else {
#pragma unroll
    for (int g = 0; g < CNT; g++)
      v[g] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, vo, g * 128, 0));
  }
}

__device__ __forceinline__ int rl32(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ int64_t rl64(int v, int lane)
{
  const uint32_t lo = rl32(v, lane), hi = rl32(v, lane + 1);
  return static_cast<int64_t>((static_cast<uint64_t>(hi) << 32) | lo);
}

// Supernode s's record, wave-uniform: one load, a word per lane, instead of one
// per field, each waited for.
struct Sn {
  int a, nc, nr, f, nch, stride;
  int64_t l_off, dinv_off, u_off;
  const ChildRec* rec;   // of its first child
  const int* inv;        // of child 0, indexed by front row; child t's t * stride further
};

__device__ __forceinline__ Sn load_sn(const CholDev& c, int s, int lane)
{
  static_assert(sizeof(SnRec) == 64, "sixteen words");
  const int w = reinterpret_cast<const int*>(c.sn_rec + s)[lane & 15];
  Sn r;
  r.a = rl32(w, 0);
  r.nc = rl32(w, 1);
  r.nr = rl32(w, 2);
  r.f = r.nc + r.nr;
  r.rec = c.child_rec + rl32(w, 3);
  r.nch = rl32(w, 4);
  r.stride = rl32(w, 5);
  r.l_off = rl64(w, 8);
  r.dinv_off = rl64(w, 10);
  r.u_off = rl64(w, 12);
  r.inv = c.inv + rl64(w, 14);
  return r;
}

// The records of CG children from the t0-th on (past the last: the last one's),
// one load: child g's in lanes 4 g .. 4 g + 3.
template <int CG>
__device__ __forceinline__ int child_words(const Sn& r, int t0, int lane)
{
  static_assert(sizeof(ChildRec) == 16 && CG <= 16, "four words a child");
  const int g = min(lane >> 2, CG - 1);
  return reinterpret_cast<const int*>(r.rec + min(t0 + g, r.nch - 1))[lane & 3];
}

// mode 0: trailing panel update after block `step`   C = C - A A^T (K = block)
// mode 1: update matrix U = -L21 L21^T + children      (K = nc, U written)
// mode m >= 3: as mode 0 after blocks `step` .. `step`+m-2 (K = m-1 blocks)
//
// Each wave holds a (16 IM) x (16 JN) block of C in accumulators and reads its
// A and B fragments straight from global memory into registers, D K-steps (of
// 4) ahead of the MFMAs that use them: no LDS, no barriers, so the waves of a
// CU never wait for each other and the whole LDS stays free for the chain's
// kernels (a diagonal block fits beside two update tiles).  A fragment read
// by two waves of a tile comes from L1/L2 the second time.  The updates are
// bound by the FP64 matrix cores: on a 12288 x 12288 C, K = 1024 / 512 / 256 /
// 128 run at 72 / 68 / 60 / 47 TFLOP/s (LDS-staged with two barriers per 16
// K-steps: 60 / 56 / 50 / 40; LDS double-buffered, one barrier: 67 / 64 / 57 /
// 49); at small K the C traffic takes over.  D = 2 leaves the 128 x 128 tile
// at two waves per SIMD with registers over for a diagonal block.
//
// An update matrix takes its children's as the tile is finished, read once and
// straight into the accumulators: a pass of its own over U, read and written again
// per child, made the two 3190 us of a pass at 10,000 buses, now 2806 (eight systems
// at 5,000: 2245 for the second pass alone, now 2319 in all).
//
// Every C entry starts from its old value (modes 0, >= 3) or 0 and takes the
// MFMAs of K in ascending order, whatever the tile shape.  Rows and columns of
// a tile past the panel compute values that are not stored (their loads stay
// in the panel, or return 0 past its end); K steps past K read 0 for both
// operands.
//
// WN waves along the columns, TM / (16 IM) along the rows, on TM rows; a tile's 128
// columns are split over gridDim.z workgroups of 16 JN WN columns (64 x 64 tiles: its
// four quarters).  System blockIdx.y.
// U: mode 1 (a kernel of its own, so that the others keep their registers).
template <bool U, int TM, int IM, int JN, int WN, int D>
__global__ void __launch_bounds__(TM / IM * WN * 4, TM / IM * WN / 32)
    k_dense_nt(CholDev c, const int* __restrict__ tsn, const int* __restrict__ ttr,
               const int* __restrict__ ttc, int mode, int step, Batch bt)
{
  constexpr int QM = 16 * IM, QN = 16 * JN, TN = QN * WN;
  // mode 1: children whose indices, column quarters whose entries are in flight
  constexpr int CG = IM * JN > 4 ? 1 : 4, VG = IM * JN > 4 ? 2 : 4;
  static_assert(TM / QM * WN == 4 || TM / QM * WN == 8, "four or eight waves");
  // the 32-row launches are the factorization's critical chain: their waves
  // take issue priority over the trailing updates they share SIMDs with
  if constexpr (TM == 32) __builtin_amdgcn_s_setprio(3);
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);
  const int s = uni(tsn[blockIdx.x]), tr = uni(ttr[blockIdx.x]), tc = uni(ttc[blockIdx.x]);
  const Sn sn = load_sn(c, s, lane);
  const int nc = sn.nc, nr = sn.nr, f = sn.f;
  const double* Ls = batch_at(c.L, sy, bt) + sn.l_off;
  // end of the views: the panel's last entry and the one after it (the second
  // row of a pair; the storage goes on there)
  const double* panel_end = Ls + static_cast<int64_t>(f) * nc + 1;
  // a workgroup's part of the task's tile: 64 x 64 tiles a quarter of 128 x 128
  constexpr bool QUARTER = !U && TM == 64;
  const int z = static_cast<int>(blockIdx.z);
  const int zc = (QUARTER ? z & 1 : z) * TN, zr = QUARTER ? (z >> 1) * TM : 0;
  // this workgroup's rows and columns of the front (R0, C0), the first column
  // of the K range and K; M, N: valid rows and columns
  int R0, C0, ka, K, M, N;
  if (U) {
    R0 = nc + tr * TM;
    C0 = nc + tc * TN;
    ka = 0;
    K = nc;
    M = min(TM, f - R0);
    N = min(TN, f - C0);
  } else {
    ka = step * BT;
    K = min(mode >= 3 ? (mode - 1) * BT : BT, nc - ka);
    R0 = ka + K + tr * (QUARTER ? BT : TM) + zr;
    C0 = ka + K + tc * BT + zc;
    M = min(TM, f - R0);
    N = min(TN, nc - C0);
  }
  if (M <= 0 || N <= 0 || (QUARTER && R0 + M <= C0)) return;
  const int m16 = lane & 15, q4 = lane >> 4;
  const int wr = (wave / WN) * QM, wc = (wave % WN) * QN;
  const uint32_t f8 = static_cast<uint32_t>(f) * 8u;

  // fragments of K-step s: A(R0 + wr + row, ka + 4 s + q4), the same for B
  double fa[D][IM], fb[D][JN];
  const double* pa = Ls + static_cast<int64_t>(ka) * f + R0 + wr;
  const double* pb = Ls + static_cast<int64_t>(ka) * f + C0 + wc;
  const uint32_t va = q4 * f8 + grow16<IM>(0, m16) * 8u, vb = q4 * f8 + grow16<JN>(0, m16) * 8u;
  const int64_t dk = 4 * static_cast<int64_t>(f);
  auto load = [&](int d, bool in) {   // the next K-step into buffer d
    frag_load<IM>(fa[d], view(pa, 8 * (panel_end - pa)), in ? va : OFF_NONE);
    frag_load<JN>(fb[d], view(pb, 8 * (panel_end - pb)), in ? vb : OFF_NONE);
    pa += dk;
    pb += dk;
  };
#pragma unroll
  for (int d = 0; d < D; d++) load(d, 4 * d + q4 < K);

  // acc[i][j][v]: C row wr + grow16<IM>(i, m16), column wc + grow16<JN>(j, 4 v + q4)
  d4 acc[IM][JN];
  const double* Cp = Ls + static_cast<int64_t>(C0 + wc) * f + R0 + wr;
  const uint32_t vc = grow16<JN>(0, q4) * f8 + grow16<IM>(0, m16) * 8u;
  auto coff = [&](int j, int v) { return static_cast<uint32_t>(grow16<JN>(j, 4 * v)) * f8; };
  // (the test of mode keeps this a block of its own, which the compiler does not
  // interleave with its neighbours: their addresses beside the accumulators would
  // spill)
  if (!U && mode != 1) {
    const rsrc_t rc = view(Cp, 8 * (panel_end - Cp));
#pragma unroll
    for (int j = 0; j < JN; j++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        double t[IM];
        frag_load<IM>(t, rc, vc + coff(j, v));
#pragma unroll
        for (int i = 0; i < IM; i++) acc[i][j][v] = t[i];
      }
  } else {
#pragma unroll
    for (int i = 0; i < IM; i++)
#pragma unroll
      for (int j = 0; j < JN; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  }

  auto mm = [&](int d) {
#pragma unroll
    for (int i = 0; i < IM; i++)
#pragma unroll
      for (int j = 0; j < JN; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[d][j], -fa[d][i], acc[i][j], 0, 0, 0);
  };
  const int nk = (K + 3) / 4, kfull = K / 4;   // K-steps; those with all four columns
  int k = 0;
  for (; k + 2 * D <= kfull; k += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      mm(d);
      load(d, true);
    }
  }
  for (; k < nk; k += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      mm(d);
      if (k + D < nk) load(d, 4 * (k + D + d) + q4 < K);
    }
  }

  // the lane's place anew, so that no address of the stores is formed before the
  // loop and held in registers through it
  int lm = m16, lq = q4;
  asm volatile("" : "+v"(lm), "+v"(lq));
  if constexpr (U) {
    // U packed by columns, entries on or below its diagonal
    double* Us = batch_at(c.U, sy, bt) + sn.u_off;
    const int gr0 = R0 - nc + wr, gc0 = C0 - nc + wc;
    // the children's update matrices, in the order of the child list: an entry
    // (r, c) of the front takes child t's entry (inv(t, r), inv(t, c)) where it has
    // both; the index loads of CG children are in flight together
    const double* Ub = batch_at(c.U, sy, bt);
    const int rlim = nr - gr0, clim = nr - gc0;   // rows, columns of the wave's block
    for (int t0 = 0; t0 < sn.nch; t0 += CG) {
      const int cw = child_words<CG>(sn, t0, lane);
      int ia[CG][IM], ib[CG][JN][4];
#pragma unroll
      for (int g = 0; g < CG; g++) {
        const bool in = t0 + g < sn.nch;
        const int* iv = sn.inv + static_cast<int64_t>(min(t0 + g, sn.nch - 1)) * sn.stride + nc;
#pragma unroll
        for (int i = 0; i < IM; i++) {
          const int r = grow16<IM>(i, lm);
          const int x = iv[gr0 + min(r, max(rlim - 1, -gr0))];
          ia[g][i] = in && r < rlim ? x : -1;
        }
#pragma unroll
        for (int j = 0; j < JN; j++)
#pragma unroll
          for (int v = 0; v < 4; v++) {
            const int cl = grow16<JN>(j, 4 * v) + grow16<JN>(0, lq);
            const int x = iv[gc0 + min(cl, max(clim - 1, -gc0))];
            ib[g][j][v] = cl < clim ? x : 0x7fffffff;   // past every row
            if (ib[g][j][v] < 0) ib[g][j][v] = 0x7fffffff;
          }
      }
#pragma unroll
      for (int g = 0; g < CG; g++) {
        bool any = false;
#pragma unroll
        for (int i = 0; i < IM; i++) any = any || ia[g][i] >= 0;
        if (!__builtin_amdgcn_ballot_w64(any)) continue;
        const int n = rl32(cw, 4 * g + 2);
        const double* uc = Ub + rl64(cw, 4 * g);
#pragma unroll
        for (int j = 0; j < JN; j++)
#pragma unroll
          for (int v0 = 0; v0 < 4; v0 += VG) {
            double x[VG][IM];
#pragma unroll
            for (int v = 0; v < VG; v++) {
              int b = ib[g][j][v0 + v];
              // 128 x 128: a column's address is formed in its turn, and its sums before the
              // next one's loads; held beside the accumulators they spilled 31 registers
              if constexpr (CG == 1) asm volatile("" : "+v"(b));
              const double* col = uc + packed_lower(0, b < n ? b : 0, n);
              // on or below the child's diagonal; the others read the column's first
#pragma unroll
              for (int i = 0; i < IM; i++) x[v][i] = col[ia[g][i] >= b ? ia[g][i] : (b < n ? b : 0)];
            }
#pragma unroll
            for (int v = 0; v < VG; v++)
#pragma unroll
              for (int i = 0; i < IM; i++)
                acc[i][j][v0 + v] = ia[g][i] >= ib[g][j][v0 + v] ? acc[i][j][v0 + v] + x[v][i]
                                                                 : acc[i][j][v0 + v];
            if constexpr (CG == 1)
#pragma unroll
              for (int i = 0; i < IM; i++) asm volatile("" : "+v"(acc[i][j]) : : "memory");
          }
      }
    }
    const bool whole = M == TM && N == TN && gr0 >= gc0 + QN;   // no entry to leave out
#pragma unroll
    for (int j = 0; j < JN; j++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int cl = grow16<JN>(j, 4 * v) + grow16<JN>(0, lq), gc = gc0 + cl;
        double* col = Us + packed_lower(gr0, gc, nr);   // row gr0 of column gc
        if (whole) {
#pragma unroll
          for (int i = 0; i < IM; i++) col[grow16<IM>(i, lm)] = acc[i][j][v];
        } else {
#pragma unroll
          for (int i = 0; i < IM; i++) {
            const int r = grow16<IM>(i, lm);
            if (wr + r < M && wc + cl < N && gr0 + r >= gc) col[r] = acc[i][j][v];
          }
        }
      }
    return;
  }
  double* Cw = const_cast<double*>(Cp);
  const bool whole = M == TM && N == TN;
#pragma unroll
  for (int j = 0; j < JN; j++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int cl = grow16<JN>(j, 4 * v) + grow16<JN>(0, lq);
      double* col = Cw + static_cast<int64_t>(cl) * f;
      if (whole) {
        // pairs of rows: 16-byte stores (8-byte aligned, as the panel is)
        if constexpr (IM % 2 == 0) {
          typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
#pragma unroll
          for (int i = 0; i < IM; i += 2)
            *reinterpret_cast<d2u*>(col + grow16<IM>(i, lm)) = d2u{acc[i][j][v], acc[i + 1][j][v]};
        } else {
#pragma unroll
          for (int i = 0; i < IM; i++) col[grow16<IM>(i, lm)] = acc[i][j][v];
        }
      } else {
#pragma unroll
        for (int i = 0; i < IM; i++) {
          const int r = grow16<IM>(i, lm);
          if (wr + r < M && wc + cl < N) col[r] = acc[i][j][v];
        }
      }
    }
}

// TRSM below a diagonal block with its whole inverse (blocks of at most 64
// columns), in place: L21(block) = A21 * Dinv^T (K = block).  TM rows per
// tile (32 or 128).  The operands go through LDS (gemm_tile), so every read of
// a tile comes before its stores.  System blockIdx.y.
template <int TM>
__global__ void __launch_bounds__(256, 2) k_trsm_inv(CholDev c, const int* __restrict__ tsn,
                                                     const int* __restrict__ ttr, int step,
                                                     Batch bt)
{
  if constexpr (TM == 32) __builtin_amdgcn_s_setprio(3);   // see k_dense_nt
  extern __shared__ double smem[];
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  const SnInfo si = sninfo(c, batch_at(c.L, sy, bt), tsn[blockIdx.x]);
  const int k0 = step * BT;
  const int b = min(BT, si.nc - k0);
  const int R0 = k0 + b + ttr[blockIdx.x] * TM;
  double* panel = si.Ls + static_cast<int64_t>(k0) * si.f;   // columns k0..k0+b
  GemmArgs g;
  g.A = panel + R0;
  g.lda = si.f;
  g.B = batch_at(c.dinv, sy, bt) + c.dinv_off[tsn[blockIdx.x]] + inv_at(si.nc, step);
  g.ldb = inv_ld(si.nc, k0 / INV_GROUP);
  g.C = panel + R0;
  g.ldc = si.f;
  g.M = min(TM, si.f - R0);
  g.N = b;
  g.K = b;
  if (g.M <= 0 || g.N <= 0) return;
  gemm_tile<TM, BT>(g, smem);
}

// Factor the diagonal block of step `step` (b <= 128) in LDS, write L_kk back
// and the inverses of its 16 x 16 diagonal blocks, or its whole inverse (b <= 64),
// to dinv (lower part).  LDS holds one BK x (BK+1) array P, padded to BK with the
// identity: L(r, c) (r >= c) at P[r][c], the inverse X(i, j) (i > j) at
// P[j][i] and X(j, j) at P[j][BK]; and the reciprocals of L's diagonal.
//
// Cholesky, blocked by 16-column panels: one to three waves factor a panel in
// registers (see potrf_factor; 1/sqrt of the pivot is v_rsq_f64 refined by two Newton
// steps, so the chain carries no division or square root); the tile columns behind it
// are updated as FP64 MFMA 16x16x4 tiles.  Inverse: the 16x16 diagonal blocks are
// inverted together (16 lanes per block, lane j computes column j); for the whole one
// blocks of 16 and 32 are then doubled with
//   inv([L11 0; L21 L22]) = [X11 0; -X22 (L21 X11)  X22],
// both products on the matrix cores; L21 X11 is parked in the slot that
// -X22 (L21 X11) then overwrites.
//
// MFMA f64 16x16x4 (lane l of 64): A operand A(l%16, l/16), B operand
// B(l/16, l%16), result element v = D(4v + l/16, l%16) of D = A B.
constexpr int PW = 16;   // panel width

// Lane `lane`'s value of v, as a wave-uniform (scalar register) value.
__device__ __forceinline__ double readlane_f64(double v, int lane)
{
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(u), lane);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(u >> 32), lane);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}

// One 16x16 tile of D = A B accumulated over K (a multiple of 4): a_at(i, k)
// and b_at(k, j) give the operands.
template <int K, class FA, class FB>
__device__ __forceinline__ d4 mfma16(int lane, FA a_at, FB b_at)
{
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  const int i = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int k0 = 0; k0 < K; k0 += 4)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a_at(i, k0 + kq), b_at(k0 + kq, i), acc, 0, 0, 0);
  return acc;
}

// X(i, j) of the inverse from its storage in P (0 above the diagonal).
template <int BK>
__device__ __forceinline__ double xinv(const double (*P)[BK + 1], int i, int j)
{
  return (i > j) ? P[j][i] : ((i == j) ? P[j][BK] : 0.0);
}

// One doubling level: for every pair of inverted diagonal blocks of size H,
// X21 = -X22 (L21 X11), in 16 x 16 tiles (HB = H/16 per side).  The pair's
// HB waves take HB tiles each: in T = L21 X11 wave wp takes tile columns
// cb = u (u < HB) in rows (wp + u) % HB; in -X22 T, tile rows rb = u in
// columns (wp + u) % HB.  As X11 and X22 are lower triangular, a tile takes
// the k-blocks kk >= cb (resp. kk <= rb) only, so every wave does the same
// HB (HB + 1) / 2 block products.  All of a wave's operands are read from
// LDS before its MFMA chains run, interleaved.
template <int BK, int H>
__device__ __forceinline__ void inverse_level(double (*P)[BK + 1], int wave, int lane)
{
  constexpr int HB = H / 16, NPR = BK / (2 * H), WPP = 4 / NPR;   // waves per pair
  const int pair = wave / WPP, wp = wave % WPP;
  const bool act = wp < HB;
  const int b1 = 2 * H * pair;
  const int i = lane & 15, kq = lane >> 4;
  d4 acc[HB];
  double fa[HB][HB][4], fb[HB][HB][4];
  // T = L21 X11, stored where X21 goes (T(r, c) at P[c][r])
  if (act) {
#pragma unroll
    for (int u = 0; u < HB; u++) {
      const int r0 = b1 + H + 16 * ((wp + u) % HB), c0 = b1 + 16 * u;
#pragma unroll
      for (int kk = u; kk < HB; kk++)
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const int k = b1 + 16 * kk + 4 * m + kq;
          fa[u][kk][m] = P[r0 + i][k];
          fb[u][kk][m] = (kk == u) ? xinv<BK>(P, k, c0 + i) : P[c0 + i][k];
        }
    }
#pragma unroll
    for (int u = 0; u < HB; u++) acc[u] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < HB; kk++)
#pragma unroll
      for (int m = 0; m < 4; m++)
#pragma unroll
        for (int u = 0; u <= kk; u++)
          acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[u][kk][m], fb[u][kk][m], acc[u], 0, 0, 0);
#pragma unroll
    for (int u = 0; u < HB; u++) {
      const int r0 = b1 + H + 16 * ((wp + u) % HB), c0 = b1 + 16 * u;
#pragma unroll
      for (int v = 0; v < 4; v++) P[c0 + i][r0 + 4 * v + kq] = acc[u][v];
    }
  }
  __syncthreads();
  // X21 = -X22 T; every read of T before the in-place writes
  if (act) {
#pragma unroll
    for (int u = 0; u < HB; u++) {
      const int r0 = b1 + H + 16 * u, c0 = b1 + 16 * ((wp + u) % HB);
#pragma unroll
      for (int kk = 0; kk <= u; kk++)
#pragma unroll
        for (int m = 0; m < 4; m++) {
          const int k = b1 + H + 16 * kk + 4 * m + kq;
          fa[u][kk][m] = (kk == u) ? xinv<BK>(P, r0 + i, k) : P[k][r0 + i];
          fb[u][kk][m] = P[c0 + i][k];
        }
    }
#pragma unroll
    for (int u = 0; u < HB; u++) acc[u] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < HB; kk++)
#pragma unroll
      for (int m = 0; m < 4; m++)
#pragma unroll
        for (int u = kk; u < HB; u++)
          acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[u][kk][m], fb[u][kk][m], acc[u], 0, 0, 0);
  }
  __syncthreads();
  if (act) {
#pragma unroll
    for (int u = 0; u < HB; u++) {
      const int r0 = b1 + H + 16 * u, c0 = b1 + 16 * ((wp + u) % HB);
#pragma unroll
      for (int v = 0; v < 4; v++) P[c0 + i][r0 + 4 * v + kq] = -acc[u][v];
    }
  }
  __syncthreads();
}

// Entry e < BK (BK + 1) / 2 of the lower triangle of a BK x BK block (BK
// even), columns folded in pairs c, BK-1-c (together BK + 1 entries), so
// consecutive e run down one column.
template <int BK>
__device__ __forceinline__ void lower_entry(int e, int& r, int& col)
{
  const int pr = e / (BK + 1), o = e - pr * (BK + 1);
  const bool first = o < BK - pr;
  col = first ? pr : BK - 1 - pr;
  r = first ? pr + o : col + o - (BK - pr);
}

// The doubling levels and the store of the whole inverse, from P holding L
// in its lower part and the inverses of the 16x16 diagonal blocks (see
// potrf_block), into the dinv slot at W (column-major, ldw; entries outside
// the b x b lower triangle stay at the zeros written when the slot was
// created).  All threads of the workgroup.
template <int BK>
__device__ __forceinline__ void inverse_full(double (*P)[BK + 1], double* W, int ldw, int b,
                                             int tid, int wave, int lane)
{
  constexpr int NL = BK * (BK + 1) / 2, PER = (NL + 255) / 256;
  if constexpr (BK >= 32) inverse_level<BK, 16>(P, wave, lane);
  if constexpr (BK >= 64) inverse_level<BK, 32>(P, wave, lane);
  // over the folded lower triangle, LDS reads first so they overlap
  constexpr int SB2 = (PER + 1) / 2;   // entries per batch
#pragma unroll
  for (int u0 = 0; u0 < PER; u0 += SB2) {
    double xv[SB2];
#pragma unroll
    for (int u = 0; u < SB2; u++) {
      int r, col;
      lower_entry<BK>(min(tid + (u0 + u) * 256, NL - 1), r, col);
      xv[u] = xinv<BK>(P, r, col);
    }
#pragma unroll
    for (int u = 0; u < SB2; u++) {
      int r, col;
      const int e = tid + (u0 + u) * 256;
      lower_entry<BK>(min(e, NL - 1), r, col);
      if (u0 + u < PER && e < NL && r < b) W[static_cast<int64_t>(col) * ldw + r] = xv[u];
    }
  }
}

// P[r][c] -= sum_k P[r][k] P[c][k] over the np 16-column panels from column
// kb0 on, for the 16 x 16 tiles e < nt whose top-left corners tile(e, r0, c0)
// gives, tile e to wave w0 + e % nw (the calling waves are w0 .. w0+nw-1),
// two tiles at a time: each panel's operand reads first, the two MFMA
// chains interleaved.  Whole tiles: the upper half of a diagonal tile is
// scratch until the inverse is written.
template <int BK, class TILE>
__device__ __forceinline__ void panel_tiles(double (*P)[BK + 1], int kb0, int np, int nt, int w0,
                                            int nw, int wave, int lane, TILE tile)
{
  const int i = lane & 15, kq = lane >> 4;
  for (int e = wave - w0; e < nt; e += 2 * nw) {
    int r0[2], c0[2];
    const bool two = e + nw < nt;
    tile(e, r0[0], c0[0]);
    tile(two ? e + nw : e, r0[1], c0[1]);
    d4 acc[2];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int v = 0; v < 4; v++) acc[h][v] = P[r0[h] + 4 * v + kq][c0[h] + i];
    for (int q = 0; q < np; q++) {
      const int kb = kb0 + PW * q;
      double fa[2][4], fb[2][4];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          fa[h][k] = -P[r0[h] + i][kb + 4 * k + kq];
          fb[h][k] = P[c0[h] + i][kb + 4 * k + kq];
        }
      // C(r, c) -= sum_k A(r, k) B(c, k): result element v is row 4v + lane/16
      // of the tile, column lane % 16
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int h = 0; h < 2; h++)
          acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[h][k], fb[h][k], acc[h], 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) P[r0[0] + 4 * v + kq][c0[0] + i] = acc[0][v];
    if (two) {
#pragma unroll
      for (int v = 0; v < 4; v++) P[r0[1] + 4 * v + kq][c0[1] + i] = acc[1][v];
    }
  }
}

// The Cholesky factor of the BK x BK block in P's lower part (b columns of the
// matrix, col0 the first, then the identity), in place; rd: the reciprocals of its
// diagonal; *bad (shared, INT_MAX before): the first column whose pivot fails.
// All threads of the workgroup, past a barrier at the end.
template <int BK>
__device__ __forceinline__ void potrf_factor(double (*P)[BK + 1], double* rd, int b, int col0,
                                             double pivot_tol, int* bad, int tid, int lane,
                                             int wave, int panels = BK / PW)
{
  // ---- blocked Cholesky, one 16-column panel at a time ----
  // Each factoring wave takes the panel's 16 x 16 diagonal block in lanes
  // 0..15 (lane l holds row kb + l; every such wave the same) and 48 of the
  // rows below in lanes 16..63, so the whole panel is factored in one pass:
  // at step k the pivot row's entries reach every lane of the wave through
  // v_readlane (read before the pivot's 1/sqrt is known, scaled after),
  // column k is scaled and the later columns take its rank-1 update.  Entries
  // above the diagonal of the 16 x 16 block are carried along, never stored,
  // so no lane-dependent branches.  Only as many waves factor as the panel's
  // rows need (three for the first panel, then two, then one); the others
  // meanwhile bring the next tile column up to date with all earlier panels
  // (left-looking, so this work stays small and even), and after the panel
  // all waves apply the panel itself to that column.
  {
    const bool dg = lane < PW;
    const int prow_off = dg ? lane : PW + 48 * wave + (lane - PW);   // row - kb
#pragma unroll 1
    for (int p = 0; p < panels; p++) {
      const int kb = p * PW;
      const int nf = max(1, (BK - kb - PW + 47) / 48);   // factoring waves
      double v[PW];
      const int r = kb + prow_off;
      if (wave < nf) {
        const int rr = min(r, BK - 1);
#pragma unroll
        for (int q = 0; q < PW; q++) v[q] = P[rr][kb + q];
      }
      // every factoring wave has read the diagonal block before wave 0 stores its factor
      // there: a wave may lag the others by more than a pass where work of other
      // streams shares its SIMD
      if (nf > 1) __syncthreads();
      if (wave < nf) {
        const bool mine = r < BK && (dg ? wave == 0 : true);   // this lane stores row r
        double myinv = 1.0;   // 1 / L(kb + lane, kb + lane), taken at step k == lane
#pragma unroll
        for (int k = 0; k < PW; k++) {
          const double dkk = readlane_f64(v[k], k);
          double lu[PW];   // unscaled entries (kb+q, kb+k) of rows q > k
#pragma unroll
          for (int q = k + 1; q < PW; q++) lu[q] = readlane_f64(v[k], q);
          // 1/sqrt(dkk), v_rsq_f64 and two Newton steps; the pivot test
          // comes after the panel, off the column-to-column chain
          double y = __builtin_amdgcn_rsq(dkk);
          const double hx = 0.5 * dkk;
          y = y * fma(-hx, y * y, 1.5);
          y = y * fma(-hx, y * y, 1.5);
          // L(r, kb+k) = v_k y; the update L(r, kb+k) L(kb+q, kb+k) is v_k y^2 lu_q
          const double wk = v[k] * (y * y);
          v[k] = (lane == k) ? dkk * y : v[k] * y;
          myinv = (lane == k) ? y : myinv;
          // formed here, so the step's masks end with the step (the compiler
          // would otherwise defer these selects to the stores, holding every
          // step's masks in scalar registers)
          asm volatile("" : "+v"(v[k]), "+v"(myinv));
#pragma unroll
          for (int q = k + 1; q < PW; q++) v[q] -= wk * lu[q];
        }
        // whole rows, also the diagonal block's carried entries above the
        // diagonal: that half of a diagonal tile is scratch until the inverse
        // is written there (one store mask, no per-entry branches)
        if (mine) {
#pragma unroll
          for (int q = 0; q < PW; q++) P[r][kb + q] = v[q];
        }
        if (wave == 0) {
          // the pivot test, sqrt(pivot) > pivot_tol, on L(kb+l, kb+l) as lane l
          // just stored it: a failed pivot leaves a small value or NaN there
          // (NaN then runs through the rest of this system's factor; the
          // system is reported and kept out of the solve).  The first
          // failing column of the first failing panel is kept.
          const double lkk = P[kb + (lane & 15)][kb + (lane & 15)];
          const uint64_t f = __builtin_amdgcn_ballot_w64(dg && kb + lane < b && !(lkk > pivot_tol));
          if (f != 0 && tid == 0 && *bad == INT_MAX) *bad = col0 + kb + __builtin_ctzll(f);
          if (dg) rd[kb + lane] = myinv;
        }
      } else if (p > 0 && p + 1 < panels) {
        // the next tile column (its tiles from the diagonal down) by the
        // panels before this one
        const int cb = kb + PW;
        panel_tiles<BK>(P, 0, p, (BK - cb) / PW, nf, 4 - nf, wave, lane,
                        [&](int e, int& r0, int& c0) {
                          r0 = cb + PW * e;
                          c0 = cb;
                        });
      }
      __syncthreads();
      if (p + 1 < panels) {
        // and by this panel
        const int cb = kb + PW;
        panel_tiles<BK>(P, kb, 1, (BK - cb) / PW, 0, 4, wave, lane, [&](int e, int& r0, int& c0) {
          r0 = cb + PW * e;
          c0 = cb;
        });
        __syncthreads();
      }
    }
  }
}

// The inverses of the 16x16 diagonal blocks of the factor in P (16 lanes each),
// stored above the diagonal and in column BK.  All threads, past a barrier.
template <int BK>
__device__ __forceinline__ void invert16(double (*P)[BK + 1], const double* rd, int tid)
{
  if (tid < BK) {
    const int bb = (tid / PW) * PW, j = tid % PW;
    double x[PW];
#pragma unroll
    for (int i = 0; i < PW; i++) {
      double t0 = (i == j) ? 1.0 : 0.0, t1 = 0.0;
#pragma unroll
      for (int k = 0; k < i; k++) {
        if (k & 1) t1 -= P[bb + i][bb + k] * x[k];
        else t0 -= P[bb + i][bb + k] * x[k];
      }
      x[i] = (i >= j) ? (t0 + t1) * rd[bb + i] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < PW; i++) {
      if (i == j) P[bb + j][BK] = x[i];
      else if (i > j) P[bb + j][bb + i] = x[i];
    }
  }
  __syncthreads();
}

// Diagonal block `step` of supernode s, by one workgroup of 256 threads with
// smem >= potrf_smem<BK>().  BK: padded block edge (32, 64 or 128) >= b.
// FULL: the whole inverse; otherwise only the inverses of its 16x16 diagonal
// blocks (the blocked TRSM's); k_inv_group forms the rest.
template <int BK, bool FULL>
__device__ __forceinline__ void potrf_block(const CholDev& c, double* L, double* dinv, int* pivot,
                                            int s, int step, double* smem)
{
  const SnInfo si = sninfo(c, L, s);
  const int k0 = step * BT;
  if (k0 >= si.nc) return;
  const int b = min(BK, si.nc - k0);
  double (*P)[BK + 1] = reinterpret_cast<double (*)[BK + 1]>(smem);
  double* rd = smem + BK * (BK + 1);   // 1 / L(r, r)
  __shared__ int bad;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar tile bookkeeping
  double* D = si.Ls + static_cast<int64_t>(k0) * si.f + k0;
  // load the lower triangle (padded with the identity past b), all of a
  // thread's entries in flight at once.  Every lane loads (entries past b or
  // past the triangle read D[0] and are replaced), so the loads are not split
  // by branches that would wait on each other.
  constexpr int NL = BK * (BK + 1) / 2, PER = (NL + 255) / 256;
  {
    double v[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
      int r, col;
      lower_entry<BK>(min(tid + u * 256, NL - 1), r, col);
      const bool in = r < b;
      const double t = D[in ? r + static_cast<int64_t>(col) * si.f : 0];
      v[u] = in ? t : (r == col ? 1.0 : 0.0);
    }
#pragma unroll
    for (int u = 0; u < PER; u++) {
      int r, col;
      lower_entry<BK>(min(tid + u * 256, NL - 1), r, col);
      if (tid + u * 256 < NL) P[r][col] = v[u];
    }
  }
  if (tid == 0) bad = INT_MAX;
  __syncthreads();

  potrf_factor<BK>(P, rd, b, si.a + k0, c.pivot_tol, &bad, tid, lane, wave);

  // L_kk back to the factor (the inverse below keeps P's lower part), the
  // stores draining while the inverse is formed
#pragma unroll
  for (int u = 0; u < PER; u++) {
    int r, col;
    const int e = tid + u * 256;
    lower_entry<BK>(min(e, NL - 1), r, col);
    const double lv = P[r][col];
    if (e < NL && r < b) D[r + static_cast<int64_t>(col) * si.f] = lv;
  }

  invert16<BK>(P, rd, tid);
  double* W = dinv + c.dinv_off[s] + inv_at(si.nc, step);
  const int ldw = inv_ld(si.nc, k0 / INV_GROUP);
  if constexpr (FULL) {
    inverse_full<BK>(P, W, ldw, b, tid, wave, lane);
  } else {
    // the 16x16 diagonal blocks of the inverse, at their places in the slot
    constexpr int NE = (BK / PW) * (PW * (PW + 1) / 2);
    for (int e = tid; e < NE; e += 256) {
      const int bb = (e / (PW * (PW + 1) / 2)) * PW;
      int r, col;
      lower_entry<PW>(e % (PW * (PW + 1) / 2), r, col);
      if (bb + r < b) W[static_cast<int64_t>(bb + col) * ldw + bb + r] = xinv<BK>(P, bb + r, bb + col);
    }
  }
  if (tid == 0 && bad != INT_MAX) atomicMin(pivot, bad);
}

template <int BK>
__global__ void __launch_bounds__(256) k_potrf_inv(CholDev c, const int* __restrict__ sns,
                                                   int step, Batch bt)
{
  __builtin_amdgcn_s_setprio(3);   // the critical chain: issue priority (see k_dense_nt)
  extern __shared__ double smem[];
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  const int s = sns[blockIdx.x];
  if (step * BT >= c.sn_first[s + 1] - c.sn_first[s]) return;
  potrf_block<BK, (BK < 128)>(c, batch_at(c.L, sy, bt), batch_at(c.dinv, sy, bt), c.pivot + sy,
                              s, step, smem);
}

// The panel of supernodes with at most 32 columns, from the assembled entries to
// the factor: the children's contributions, the diagonal block's factor and
// inverse, and L21 = A21 Dinv^T for one tile of 128 rows per task.  Every tile forms
// the diagonal block itself, and the first one writes its inverse; the block in the
// panel stays as assembled, as other tiles may still have to read it: the sweeps
// use the inverse alone.  In place of an extend-add, a diagonal-block and a TRSM
// launch per tree level: these levels are bound by launches and latency, 13-25 us
// each in one launch against 27-45 in three (1,000 buses).  Children's entries are
// added in the order of the child list, with two children's loads in flight.
// System blockIdx.y.
constexpr int FP = 32;
static_assert(FP == FRONT_NC, "a narrow panel's slot is FP x FP");

__global__ void __launch_bounds__(256) k_front_panel(CholDev c, const int* __restrict__ tsn,
                                                     const int* __restrict__ ttr, Batch bt)
{
  __builtin_amdgcn_s_setprio(3);   // the critical chain: issue priority (see k_dense_nt)
  __shared__ double Ps[FP * (FP + 1) + FP];
  __shared__ double As[FP][BT + 2];   // the tile's rows of A21, column-major
  __shared__ int bad;
  double (*P)[FP + 1] = reinterpret_cast<double (*)[FP + 1]>(Ps);
  double* rd = Ps + FP * (FP + 1);
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int s = uni(tsn[blockIdx.x]), tile = uni(ttr[blockIdx.x]);
  const Sn sn = load_sn(c, s, lane);
  const int a0 = sn.a, nc = sn.nc, f = sn.f;
  double* Ls = batch_at(c.L, sy, bt) + sn.l_off;
  const double* Ub = batch_at(c.U, sy, bt);
  constexpr int NL = FP * (FP + 1) / 2, PER = (NL + 255) / 256;
  constexpr int CPT = FP / 2, KB = 4;   // columns of a thread's row of the tile, per step
  // thread: front row R, columns h, h + 2, .. of the tile; entries of the triangle
  const int R = nc + tile * BT + (tid & (BT - 1)), h = uni(tid >> 7);
  const bool live = R < f;
  double va[CPT], vd[PER];
#pragma unroll
  for (int k = 0; k < CPT; k++) {
    const int col = h + 2 * k;
    va[k] = (live && col < nc) ? Ls[static_cast<int64_t>(col) * f + R] : 0.0;
  }
  int dr[PER], dc[PER];
#pragma unroll
  for (int u = 0; u < PER; u++) {
    lower_entry<FP>(min(tid + u * 256, NL - 1), dr[u], dc[u]);
    vd[u] = dr[u] < nc ? Ls[static_cast<int64_t>(dc[u]) * f + dr[u]] : (dr[u] == dc[u] ? 1.0 : 0.0);
  }
  // G children from t0 on, their loads in flight together
  auto add_children = [&](auto count, int t0) {
    constexpr int G = decltype(count)::value;
    const int cw = child_words<G>(sn, t0, lane);
    // their rows at this thread's front row, at the panel's columns (lane: column)
    // and at its entries of the triangle
    int ir[G], ic[G], dra[G][PER], dca[G][PER];
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int* iv = sn.inv + static_cast<int64_t>(t0 + g) * sn.stride;
      ir[g] = iv[live ? R : 0];
      ic[g] = iv[min(lane, nc - 1)];
#pragma unroll
      for (int u = 0; u < PER; u++) {
        dra[g][u] = iv[min(dr[u], nc - 1)];
        dca[g][u] = iv[min(dc[u], nc - 1)];
      }
    }
    double xd[G][PER], xa[G][CPT];
#pragma unroll
    for (int g = 0; g < G; g++) {
      const int n = rl32(cw, 4 * g + 2);
      const double* uc = Ub + rl64(cw, 4 * g);
      if (!live) ir[g] = -1;
      // lane l: where the child's column for front column l starts
      const int64_t cb = packed_lower(0, max(ic[g], 0), n);
      const int clo = static_cast<int>(cb), chi = static_cast<int>(cb >> 32);
#pragma unroll
      for (int u = 0; u < PER; u++) {
        if (dr[u] >= nc) dra[g][u] = -1;
        const bool ok = dra[g][u] >= 0 && dca[g][u] >= 0;
        xd[g][u] = uc[ok ? packed_lower(dra[g][u], dca[g][u], n) : 0];
      }
#pragma unroll
      for (int k0 = 0; k0 < CPT; k0 += KB) {
        if (h + 2 * k0 >= nc) break;   // uniform
#pragma unroll
        for (int k = k0; k < k0 + KB; k++) {   // past nc: a repeat, not added
          const int l = h + 2 * k;
          const int64_t at = static_cast<int64_t>(
              (static_cast<uint64_t>(static_cast<uint32_t>(rl32(chi, l))) << 32) |
              static_cast<uint32_t>(rl32(clo, l)));
          xa[g][k] = uc[at + max(ir[g], max(rl32(ic[g], l), 0))];
        }
      }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
#pragma unroll
      for (int u = 0; u < PER; u++)
        vd[u] = (dra[g][u] >= 0 && dca[g][u] >= 0) ? vd[u] + xd[g][u] : vd[u];
#pragma unroll
      for (int k0 = 0; k0 < CPT; k0 += KB) {
        if (h + 2 * k0 >= nc) break;
#pragma unroll
        for (int k = k0; k < k0 + KB; k++) {
          const bool has = h + 2 * k < nc && rl32(ic[g], h + 2 * k) >= 0;
          va[k] = has && ir[g] >= 0 ? va[k] + xa[g][k] : va[k];
        }
      }
    }
  };
  int t0 = 0;
  for (; t0 + 2 <= sn.nch; t0 += 2) add_children(std::integral_constant<int, 2>{}, t0);
  if (t0 < sn.nch) add_children(std::integral_constant<int, 1>{}, t0);
#pragma unroll
  for (int u = 0; u < PER; u++)
    if (tid + u * 256 < NL) P[dr[u]][dc[u]] = vd[u];
#pragma unroll
  for (int k = 0; k < CPT; k++) As[h + 2 * k][tid & (BT - 1)] = va[k];
  if (tid == 0) bad = INT_MAX;
  __syncthreads();
  // at most 16 columns: the second panel is the identity, and stays out of all below
  const int panels = nc <= PW ? 1 : 2;
  potrf_factor<FP>(P, rd, nc, a0, c.pivot_tol, &bad, tid, lane, wave, panels);
  if (panels == 1 && tid < PW) rd[PW + tid] = 1.0;
  if (panels == 1) __syncthreads();
  invert16<FP>(P, rd, tid);
  if (panels == 2) inverse_level<FP, 16>(P, wave, lane);
  if (tile == 0) {
    double* W = batch_at(c.dinv, sy, bt) + sn.dinv_off;
#pragma unroll
    for (int u = 0; u < PER; u++)
      if (tid + u * 256 < NL && dr[u] < nc)
        W[static_cast<int64_t>(dc[u]) * FP + dr[u]] = xinv<FP>(P, dr[u], dc[u]);
    if (tid == 0 && bad != INT_MAX) atomicMin(c.pivot + sy, bad);
  }
  // L21: wave w takes rows 32 w .. 32 w + 31 of the tile, in two by two MFMA tiles
  const int rows = f - (nc + tile * BT), r0 = 32 * wave;
  if (r0 >= rows) return;   // no barrier follows
  const int m16 = lane & 15, q4 = lane >> 4;
  d4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k0 = 0; k0 < FP; k0 += 4) {
    if (k0 >= nc) break;
    double fa[2], fb[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      fa[i] = As[k0 + q4][r0 + 16 * i + m16];
      fb[i] = xinv<FP>(P, 16 * i + m16, k0 + q4);
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[j], fa[i], acc[i][j], 0, 0, 0);
  }
  double* C = Ls + nc + tile * BT + r0;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int row = 16 * i + m16, col = 16 * j + 4 * v + q4;
        if (r0 + row < rows && col < nc) C[static_cast<int64_t>(col) * f + row] = acc[i][j][v];
      }
}

// The inverses of groups of up to four 128-column diagonal blocks, from the factor and
// the inverses of its 16 x 16 diagonal blocks (which the factorization left): a
// workgroup per strip of 16 columns solves L X = E, 128 rows at a time, wave w rows
// 16 w .. 16 w + 15 of them. First all the blocks before, in one product (operands read
// straight into MFMA fragments, X from LDS); then the block's eight panels by
// substitution, each wave's sums staying in its accumulators, whose lane layout
// (element v = D[4 v + l/16][l%16]) is the B operand's of k-step v.
// By substitution, and not with products of the 128-wide blocks' own inverses (doubled
// from the 16 x 16 ones), which lose the square of a block's condition number: backward
// error of a solve with a Gaussian kernel matrix (condition 1e11) of 512 / 1,024: 2.6e-13
// / 1.7e-13, with products 2.3e-10 / 9.5e-12, sweeps through 128-wide inverses 1.5e-11 /
// 3.6e-14. On the grids' H_gamma, gamma 1e4 to 1e6 and Ds spread 1e-2..1e2 to 1e-4..1e8,
// backward and forward errors are those of 128-wide inverses; on dense matrices of random
// eigenvectors up to 7 times theirs, and below the unit roundoff.
// With them a sweep passes a group of up to 512 columns in one product in place of a
// chain of four. Bound by the first strip's chain: 36 us a factorization at 1,000 buses,
// 125 at 20,000, 217 at eight systems of 5,000 (products: 48, 128, 209 in two launches).
// Loads four K-steps ahead: with 8 and 16 the kernel spills (217 and 275 us, eight of
// 5,000). Task: supernode, 32 group + strip; system blockIdx.y.
constexpr int IG_LD = PW + 1;   // row of the strip in LDS
constexpr size_t IG_SMEM = INV_GROUP * IG_LD * sizeof(double);   // two workgroups per CU

__global__ void __launch_bounds__(512, 4) k_inv_group(CholDev c, const int* __restrict__ tsn,
                                                   const int* __restrict__ tix, Batch bt)
{
  extern __shared__ double smem[];
  double (*Xs)[IG_LD] = reinterpret_cast<double (*)[IG_LD]>(smem);
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  constexpr int NP = BT / PW;   // panels of a block, a wave each
  const int lane = threadIdx.x & 63, w = uni(threadIdx.x >> 6);
  const int m16 = lane & 15, q4 = lane >> 4;
  const int s = uni(tsn[blockIdx.x]), ix = uni(tix[blockIdx.x]), g = ix >> 5, cs = (ix & 31) * PW;
  const SnInfo si = sninfo(c, batch_at(c.L, sy, bt), s);
  const int nc = uni(si.nc), f = uni(si.f);
  const int g0 = g * INV_GROUP, ng = min(INV_GROUP, nc - g0), nb = (ng + BT - 1) / BT;
  const int jb = cs / BT, pj = (cs - BT * jb) / PW;   // the strip's block and panel
  const int ld = inv_ld(nc, g);
  const uint32_t f8 = static_cast<uint32_t>(f) * 8u;
  double* W = batch_at(c.dinv, sy, bt) + uni64(c.dinv_off[s]) +
              static_cast<int64_t>(g) * INV_GROUP * INV_GROUP;
  const double* Lg = batch_at(c.L, sy, bt) + uni64(c.l_off[s]) + static_cast<int64_t>(g0) * f;
  auto load = [](rsrc_t v, uint32_t vo, uint32_t so) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(v, vo, so, 0));
  };
  constexpr int D = 4;   // K-steps of the product whose loads are in flight
  for (int ib = jb; ib < nb; ib++) {
    // this lane's row of the factor (past the supernode's columns the last one: its X is
    // 0, as the inverses past them hold zeros), its columns in this block
    const int row = BT * ib + PW * w, cols = min(BT, nc - g0 - BT * ib);
    const uint32_t vr = static_cast<uint32_t>(min(g0 + row + m16, nc - 1)) * 8u;
    const int p0 = ib == jb ? pj : 0;   // rows above are 0
    // L(row, 16 q + 4 v + q4) of the block, q < w, and inv16 of the wave's own panel
    // (a quadruple of columns that ends past the block's is another one: rows that
    // would use it are past the supernode's columns)
    double lw[NP - 1][4], iw[4];
    {
      const rsrc_t rl = view(Lg + static_cast<int64_t>(BT * ib) * f, static_cast<int64_t>(cols) * f8);
      const uint32_t vo = vr + static_cast<uint32_t>(min(q4, cols - 1)) * f8;
#pragma unroll
      for (int q = 0; q < NP - 1; q++)
#pragma unroll
        for (int v = 0; v < 4; v++)
          lw[q][v] = q >= p0 && q < w
                         ? load(rl, vo, static_cast<uint32_t>(min(PW * q + 4 * v, max(cols - 4, 0))) * f8)
                         : 0.0;
#pragma unroll
      for (int v = 0; v < 4; v++) iw[v] = W[static_cast<int64_t>(row + 4 * v + q4) * ld + row + m16];
    }
    // E - L X over the blocks before: element v is row 4 v + q4, column m16
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    if (ib == jb) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        acc[v] = w == pj && 4 * v + q4 == m16 ? 1.0 : 0.0;
        if (w < pj) Xs[row + 4 * v + q4][m16] = 0.0;
      }
    } else {
      const int K = BT * (ib - jb);
      const rsrc_t ra = view(Lg + static_cast<int64_t>(BT * jb) * f, static_cast<int64_t>(K) * f8);
      const double (*X)[IG_LD] = Xs + BT * jb;
      const uint32_t vo = vr + static_cast<uint32_t>(q4) * f8;
      auto at = [&](int k) { return load(ra, vo, static_cast<uint32_t>(min(k, K - 4)) * f8); };
      double a[D];
#pragma unroll
      for (int u = 0; u < D; u++) a[u] = at(4 * u);
      for (int k0 = 0; k0 < K; k0 += 4 * D) {
#pragma unroll
        for (int u = 0; u < D; u++) {
          const int k = k0 + 4 * u;
          const double v = -a[u];
          a[u] = at(k + 4 * D);
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v, X[k + q4][m16], acc, 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int p = 0; p < NP; p++) {
      if (p < p0) continue;
      if (w == p) {
        d4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int v = 0; v < 4; v++)
          x = __builtin_amdgcn_mfma_f64_16x16x4f64(iw[v], acc[v], x, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const int r = row + 4 * v + q4;
          Xs[r][m16] = x[v];
          if (r < ng && r >= cs + PW) W[static_cast<int64_t>(cs + m16) * ld + r] = x[v];
        }
      }
      __syncthreads();
      if (p + 1 < NP && w > p) {
#pragma unroll
        for (int v = 0; v < 4; v++)
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-lw[p < NP - 1 ? p : 0][v],
                                                     Xs[BT * ib + PW * p + 4 * v + q4][m16], acc, 0, 0, 0);
      }
    }
  }
}

// L21 = A21 L_kk^{-T} for the rows below 128-wide diagonal block `step`, by
// blocked forward substitution over its eight 16-column panels (no inverse of
// the whole block needed): X_p^T = inv16(L_pp) (A_p^T - sum_{q<p} L_pq X_q^T).
// A wave owns 16-row groups; a group's X_q^T live in MFMA accumulators, whose
// lane layout (element v = D[4v + l/16][l%16]) is the B operand's of k-step
// v, so they feed the later panels' products without going through LDS.  The
// 28 blocks L_pq (p > q) and the 8 inverses inv16(L_pp) are staged in LDS first (each
// 16 x 16, column-major), and A is loaded panels ahead of its use: beside a trailing
// update a load takes several times its time alone.  Few registers: a 64-row tile
// fits beside two workgroups of the trailing update on one CU, so the critical path's
// TRSM does not wait for them to drain.  TM rows per tile (64 or 128: 4 or 8 groups);
// every row takes the same operations in the same order whatever the tile, so both
// shapes give the same bits.  One 4,284-column supernode (5,000 buses), mean of its
// steps beside the trailing updates: 32-row tiles with one panel ahead 19.2 us, now
// 15.7.  In place.  System blockIdx.y.
constexpr int TRSM_NB = (BT / PW) * (BT / PW - 1) / 2;   // blocks L_pq, p > q
constexpr size_t TRSM_SMEM = (TRSM_NB + BT / PW) * PW * PW * sizeof(double);

template <int TM>
__global__ void __launch_bounds__(256, TM == 64 ? 4 : 1)
    k_trsm(CholDev c, const int* __restrict__ tsn, const int* __restrict__ ttr, int step, Batch bt)
{
  __builtin_amdgcn_s_setprio(3);   // the critical chain: issue priority (see k_dense_nt)
  constexpr int NG = TM / 16, NGW = (NG + 3) / 4;   // groups, groups per wave
  constexpr int NPN = BT / PW;                       // panels
  extern __shared__ double smem[];
  double* Ls = smem;                                 // block (p, q) at (p(p-1)/2 + q) * 256
  double* Is = smem + TRSM_NB * PW * PW;             // inv16(L_pp) at p * 256
  const int sy = batch_sys(bt);
  if (sy < 0) return;
  const int s = tsn[blockIdx.x], tr = ttr[blockIdx.x];
  const SnInfo si = sninfo(c, batch_at(c.L, sy, bt), s);
  const int k0 = step * BT;
  const int b = min(BT, si.nc - k0);
  const int R0 = k0 + b + tr * TM;
  const int M = min(TM, si.f - R0);
  if (b <= 0 || M <= 0) return;   // uniform over the workgroup
  const int64_t f = si.f;
  const double* Lkk = si.Ls + static_cast<int64_t>(k0) * f + k0;   // L(k0 + r, k0 + c) at c*f + r
  double* A = si.Ls + static_cast<int64_t>(k0) * f + R0;            // A(row, col) at col*f + row
  const double* W = batch_at(c.dinv, sy, bt) + c.dinv_off[s] + inv_at(si.nc, step);
  const int ldw = inv_ld(si.nc, k0 / INV_GROUP);
  const int np = (b + PW - 1) / PW;
  const int lane = threadIdx.x & 63, wave = uni(threadIdx.x >> 6);
  const int i16 = lane & 15, k4 = lane >> 4;
  const uint32_t f8 = static_cast<uint32_t>(f) * 8u, w8 = static_cast<uint32_t>(ldw) * 8u;
  auto load = [](rsrc_t v, uint32_t vo, uint32_t so) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(v, vo, so, 0));
  };
  // A_p^T of each group, into the place of X_p^T: element v = A(row i16, column 16p + 4v
  // + k4), at byte va of view(A) and the column quadruple's uniform offset; rows and
  // columns past the end are off the view (they read 0 and are not stored)
  d4 x[NGW][NPN];
  const rsrc_t av = view(A, static_cast<int64_t>(b) * f8);
  const int last4 = (b - 1) / 4;   // the last column quadruple, perhaps partial
  uint32_t va[NGW], vlast[NGW];
#pragma unroll
  for (int gi = 0; gi < NGW; gi++) {
    const int g = wave + 4 * gi, row = 16 * g + i16;
    va[gi] = g < NG && row < M
                 ? static_cast<uint32_t>(row) * 8u + static_cast<uint32_t>(k4) * f8 : OFF_NONE;
    vlast[gi] = 4 * last4 + k4 < b ? va[gi] : OFF_NONE;
  }
  auto off_a = [&](int gi, int q) {
    const uint32_t full = va[gi], last = vlast[gi];   // values: chosen by address they are in scratch
    return q < last4 ? full : q == last4 ? last : OFF_NONE;
  };
  // stage: thread t holds entry (row t % 16, column t / 16) of every block, NBAT loads in
  // flight together; rows at or past b (the panel rows below a partial block) and blocks
  // past it read as 0
  {
    const int rr = threadIdx.x % PW, cc = threadIdx.x / PW, nfull = b / PW;
    const rsrc_t vl = view(Lkk, static_cast<int64_t>(b) * f8), vw = view(W, static_cast<int64_t>(BT) * w8);
    const uint32_t full = static_cast<uint32_t>(rr) * 8u + static_cast<uint32_t>(cc) * f8;
    const uint32_t part = rr < b - PW * nfull ? full : OFF_NONE;
    const uint32_t wo = static_cast<uint32_t>(rr) * 8u + static_cast<uint32_t>(cc) * w8;
    constexpr int NBAT = 18;
#pragma unroll
    for (int t0 = 0; t0 < TRSM_NB + NPN; t0 += NBAT) {
      double v[NBAT];
#pragma unroll
      for (int t = t0; t < t0 + NBAT; t++) {
        int p = 1;
        while ((p + 1) * p / 2 <= t) p++;   // compile-time after unrolling
        const int q = t - p * (p - 1) / 2, pi = t - TRSM_NB;
        v[t - t0] = t < TRSM_NB
                        ? load(vl, p < nfull ? full : p == nfull ? part : OFF_NONE,
                               static_cast<uint32_t>(PW * p) * 8u + static_cast<uint32_t>(PW * q) * f8)
                        : load(vw, pi < np ? wo : OFF_NONE, static_cast<uint32_t>(PW * pi) * (8u + w8));
      }
#pragma unroll
      for (int t = t0; t < t0 + NBAT; t++) smem[t * PW * PW + threadIdx.x] = v[t - t0];
    }
  }
  // A of the panels ahead, in their X's registers: five for one group a wave (112
  // registers in all), the next one for two
  constexpr int AHEAD = NGW == 1 ? 5 : 1;
  auto load_a = [&](int p) {
#pragma unroll
    for (int gi = 0; gi < NGW; gi++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        x[gi][p][v] = load(av, off_a(gi, 4 * p + v), static_cast<uint32_t>(PW * p + 4 * v) * f8);
  };
#pragma unroll
  for (int p = 0; p < AHEAD; p++) load_a(p);
  __syncthreads();
  if (PW * wave >= M) return;   // no barrier follows
#pragma unroll
  for (int p = 0; p < NPN; p++) {
    if (p >= np) break;
    d4 acc[NGW];
#pragma unroll
    for (int gi = 0; gi < NGW; gi++) acc[gi] = x[gi][p];
    if (p + AHEAD < NPN) load_a(p + AHEAD);
    // - sum_{q<p} L_pq X_q^T: A operand -L(16p + i16, 16q + 4 s4 + k4)
#pragma unroll
    for (int q = 0; q < NPN; q++) {
      if (q >= p) break;
      const double* blk = Ls + (p * (p - 1) / 2 + q) * PW * PW;
#pragma unroll
      for (int s4 = 0; s4 < 4; s4++) {
        const double a = -blk[(4 * s4 + k4) * PW + i16];
#pragma unroll
        for (int gi = 0; gi < NGW; gi++)
          acc[gi] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[gi][q][s4], acc[gi], 0, 0, 0);
      }
    }
    // X_p^T = inv16(L_pp) acc: A operand inv16(i16, 4 s4 + k4)
    d4 r[NGW];
#pragma unroll
    for (int gi = 0; gi < NGW; gi++) r[gi] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s4 = 0; s4 < 4; s4++) {
      const double a = Is[p * PW * PW + (4 * s4 + k4) * PW + i16];
#pragma unroll
      for (int gi = 0; gi < NGW; gi++)
        r[gi] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, acc[gi][s4], r[gi], 0, 0, 0);
    }
#pragma unroll
    for (int gi = 0; gi < NGW; gi++) {
      x[gi][p] = r[gi];
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (off_a(gi, 4 * p + v) != OFF_NONE)
          A[(PW * p + 4 * v + k4) * f + 16 * (wave + 4 * gi) + i16] = r[gi][v];
    }
  }
}

}  // namespace

// Columns of a 32-row update tile per workgroup: see k_dense_nt's launch below.
constexpr int SHORT_TN = 64;
// LDS that keeps an update tile off the compute unit of a 128-wide diagonal
// block (130 of the 160 KB), for launches small enough to find room elsewhere:
// FP64 VALU instructions wait for the matrix instructions of the waves they
// share a SIMD with, and a diagonal block beside a tile takes 46 us instead of
// 28.  A big trailing update keeps no LDS: its tiles fill every compute unit
// for longer than the block would wait (5,000 buses: factor 3.47 -> 3.36 ms,
// 10,000: 11.3 -> 11.16; with the LDS for every launch 20,000: 51.1 -> 51.9).
constexpr size_t ALONE_LDS = 31 * 1024;

void dense_nt(const CholDev& c, int ntasks, const int* tsn, const int* ttr, const int* ttc,
              int mode, int step, const Batch& b, hipStream_t st, bool short_rows, hipEvent_t done,
              bool alone, bool quarters)
{
  if (ntasks <= 0 || b.count <= 0) return;
  // `done` rides on the launch itself (its completion signal), so no marker
  // of its own sits between this kernel and the next one of the stream
  if (short_rows)
    hipExtLaunchKernelGGL((k_dense_nt<false, 32, 2, 1, 4, 8>), dim3(ntasks, b.count, BT / SHORT_TN),
                          dim3(256), 0, st, nullptr, done, 0, c, tsn, ttr, ttc, mode, step, b);
  else if (quarters)
    hipExtLaunchKernelGGL((k_dense_nt<false, 64, 2, 2, 2, 4>), dim3(ntasks, b.count, 4), dim3(256),
                          alone ? ALONE_LDS : 0, st, nullptr, done, 0, c, tsn, ttr, ttc, mode, step, b);
  else
    hipExtLaunchKernelGGL((k_dense_nt<false, 128, 4, 4, 2, 2>), dim3(ntasks, b.count), dim3(256),
                          alone ? ALONE_LDS : 0, st, nullptr, done, 0, c, tsn, ttr, ttc, mode, step, b);
  HIPCHK(hipGetLastError());
}

void update_matrices(const CholDev& c, int ntasks, const int* tsn, const int* ttr, const int* ttc,
                     bool small, const Batch& b, hipStream_t st)
{
  if (ntasks <= 0 || b.count <= 0) return;
  const dim3 grid(ntasks, b.count);
  if (small) k_dense_nt<true, 64, 2, 2, 2, 4><<<grid, 256, 0, st>>>(c, tsn, ttr, ttc, 1, 0, b);
  else k_dense_nt<true, 128, 4, 2, 4, 2><<<grid, 512, 0, st>>>(c, tsn, ttr, ttc, 1, 0, b);
  HIPCHK(hipGetLastError());
}

void front_panel(const CholDev& c, int ntasks, const int* tsn, const int* ttr, const Batch& b,
                 hipStream_t st)
{
  if (ntasks <= 0 || b.count <= 0) return;
  k_front_panel<<<dim3(ntasks, b.count), 256, 0, st>>>(c, tsn, ttr, b);
  HIPCHK(hipGetLastError());
}

void trsm_inv(const CholDev& c, int ntasks, const int* tsn, const int* ttr, int step,
              const Batch& b, hipStream_t st, bool short_rows)
{
  if (ntasks <= 0 || b.count <= 0) return;
  constexpr size_t SM = 2 * KC * LDA_S * sizeof(double);
  const dim3 grid(ntasks, b.count);
  if (short_rows) k_trsm_inv<32><<<grid, 256, SM, st>>>(c, tsn, ttr, step, b);
  else k_trsm_inv<128><<<grid, 256, SM, st>>>(c, tsn, ttr, step, b);
  HIPCHK(hipGetLastError());
}

void inv_groups(const CholDev& c, int ntasks, const int* tsn, const int* tix, const Batch& b,
                hipStream_t st)
{
  if (ntasks <= 0 || b.count <= 0) return;
  static const bool attr = [] {
    HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_inv_group),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(IG_SMEM)));
    return true;
  }();
  (void)attr;
  k_inv_group<<<dim3(ntasks, b.count), 512, IG_SMEM, st>>>(c, tsn, tix, b);
  HIPCHK(hipGetLastError());
}

void trsm(const CholDev& c, int ntasks, const int* tsn, const int* ttr, int step, const Batch& b,
          hipStream_t st, bool short_rows)
{
  if (ntasks <= 0 || b.count <= 0) return;
  static const bool attr = [] {
    HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_trsm<64>),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(TRSM_SMEM)));
    HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_trsm<128>),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(TRSM_SMEM)));
    return true;
  }();
  (void)attr;
  const dim3 grid(ntasks, b.count);
  if (short_rows) k_trsm<64><<<grid, 256, TRSM_SMEM, st>>>(c, tsn, ttr, step, b);
  else k_trsm<128><<<grid, 256, TRSM_SMEM, st>>>(c, tsn, ttr, step, b);
  HIPCHK(hipGetLastError());
}

template <int BK>
static size_t potrf_smem()
{
  // P and the reciprocals of the diagonal
  return (BK * (BK + 1) + BK) * sizeof(double);
}

template <int BK>
static void launch_potrf(const CholDev& c, int nsn, const int* sns, int step, const Batch& b,
                         hipStream_t st)
{
  // set once per process; a function-local static initialises thread-safely
  static const bool attr = [] {
      HIPCHK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_potrf_inv<BK>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(potrf_smem<BK>())));
    return true;
  }();
  (void)attr;
  k_potrf_inv<BK><<<dim3(nsn, b.count), 256, potrf_smem<BK>(), st>>>(c, sns, step, b);
  HIPCHK(hipGetLastError());
}

void potrf_inv(const CholDev& c, int nsn, const int* sns, int step, int max_b, const Batch& b,
               hipStream_t st)
{
  if (nsn <= 0 || b.count <= 0) return;
  if (max_b <= 32) launch_potrf<32>(c, nsn, sns, step, b, st);
  else if (max_b <= 64) launch_potrf<64>(c, nsn, sns, step, b, st);
  else launch_potrf<128>(c, nsn, sns, step, b, st);
}

}  // namespace dev
}  // namespace hykkt
