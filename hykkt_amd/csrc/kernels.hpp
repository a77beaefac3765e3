// kernels.hpp -- launchers for the gfx950 HIP kernels (device pointers only).
//
// Systems of a launch.  Every per-system launcher takes a Batch: `count`
// systems that share one sparsity pattern, whose per-system buffers (values,
// vectors, factor storage) sit `vs` doubles apart -- system k's copy of a
// buffer p is p + k*vs -- while index arrays (patterns, maps, task lists) are
// shared.  System k runs in blockIdx.y == k (or, for the triangular sweeps, in
// every count-th item), with exactly the arithmetic it gets alone, so a
// system's results do not depend on the batch it is in.  `mask`, when not
// null, holds one int per system; systems with 0 are skipped.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace hykkt {
namespace dev {

void check(hipError_t e, const char* what);
#define HIPCHK(x) ::hykkt::dev::check((x), #x)

struct Batch {
  int count = 1;
  int64_t vs = 0;             // per-system stride of the buffers (doubles)
  const int* mask = nullptr;  // per system: 0 = skip
};
inline Batch masked(const Batch& b, const int* m) { return Batch{b.count, b.vs, m}; }

// The bit pattern a sweep's exchanged values hold until they are written: a
// signalling-NaN payload no arithmetic result carries.
constexpr uint64_t SWEEP_SENTINEL = 0x7ff4dead0badf00dull;
// The buffers of one solve to fill with it before the sweeps (p[j], n[j] doubles
// per system) and the sweeps' four item counters to zero; empty: nothing to do.
struct SweepFill {
  double* p[4] = {};
  int64_t n[4] = {};
  int* ticket = nullptr;
};

// ---------------------------------------------------------------- vectors
void fill(double* p, double v, int64_t n, const Batch& b, hipStream_t st);
// p[i] = v for i < n, one array (no batch)
void fill_i(int* p, int v, int64_t n, hipStream_t st);
void copy(double* dst, const double* src, int64_t n, const Batch& b, hipStream_t st);
// dst[i] = src[map[i]] with 64-bit positions (one system)
void gather64(double* dst, const double* src, const int64_t* map, int64_t n, hipStream_t st);
// y[i] *= s[i]  (vec_scale, matrix_vector_ops.cu:385-392)
void vec_scale(double* y, const double* s, int n, const Batch& b, hipStream_t st);
// Caller memory into arena slots: for systems s < b.count, array j < COPY_ARRAYS of
// system s from src[s * COPY_ARRAYS + j] (device pointers, len[j] doubles; null:
// zeros if zero_null[j], else left alone) to dst[j] + s*vs, and scalar[s] to
// dst_scalar + s*vs.  The pointers and scalars travel as kernel arguments,
// COPY_SYSTEMS systems a launch: nothing is staged or copied ahead.  start (may be
// null): event recorded as the first launch starts.
constexpr int COPY_ARRAYS = 9, COPY_SYSTEMS = 16;
void copy_in(double* const* dst, const int64_t* len, const bool* zero_null,
             const double* const* src, double* dst_scalar, const double* scalar, const Batch& b,
             hipStream_t st, hipEvent_t start = nullptr);

// ---------------------------------------------------------------- sparse
// jd_vs = Ds-row-scaled Jd (skipped if jd_vs is null); ryd_s = ryd*ds + rs
// (row_scale :490-509, add_vecs :310-317).  word0, word1 (may be null): one int per
// system each, set to INT_MAX.
void row_scale(int d, const int* jd_rp, const double* jd_v, const double* ds,
               const double* ryd, const double* rs, double* jd_vs, double* ryd_s,
               const Batch& b, hipStream_t st, int* word0 = nullptr, int* word1 = nullptr);
// Row blocks of a CSR matrix for the LDS-staged SpMV: consecutive rows with
// at most spmv_lds_entries() entries together (a longer row is a block of its
// own); blocks[k] = first row of block k, blocks[nblk] = nrows.
int spmv_lds_entries();
// y_out[i] = alpha*t + beta*y_in[i] (beta == 0: alpha*t),
// t = sum over the row of fma(v[map ? map[q] : q], x[ci[q]], t) in column
// order.  The row block's values and x entries are staged through LDS with
// coalesced loads, then each row is summed by one thread in that order.
// alpha_ps (may be null): per-system alpha (arena slot) instead of alpha.
// dot_w (may be null): also dot_part[blk] = sum over the block's rows of
// y_out[i] * dot_w[i] (per-system, for a fused w.r).  y_map (may be null): y_in is
// read at y_map[i].  fill: sweep buffers to prepare on the way.
void spmv(int nrows, const int* rp, const int* ci, const int* map, const double* v, double alpha,
          const double* alpha_ps, const double* x, double beta, const double* y_in,
          double* y_out, const int* blocks, int nblk, const Batch& b, hipStream_t st,
          const double* dot_w = nullptr, double* dot_part = nullptr, const int* y_map = nullptr,
          const SweepFill& fill = SweepFill{});
// y = A x, the same sums, without row blocks planned ahead (64 rows a workgroup).
void spmv_rows(int nrows, const int* rp, const int* ci, const double* v, const double* x, double* y,
               const Batch& b, hipStream_t st);
// out[p] = d_v[d_src[p]] (or 0) + alpha_p*acc, acc = sum fma(av[ta], bv[tb]) over terms of p
void spgemm_values(int nnz_out, const int* d_src, const double* d_v, const int* term_ptr,
                   const int* ta, const int* tb, const double* av, const double* bv,
                   double alpha_p, double* out, const Batch& b, hipStream_t st);
// out[ent_dst[e]] = value of entry ent_src[e] (as spgemm_values, alpha_p from
// the per-system slot alpha_ps)
void spgemm_scatter(int nent, const int* ent_src, const int64_t* ent_dst, const int* d_src,
                    const double* d_v, const int* term_ptr, const int* ta, const int* tb,
                    const double* av, const double* bv, const double* alpha_ps, double* out,
                    const Batch& b, hipStream_t st);
// out[dst[e]] = vals[src[e]] for e < n
void scatter(double* out, const int64_t* dst, const double* vals, const int* src, int n,
             const Batch& b, hipStream_t st);
// add `delta` at out[pos[i]] for i < n (add_diag hook, matrix_vector_ops.cu:344-358)
void add_at(double* out, const int64_t* pos, int n, double delta, const Batch& b,
            hipStream_t st);

// ---------------------------------------------------------------- Ruiz
// adapt_row_max (matrix_vector_ops.cu:218-266). Jt rows read as jt_v[jt_map ? jt_map[q] : q].
// zero_row (may be null; one int per system): receives the smallest row index
// whose entries are all zero (its scale is 1/sqrt(0)); the caller initialises it.
void ruiz_rowmax(int n, int totn, const int* h_rp, const double* h_v, const int* jt_rp,
                 const int* jt_map, const double* jt_v, const int* j_rp, const double* j_v,
                 double* scale, int* zero_row, const Batch& b, hipStream_t st);
// One pass of the solver's Ruiz scaling over [H~ Jc^T; Jc], Jc^T's values read from
// Jc's through jt_map: with scale_in, the last scale applied (h_v in place, j_src
// -> j_dst, rhs1 in place, rhs2_src -> rhs2, max_d, which `first` starts); with
// scale_out, the next scale formed from the scaled rows (and zero_row as above).
// j_dst must not be j_src where both are given.
struct RuizPass {
  int n, m;
  const int *h_rp, *h_ci;
  double* h_v;
  const int *jt_rp, *jt_ci, *jt_map, *j_rp, *j_ci;
  const double* j_src;
  double* j_dst;
  const double* scale_in;
  double* scale_out;
  double* rhs1;
  const double* rhs2_src;
  double* rhs2;
  double* max_d;
  int first;
  int* zero_row;
};
void ruiz_pass(const RuizPass& c, const Batch& b, hipStream_t st);
// adapt_diag_scale (matrix_vector_ops.cu:146-186); jt_v_scaled may be null (Jt shares J).
// first != 0: max_d is written as 1*scale (reset, :268-283, fused).
void ruiz_scale(int n, int totn, const int* h_rp, const int* h_ci, double* h_v,
                const int* jt_rp, const int* jt_ci, double* jt_v_scaled,
                const int* j_rp, const int* j_ci, double* j_v, const double* scale,
                double* rhs1, double* rhs2, double* max_d, int first, const Batch& b,
                hipStream_t st);

// ---------------------------------------------------------------- reductions
// Block partial sums of a length-n reduction: reduce_blocks(n) blocks, a
// function of n only (the same for every batch).
__host__ __device__ inline int reduce_blocks_of(int64_t n)
{
  const int64_t g = (n + 255) / 256;
  return static_cast<int>(g < 1 ? 1 : (g > 256 ? 256 : g));
}
inline int reduce_blocks(int64_t n) { return reduce_blocks_of(n); }
// Deterministic partial sums of a[i]*b[i] in part: reduce_blocks(n) per system.
void dot_partial(int n, const double* a, const double* bv, double* part, const Batch& b,
                 hipStream_t st);

// ---------------------------------------------------------------- CG
// CG scalars per system: gam (r.r) and alpha of iteration k at the parity of k,
// the last r.r.
enum { CG_GAM = 0, CG_ALPHA = 2, CG_RR = 4, CG_SLOTS = 8 };
// Per-system ints (one array each, indexed by system): live (1 while the
// system iterates), iters, status.
struct CgFlags {
  int* live;
  int* iters;
  int* status;
};
// The CG's vectors of system 0: x, r, w, p, s (m); t1, t2 (n, the solves' right-
// hand side and solution); optionally q, z (n); scalars; partials of r.r
// (reduce_blocks(m)) and of w.r (np2).
struct CgVecs {
  int m, n;
  double *x, *r, *w, *p, *s, *t1, *t2, *q, *z, *sc, *part, *part2;
  int np2;
};
// The flags of all b.count systems (live: those of b.mask); p = s = rhs, q = z =
// 0 and, with x0_zero, x = 0, r = rhs and the partials of r.r.
void cg_start(const CgVecs& c, const double* rhs, bool x0_zero, const CgFlags& f, const Batch& b,
              hipStream_t st);
// The stopping test after k updates, then t1 = Jh^T r and the sweeps' buffers filled.
void cg_apply(const CgVecs& c, int k, double tol, int itmax, const int* jth_rp, const int* jth_ci,
              const double* jth_v, const SweepFill& fill, const CgFlags& f, const Batch& b,
              hipStream_t st);
// Iteration k's update of x, r, p, s (and q, z) and the partials of r.r.
void cg_update(const CgVecs& c, int k, const CgFlags& f, const Batch& b, hipStream_t st);

// ---------------------------------------------------------------- pass
// After the factorization: jh_v[i] = jcs[jh_map[i]], jth_v[i] = jcs[jth_map[i]]; ok = 0
// and a zero solution for systems with a failing pivot, else ok = 1.  start
// (may be null): event recorded as the launch starts.
struct AfterFactor {
  const int* pivot;
  int* ok;
  const double* jcs;
  const int *jh_map, *jth_map;
  double *jh_v, *jth_v;
  int nnz, n, m, d;
  double *dx, *dsv, *dyc, *dyd;
};
void after_factor(const AfterFactor& c, const Batch& b, hipStream_t st, hipEvent_t start = nullptr);
// The solution of the 4x4 system from the CG's iterate: dx[i] = (h0[ipos[i]] -
// z[ipos[i]]) max_d[i], dyc = x max_d[n..], dsv = Jd dx - ryd (has_jd = 0: -ryd), dyd =
// dsv Ds - rs; base_* (may be null): added to the results.
struct Recover {
  int n, m, d, has_jd;
  const double *h0, *z, *x, *max_d;
  const int *ipos, *jd_rp, *jd_ci;
  const double *jd_v, *ryd, *ds, *rs;
  double *dx, *dsv, *dyc, *dyd;
  const double *base_dx, *base_dsv, *base_dyc, *base_dyd;
  int nbd;   // set by recover()
};
void recover(Recover c, const Batch& b, hipStream_t st, hipEvent_t start = nullptr);
// Signed residual rows e_x = rx - H dx - Jc^T dyc - Jd^T dyd (ct_*, dt_*: the
// transposes' patterns and their maps into the values), e_y = ry - Jc dx, e_s = rs -
// (Ds ds - dyd), e_d = ryd - (Jd dx - ds), and partial sums of squares for
// finish() (residual_partials() doubles per system).
struct Residual {
  int n, m, d, has_jd;
  const int *h_rp, *h_ci, *ct_rp, *ct_ci, *ct_map, *dt_rp, *dt_ci, *dt_map, *jc_rp, *jc_ci, *jd_rp,
      *jd_ci;
  const double *h_v, *jc_v, *jd_v, *ds, *rx, *rs, *ry, *ryd, *dx, *dsv, *dyc, *dyd;
  double *e_x, *e_s, *e_y, *e_d, *part;
  int nbn, nbm, nbd, stride;   // set by residual()
};
int residual_partials(int n, int m, int d);
void residual(Residual& c, const Batch& b, hipStream_t st);
// What the host reads of a pass, per system: squared norms of residual rows 1, 3,
// 2, 4 and of rx, rs, ry, ryd; the CG's r.r at exit, iterations, status and live
// flag; the zero-row and pivot words (INT_MAX: none), the sweeps' error word.
enum {
  FIN_RES = 0, FIN_RR = 8, FIN_ITERS, FIN_STATUS, FIN_LIVE, FIN_ZERO_ROW, FIN_PIVOT, FIN_SWEEP_ERR,
  FIN_SLOTS = 16
};
struct Finish {
  double* out;   // FIN_SLOTS doubles per system, in memory the host can read
  const int *zero_row, *pivot, *sweep_err;
  const double* part;   // set by finish()
  int np[8], stride;
};
// After k updates: the CG's stopping test, the residual's sums (r: of the launch
// before; may be null) and out.  stop (may be null): event recorded at the end.
void finish(Finish c, const Residual* r, const CgVecs& v, int k, double tol, int itmax,
            const CgFlags& f, const Batch& b, hipStream_t st, hipEvent_t stop = nullptr);
// dst[j] <- src[j] (n[j] doubles) for the systems with keep != 0 (null: all)
struct Keep {
  const double* src[4];
  double* dst[4];
  int n[4];
};
void keep_where(const Keep& c, const int* keep, const Batch& b, hipStream_t st);

// The allocation-free entry point's device scratch (noalloc.hip): its size
// in bytes, and its address on the current device (taken once per device).
size_t noalloc_scratch_bytes();
void* noalloc_scratch();

// ---------------------------------------------------------------- Cholesky
// Offset of (r, c), r >= c, in an n x n lower triangle packed by columns: c n - c
// (c + 1) / 2 + r, with one 32 x 32 bit product.
__host__ __device__ inline int64_t packed_lower(int r, int c, int n)
{
  const uint32_t uc = static_cast<uint32_t>(c), m = 2u * static_cast<uint32_t>(n) - uc - 1u;
  return static_cast<int64_t>((static_cast<uint64_t>(uc) * m) >> 1) + r;
}

// A child of a supernode, in child-list order: its update matrix and that one's size.
struct ChildRec {
  int64_t u_off;
  int nr, pad;
};
// What a workgroup needs to know of a supernode.  Child t's row of its update matrix
// at front row r, or -1: inv[inv_off + t * inv_rows + r] (the rows below the
// supernode's columns; for at most FRONT_NC columns those, too).  nch = 0: no children,
// or extend_add() adds them.
struct SnRec {
  int a, nc, nr;      // first column, columns, rows below them
  int child0, nch;    // its children in child_rec
  int inv_rows;
  int pad[2];
  int64_t l_off, dinv_off, u_off, inv_off;
};
// Widest supernode that front_panel() takes.
constexpr int FRONT_NC = 32;

// Inverses of the factor's diagonal blocks, in groups of INV_GROUP columns: group g
// of a supernode is a column-major inv_ld x inv_ld matrix at g * INV_GROUP^2 from
// the supernode's slot, its lower triangle the inverse of L's (supernodes of at most
// FRONT_NC columns: one 32 x 32 matrix).
constexpr int INV_GROUP = 512;
__host__ __device__ inline int inv_ld(int nc, int g)
{
  if (nc <= FRONT_NC) return FRONT_NC;
  const int n = nc - g * INV_GROUP;
  return n >= INV_GROUP ? INV_GROUP : (n + 127) / 128 * 128;
}
__host__ __device__ inline int64_t inv_size(int nc)
{
  const int g = (nc - 1) / INV_GROUP, ld = inv_ld(nc, g);
  return static_cast<int64_t>(g) * INV_GROUP * INV_GROUP + static_cast<int64_t>(ld) * ld;
}
// Its diagonal block `step` (128 columns).
__host__ __device__ inline int64_t inv_at(int nc, int step)
{
  const int g = step / (INV_GROUP / 128), i = step - g * (INV_GROUP / 128);
  return static_cast<int64_t>(g) * INV_GROUP * INV_GROUP +
         static_cast<int64_t>(i) * 128 * (inv_ld(nc, g) + 1);
}

// The factor storage of system 0 (system k's at + k*vs, vs of the Batch).
struct CholDev {
  int n, ns;
  const int* sn_first;      // ns+1
  const int* rows_ptr;      // ns+1
  const int* rows;
  const int* rel;
  const int64_t* l_off;     // ns+1
  const int64_t* u_off;     // ns+1: U(s) offsets in the reused update space
  const ChildRec* child_rec;   // by position in the plan's child_list
  const SnRec* sn_rec;
  const int* inv;              // see SnRec
  double* L;
  double* U;
  int* pivot;               // one int per system: first failing pivot (min), INT_MAX if none
  double pivot_tol;
  double* dinv;             // inverses of the diagonal blocks (see inv_ld)
  const int64_t* dinv_off;  // ns+1, supernode s's slot in dinv
};

// Extend-add tasks: task t = (parent p, front column col: of the panel or below it);
// contributions [cptr[t], cptr[t+1]) are (child, child-local column) pairs.
void extend_add(const CholDev& c, int ntasks, const int* task_p, const int* task_col,
                const int* cptr, const int* contrib_child, const int* contrib_col,
                const Batch& b, hipStream_t st);
// Factor + invert the (<= 128 wide) diagonal block of step `step` of each
// supernode; max_b = largest block in the launch (selects the LDS footprint).
// dinv slots must be zero-initialized once (only the b x b lower part is written).
// Blocks wider than 64 (max_b > 64) leave only the inverses of their 16x16
// diagonal blocks in the slot: their TRSM is trsm(), the whole inverse comes
// from inv_groups() after the last level.
void potrf_inv(const CholDev& c, int nsn, const int* sns, int step, int max_b, const Batch& b,
               hipStream_t st);
// L21 = A21 L_kk^{-T} below the 128-wide diagonal blocks of step `step` by blocked
// substitution (tasks: supernode, tile row of TM = 64 (short_rows) or 128 rows).
void trsm(const CholDev& c, int ntasks, const int* task_sn, const int* task_tr, int step,
          const Batch& b, hipStream_t st, bool short_rows);
// The groups' whole inverses, from the factor and the inverses of its 16x16 diagonal
// blocks (tasks: supernode, 32 * group + strip of 16 columns; a group's last strip has
// nothing to form).
void inv_groups(const CholDev& c, int ntasks, const int* tsn, const int* tix, const Batch& b,
                hipStream_t st);

// MFMA update tiles over (supernode, tile row, tile col) tasks.  mode 0: trailing
// panel update after block `step`; mode m >= 3: after blocks `step` .. `step`+m-2
// (K = (m-1) blocks).  Tiles of 128 x 128, or of 32 rows x 128 columns
// (short_rows), or each 128 x 128 tile as four of 64 x 64 (quarters).  done: optional
// event recorded by the launch's own completion.  alone: tiles keep off a compute
// unit that factors a 128-wide diagonal block.
void dense_nt(const CholDev& c, int ntasks, const int* task_sn, const int* task_tr,
              const int* task_tc, int mode, int step, const Batch& b, hipStream_t st,
              bool short_rows = false, hipEvent_t done = nullptr, bool alone = false,
              bool quarters = false);
// The update matrices U = -L21 L21^T + the children's, tasks as above with tiles of
// 128 x 128 (small: 64 x 64) entries of U.
void update_matrices(const CholDev& c, int ntasks, const int* task_sn, const int* task_tr,
                     const int* task_tc, bool small, const Batch& b, hipStream_t st);
// Supernodes of at most FRONT_NC columns: children's entries added to the panel,
// diagonal block factored and inverted, L21 formed; tasks (supernode, tile of 128
// rows below the columns; a supernode without such rows: one task).
void front_panel(const CholDev& c, int ntasks, const int* task_sn, const int* task_tile,
                 const Batch& b, hipStream_t st);
// TRSM of the rows below blocks of at most 64 columns with their whole inverses,
// in place (tasks as trsm()'s).
void trsm_inv(const CholDev& c, int ntasks, const int* task_sn, const int* task_tr, int step,
              const Batch& b, hipStream_t st, bool short_rows);

// Whether kernels of the two streams run at the same time: a kernel on `a` waits
// (a bounded number of polls) for a word that one on `b` sets.  Streams that
// share a hardware queue never do.  Synchronizes both; words: 2 ints of device
// memory.
bool streams_overlap(hipStream_t a, hipStream_t b, int* words);

// Single-launch supernodal solves over the whole tree.  Work items are parts
// of the fronts, dispatched in a dependency-respecting order;
// items synchronise on the values they exchange, whose buffers are filled
// with a sentinel (fill_sentinel) before each sweep.  With several systems,
// launch item i*count + k is item i of system k.
constexpr int FOREST_NC = 32;   // most columns of a forest supernode
constexpr int FOREST_F = 512;   // most front rows of one
constexpr int FOREST_WAVE_F = 64;   // most front rows of one that takes one wave

// What a sweep item needs to know of a forest supernode.
struct ForestSn {
  int a, nc, nr, pad;        // first column, columns, rows below them
  int64_t l_off, dinv_off;   // panel, inverted diagonal block
  int64_t uvec_off;          // its update vector in ubuf
  int64_t front_off;         // its front rows in the pull_ptr index
  int64_t rows_off;          // its rows in CholDev::rows
  int64_t pad2;
};

// Items of the top of the tree (see kernels_trsv.hip): their kinds, the rows of a
// pivot or chunk item, the waves that share a column set of an item of rows below
// nc columns (16 columns each; the other waves take further sets of 128 rows), and
// how many times a backward item's 1024 rows (16 columns) halve (its columns
// double) for so many rows.
constexpr int TOP_RHS = 0, TOP_PIVOT = 1, TOP_CHUNK = 2, TOP_BELOW = 3;
constexpr int TOP_ROWS = 64;
__host__ __device__ inline int top_waves(int nc)
{
  return nc > 128 ? 16 : nc > 64 ? 8 : nc > 32 ? 4 : 2;
}
__host__ __device__ inline int top_shape(int rows)
{
  return rows > 512 ? 0 : rows > 256 ? 1 : rows > 128 ? 2 : 3;
}

struct SolveDev {
  // Items of the small-supernode forest (fwd_items, bwd_items: 4 ints each, indices
  // into `forest`; see kernels_forest.hip) and of the top of the tree (*_top: 4 ints
  // per item) are separate launches: forward forest then top, backward top then
  // forest.  Top items: supernode, kind, index, group (forward chunks).
  const ForestSn* forest;
  const int* fwd_items;
  int n_fwd;
  const int* bwd_items;
  int n_bwd;
  const int* fwd_items_top;
  int n_fwd_top;
  const int* bwd_items_top;
  int n_bwd_top;
  const int64_t* uvec_off;  // ns+1 offsets of the forward update vectors in ubuf
  const int* pull_ptr;      // front-row pull lists (children contributions)
  const int* pull_src;
  const int64_t* front_off; // ns+1: offset of s's front rows in the pull_ptr index
  double* ubuf;             // forward update vectors (sentinel-filled per sweep; per system)
  double* exch;             // the top's other exchanged values (sentinel-filled per sweep):
                            // n backward right-hand sides, then forward chunks, chunk j of
                            // s's pivot rows at exch_off[s] + j * nc
  const int64_t* exch_off;
  int* err;                 // 1: a wait hit its bound (sticky until the host clears it)
  int* ticket;              // 4 item counters (forward forest, forward top, backward top,
                            // backward forest), zeroed with the first sentinel fill of a solve
  int cap_top = 0;          // most workgroups of a top-of-tree sweep launch (0: one per item)
  int cap_forest = 0;       // most workgroups of a forest sweep launch (0: one per item)
};
// Workgroups of a forest sweep one compute unit holds at once.
int forest_blocks_per_cu();
// The buffers of f filled with the sentinel, in a launch of its own.
void fill_sentinel(const SweepFill& f, const Batch& b, hipStream_t st);
// L y = b (b, y internal order; y sentinel-filled, ubuf sentinel-filled): the
// forest, then the top of the tree.
void solve_forward_forest(const CholDev& c, const SolveDev& sd, const double* rhs, double* y,
                          const Batch& b, hipStream_t st);
void solve_forward_top(const CholDev& c, const SolveDev& sd, const double* rhs, double* y,
                       const Batch& b, hipStream_t st);
// L^T x = y (x and exch sentinel-filled): the top of the tree, then the forest.
void solve_backward_top(const CholDev& c, const SolveDev& sd, const double* y, double* x,
                        const Batch& b, hipStream_t st);
void solve_backward_forest(const CholDev& c, const SolveDev& sd, const double* y, double* x,
                           const Batch& b, hipStream_t st);

}  // namespace dev
}  // namespace hykkt
