// solver.cpp -- HykktSolver::execute() on one MI355X, for one system or a
// batch of systems that share one sparsity pattern.
//
// Step order follows HykktSolver.cpp:240-457 (+ check_error :846-930).
// Everything per solve runs on one HIP stream.  Every per-system buffer of a
// pattern lives in one arena, system k's copy `stride` doubles after system
// k-1's, so each launch covers all the systems of the batch (system
// blockIdx.y) and a system's arithmetic is the same alone or in a batch.
// The host reads a pass's results once: the device writes them to pinned memory.
#include "solver.hpp"

#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <numeric>

namespace hykkt {

// Per-system arena slots (offsets in doubles from the system's base).
struct Solver::Slots {
  int64_t in[IN_COUNT] = {}, gam = 0;
  int64_t jd_vs = 0, ryd_s = 0, rx_til = 0, htil = 0, jcs = 0, ry_s = 0, max_d = 0, scale = 0, scale2 = 0;
  int64_t jch_v = 0, jcth_v = 0, rxp = 0, t1 = 0, t2 = 0;
  int64_t cx = 0, cr = 0, cw = 0, cp = 0, cs = 0, schur = 0, sc = 0, part = 0, part2 = 0, rpart = 0;
  int64_t h0 = 0, cq = 0, cz = 0;
  int64_t dx = 0, dsv = 0, dyc = 0, dyd = 0;
  Rows e[2];   // residual rows: a pass's, and the ones the next pass corrects
  int64_t e_rxt = 0, e_ysc = 0, e_rxp = 0, e_schur = 0;
  int64_t e_cx = 0, c_dx = 0, c_dsv = 0, c_dyc = 0, c_dyd = 0;
  int64_t L = 0, U = 0, dinv = 0, y = 0, ubuf = 0, exch = 0;
  int64_t stride = 0;
};

// per-system int flags, one array of `cap` each
enum { FL_PIVOT = 0, FL_ZERO_ROW, FL_LIVE, FL_ACT, FL_KEEP, FL_CG_IT, FL_CG_ST, FL_OK, FL_COUNT };

struct Solver::Sym {
  int n = 0, m = 0, d = 0, nnz_h = 0, nnz_jc = 0, nnz_jd = 0, nnz_ds = 0;
  bool has_jd = false;
  Pattern H, Jc, Jd;
  TransposeMap jct, jdt;
  SpgemmPlan htp, hgp;
  std::vector<int> perm, rev;
  Pattern hgp_pat, jcp_pat, jctp_pat;
  std::vector<int> hgp_map, jcp_map, jctp_map;
  std::unique_ptr<CholEngine> chol;
  std::vector<int> phat, ipos;
  DevBuf<int> h_rp, h_ci, jc_rp, jc_ci, jd_rp, jd_ci;
  DevBuf<int> jct_rp, jct_ci, jct_map, jdt_rp, jdt_ci, jdt_map;
  DevBuf<int> ht_rp, ht_ci, ht_dsrc, ht_tp, ht_ta, ht_tb;
  DevBuf<int> hg_dsrc, hg_tp, hg_ta, hg_tb, ent_src;
  DevBuf<int> jch_rp, jch_ci, jch_map, jcth_rp, jcth_ci, jcth_map;
  DevBuf<int> phat_d, ipos_d;
  // row blocks of the LDS-staged SpMVs: Jd^T, Jc^T (internal order), Jc
  DevBuf<int> jdt_blk, jcth_blk, jch_blk;
  int jdt_nblk = 0, jcth_nblk = 0, jch_nblk = 0;
  // algorithmic work of one system's H~ and H_gamma value kernels (profiler)
  double ht_flops = 0, ht_bytes = 0, hg_flops = 0, hg_bytes = 0;
  // per-system storage for `cap` systems, and its flags and staging
  Slots z;
  int cap = 0;
  DevBuf<double> arena;
  DevBuf<int> flags;         // FL_COUNT arrays of cap ints
  // pinned: what the host reads of a pass (written by the device), and the
  // per-system flags it sends
  HostBuf<double> fin;
  HostBuf<int> flag_host;
  int* flag(int which) { return flags.p + static_cast<int64_t>(which) * cap; }
  // the engine's second stream may still be zeroing the factor storage in
  // the arena (prezero_L): let it finish before the members are freed
  ~Sym()
  {
    if (chol) chol->quiesce();
  }
};

namespace {

template <class T>
void upload_or_dummy(DevBuf<T>& b, const std::vector<T>& v)
{
  if (v.empty()) b.upload(std::vector<T>{T{}});
  else b.upload(v);
}

// Row blocks of the LDS-staged SpMV (see dev::spmv): up to 256 rows whose
// entries fit the LDS stage together; a longer row is a block of its own.
std::vector<int> spmv_blocks(const std::vector<int>& rp, int nrows)
{
  const int E = dev::spmv_lds_entries(), R = 256;
  std::vector<int> b{0};
  int r = 0;
  while (r < nrows) {
    const int e0 = rp[r];
    int r1 = r + 1;
    if (rp[r + 1] - e0 <= E)
      while (r1 < nrows && r1 - r < R && rp[r1 + 1] - e0 <= E) r1++;
    b.push_back(r1);
    r = r1;
  }
  return b;
}

}  // namespace

Solver::Solver(double gamma, int capacity) : gamma_(gamma), cap_(capacity)
{
  HYKKT_REQUIRE(capacity >= 1, HYKKT_E_ARG, "batch capacity must be at least 1");
  hykkt_default_options(&opts);
  HIPCHK(hipStreamCreate(&st_));
  for (auto& e : ev_) HIPCHK(hipEventCreate(&e));
  sys_in_.resize(cap_);
  st_k_.resize(cap_);
}

Solver::~Solver()
{
  sym_.reset();
  for (auto& e : ev_)
    if (e) (void)hipEventDestroy(e);
  if (st_) (void)hipStreamDestroy(st_);
}

double* Solver::P(int64_t off) const { return sym_->arena.p + off; }

void Solver::set_block(int which, const int* rp, const int* ci, const double* v, int n, int m,
                       int nnz)
{
  HYKKT_REQUIRE(which >= 0 && which < 4, HYKKT_E_ARG, "bad block id");
  HYKKT_REQUIRE(n >= 0 && m >= 0 && nnz >= 0, HYKKT_E_ARG, "negative dimension");
  HYKKT_REQUIRE(rp || n == 0, HYKKT_E_ARG, "null row pointer");
  HYKKT_REQUIRE((ci && v) || nnz == 0, HYKKT_E_ARG, "null column/value pointer");
  if (which == BLK_H || which == BLK_DS)
    HYKKT_REQUIRE(n == m, HYKKT_E_ARG, "H and Ds must be square");   // HykktSolver.cpp:165,172
  blk_[which] = BlockIn{rp, ci, v, n, m, nnz, true};
  file_path_ = false;
  if (which == BLK_JD) {
    // HykktSolver.cpp:188-191: the API path cannot detect pattern changes.
    jd_flag_ = nnz > 0;
    status_ = true;
  }
}

void Solver::set_vec(int which, const double* v, int n)
{
  HYKKT_REQUIRE(which >= 0 && which < 8, HYKKT_E_ARG, "bad vector id");
  HYKKT_REQUIRE(v || n == 0, HYKKT_E_ARG, "null vector");
  vecs_[which] = v;
  vec_n_[which] = n;
}

void Solver::set_perm(const int* perm, int n)
{
  std::vector<int> p(perm, perm + n), seen(n, 0);
  for (int v : p) {
    HYKKT_REQUIRE(v >= 0 && v < n && !seen[v], HYKKT_E_ARG, "not a permutation");
    seen[v] = 1;
  }
  user_perm_ = std::move(p);
  sym_.reset();   // re-analyse with the new ordering
}

void Solver::bind_system(int k, double gamma, const double* const vals[IN_COUNT])
{
  HYKKT_REQUIRE(k >= 0 && k < cap_, HYKKT_E_ARG, "system index beyond the batch capacity");
  for (int j = 0; j < IN_COUNT; j++)
    HYKKT_REQUIRE(vals[j] || j == IN_Y0 || j == IN_JD, HYKKT_E_ARG,
                  "null value array for a batch system");
  SystemIn& s = sys_in_[k];
  for (int j = 0; j < IN_COUNT; j++) s.v[j] = vals[j];
  s.gamma = gamma;
  s.set = true;
}

void Solver::read_files(const char* const files[8], int skip)
{
  // HykktSolver::read_matrix_files, HykktSolver.cpp:113-161
  fblk_[BLK_H] = read_mm_csr(files[0], skip, true);
  fblk_[BLK_DS] = read_mm_csr(files[1], skip, false);
  fblk_[BLK_JC] = read_mm_csr(files[2], skip, false);
  fblk_[BLK_JD] = read_mm_csr(files[3], skip, false);
  for (int k = 0; k < 4; k++) fvec_[k] = read_rhs(files[4 + k]);
  HYKKT_REQUIRE(static_cast<int>(fvec_[0].size()) == fblk_[BLK_H].n &&
                    static_cast<int>(fvec_[1].size()) == fblk_[BLK_DS].n &&
                    static_cast<int>(fvec_[2].size()) == fblk_[BLK_JC].n &&
                    static_cast<int>(fvec_[3].size()) == fblk_[BLK_JD].n,
                HYKKT_E_IO, "rhs length does not match its block");
  bool jd_flag = fblk_[BLK_JD].nnz() > 0;
  status_ = (jd_flag_ == jd_flag) || !sym_;
  jd_flag_ = jd_flag;
  for (int k = 0; k < 4; k++) {
    CsrHost& b = fblk_[k];
    blk_[k] = BlockIn{b.rp.data(), b.ci.empty() ? nullptr : b.ci.data(),
                      b.v.empty() ? nullptr : b.v.data(), b.n, b.m, b.nnz(), true};
  }
  for (int k = 0; k < 4; k++) {
    vecs_[k] = fvec_[k].data();
    vec_n_[k] = static_cast<int>(fvec_[k].size());
  }
  if (!vecs_[VEC_Y] || vec_n_[VEC_Y] != fblk_[BLK_JC].n) {
    fvec_[VEC_Y].assign(fblk_[BLK_JC].n, 0.0);   // h_y_ zeros (HykktSolver.cpp:153)
    vecs_[VEC_Y] = fvec_[VEC_Y].data();
    vec_n_[VEC_Y] = fblk_[BLK_JC].n;
  }
  file_path_ = true;
}

bool Solver::pattern_matches() const
{
  const Sym& S = *sym_;
  return blk_[BLK_H].n == S.n && blk_[BLK_H].nnz == S.nnz_h && blk_[BLK_JC].n == S.m &&
         blk_[BLK_JC].nnz == S.nnz_jc && blk_[BLK_JD].nnz == S.nnz_jd &&
         blk_[BLK_DS].n == S.d && blk_[BLK_DS].nnz == S.nnz_ds;
}

// ------------------------------------------------------------------ symbolic
void Solver::analyze()
{
  auto t0 = std::chrono::steady_clock::now();
  sym_.reset();
  auto S = std::make_unique<Sym>();
  const BlockIn &H = blk_[BLK_H], &Ds = blk_[BLK_DS], &Jc = blk_[BLK_JC], &Jd = blk_[BLK_JD];
  const int n = H.n, m = Jc.n, d = Ds.n;
  HYKKT_REQUIRE(Jc.m == n, HYKKT_E_ARG, "Jc must have n columns");
  HYKKT_REQUIRE(Jd.n == d && (Jd.m == n || Jd.nnz == 0), HYKKT_E_ARG,
                "Jd must be d x n with d = size of Ds");
  HYKKT_REQUIRE(Ds.nnz == d, HYKKT_E_ARG, "Ds must hold one diagonal entry per row");
  S->n = n;
  S->m = m;
  S->d = d;
  S->nnz_h = H.nnz;
  S->nnz_jc = Jc.nnz;
  S->nnz_jd = Jd.nnz;
  S->nnz_ds = Ds.nnz;
  S->has_jd = Jd.nnz > 0;
  const bool on_dev = opts.inputs_on_device != 0;
  auto fetch = [&](const BlockIn& b, Pattern& p, int rows, int cols) {
    p.n = rows;
    p.m = cols;
    p.rp.resize(static_cast<size_t>(rows) + 1);
    p.ci.resize(b.nnz);
    if (on_dev) {
      HIPCHK(hipMemcpy(p.rp.data(), b.rp, sizeof(int) * (rows + 1), hipMemcpyDeviceToHost));
      if (b.nnz) HIPCHK(hipMemcpy(p.ci.data(), b.ci, sizeof(int) * b.nnz, hipMemcpyDeviceToHost));
    } else {
      std::memcpy(p.rp.data(), b.rp, sizeof(int) * (rows + 1));
      if (b.nnz) std::memcpy(p.ci.data(), b.ci, sizeof(int) * b.nnz);
    }
    HYKKT_REQUIRE(p.rp[0] == 0 && p.rp[rows] == b.nnz, HYKKT_E_ARG, "bad CSR row pointer");
    for (int i = 0; i < rows; i++) {
      HYKKT_REQUIRE(p.rp[i + 1] >= p.rp[i], HYKKT_E_ARG, "CSR row pointer not monotone");
      for (int q = p.rp[i]; q < p.rp[i + 1]; q++) {
        HYKKT_REQUIRE(p.ci[q] >= 0 && p.ci[q] < cols, HYKKT_E_ARG, "column index out of range");
        HYKKT_REQUIRE(q == p.rp[i] || p.ci[q] > p.ci[q - 1], HYKKT_E_ARG,
                      "CSR columns must be sorted and unique");
      }
    }
  };
  fetch(H, S->H, n, n);
  fetch(Jc, S->Jc, m, n);
  Pattern dsp;
  fetch(Ds, dsp, d, d);
  for (int i = 0; i < d; i++)
    HYKKT_REQUIRE(dsp.rp[i + 1] - dsp.rp[i] == 1 && dsp.ci[dsp.rp[i]] == i, HYKKT_E_ARG,
                  "Ds must be diagonal with one entry per row");
  if (S->has_jd) fetch(Jd, S->Jd, d, n);
  else {
    S->Jd.n = d;
    S->Jd.m = n;
    S->Jd.rp.assign(static_cast<size_t>(d) + 1, 0);
  }

  // transposes (csr2csc every solve in the reference, HykktSolver.cpp:292-303,670-681)
  S->jct = transpose_map(S->Jc);
  S->jdt = transpose_map(S->Jd);
  // H~ = H + Jd^T (Ds Jd)  (HykktSolver.cpp:289-337, 685-697)
  if (S->has_jd) {
    S->htp = spgemm_plan(S->jdt.at, S->jdt.map, S->Jd, S->H);
  } else {
    S->htp.e = S->H;
    S->htp.d_src.resize(S->H.nnz());
    std::iota(S->htp.d_src.begin(), S->htp.d_src.end(), 0);
    S->htp.term_ptr.assign(static_cast<size_t>(S->H.nnz()) + 1, 0);
  }
  // H_gamma = H~ + gamma Jc^T Jc  (HykktSolver.cpp:352-383)
  S->hgp = spgemm_plan(S->jct.at, S->jct.map, S->Jc, S->htp.e);
  const Pattern& HG = S->hgp.e;
  // ordering + reference maps (HykktSolver.cpp:760-798)
  if (!user_perm_.empty()) {
    HYKKT_REQUIRE(static_cast<int>(user_perm_.size()) == n, HYKKT_E_ARG,
                  "permutation length differs from n");
    S->perm = user_perm_;
  } else {
    S->perm = amd_order(HG);
  }
  perm_reverse(S->perm, S->rev);
  perm_map_rc(HG, S->perm, S->rev, S->hgp_pat, S->hgp_map);
  perm_map_c(S->Jc, S->rev, S->jcp_pat, S->jcp_map);
  perm_map_r(S->jct.at, S->perm, S->jctp_pat, S->jctp_map);
  // Cholesky analysis of the lower triangle of P Hg P^T (CholeskyClass.cpp:31-58)
  S->chol = std::make_unique<CholEngine>(S->hgp_pat, CholOptions{}, st_);
  S->chol->set_profiler(&prof);
  const CholPlan& pl = S->chol->plan();
  S->phat.resize(n);
  S->ipos.resize(n);
  for (int k = 0; k < n; k++) {
    S->phat[k] = S->perm[pl.post[k]];
    S->ipos[S->phat[k]] = k;
  }
  std::vector<int> ent(pl.a_src.size());
  for (size_t e = 0; e < ent.size(); e++) ent[e] = S->hgp_map[pl.a_src[e]];
  // Jc with internal column order, and its transpose; maps into Jc positions
  Pattern jch;
  std::vector<int> jch_map;
  perm_map_c(S->Jc, S->ipos, jch, jch_map);
  TransposeMap jcht = transpose_map(jch);
  std::vector<int> jcth_map(jcht.map.size());
  for (size_t q = 0; q < jcth_map.size(); q++) jcth_map[q] = jch_map[jcht.map[q]];

  // ---- device index arrays ----
  S->h_rp.upload(S->H.rp);
  upload_or_dummy(S->h_ci, S->H.ci);
  S->jc_rp.upload(S->Jc.rp);
  upload_or_dummy(S->jc_ci, S->Jc.ci);
  S->jd_rp.upload(S->Jd.rp);
  upload_or_dummy(S->jd_ci, S->Jd.ci);
  S->jct_rp.upload(S->jct.at.rp);
  upload_or_dummy(S->jct_ci, S->jct.at.ci);
  upload_or_dummy(S->jct_map, S->jct.map);
  S->jdt_rp.upload(S->jdt.at.rp);
  upload_or_dummy(S->jdt_ci, S->jdt.at.ci);
  upload_or_dummy(S->jdt_map, S->jdt.map);
  S->ht_rp.upload(S->htp.e.rp);
  upload_or_dummy(S->ht_ci, S->htp.e.ci);
  upload_or_dummy(S->ht_dsrc, S->htp.d_src);
  S->ht_tp.upload(S->htp.term_ptr);
  upload_or_dummy(S->ht_ta, S->htp.ta);
  upload_or_dummy(S->ht_tb, S->htp.tb);
  upload_or_dummy(S->hg_dsrc, S->hgp.d_src);
  S->hg_tp.upload(S->hgp.term_ptr);
  upload_or_dummy(S->hg_ta, S->hgp.ta);
  upload_or_dummy(S->hg_tb, S->hgp.tb);
  upload_or_dummy(S->ent_src, ent);
  {
    // E = D + alpha A B with the pattern reused: each value of A, B, D and E
    // moved once, E's indices and row pointers once (the scatter also reads
    // each entry's 64-bit slot in the factor storage); 2 flops per term and
    // one per D entry.  H~ = H + Jd^T (Ds Jd), H_gamma = H~ + gamma Jc^T Jc
    // (its lower triangle).
    const double ht_terms = static_cast<double>(S->htp.ta.size());
    double hg_terms = 0;
    for (int e : ent) hg_terms += S->hgp.term_ptr[e + 1] - S->hgp.term_ptr[e];
    const double ne = static_cast<double>(S->htp.e.nnz()), ng = static_cast<double>(ent.size());
    S->ht_flops = 2.0 * ht_terms + S->nnz_h;
    S->ht_bytes = 8.0 * (2.0 * S->nnz_jd + S->nnz_h + ne) + 4.0 * (ne + n + 1);
    S->hg_flops = 2.0 * hg_terms + ng;
    S->hg_bytes = 8.0 * (2.0 * S->nnz_jc + ne + ng) + 4.0 * (ng + n + 1) + 8.0 * ng;
  }
  S->jch_rp.upload(jch.rp);
  upload_or_dummy(S->jch_ci, jch.ci);
  upload_or_dummy(S->jch_map, jch_map);
  S->jcth_rp.upload(jcht.at.rp);
  upload_or_dummy(S->jcth_ci, jcht.at.ci);
  upload_or_dummy(S->jcth_map, jcth_map);
  S->phat_d.upload(S->phat);
  S->ipos_d.upload(S->ipos);
  {
    std::vector<int> b = spmv_blocks(S->jdt.at.rp, n);
    S->jdt_nblk = static_cast<int>(b.size()) - 1;
    S->jdt_blk.upload(b);
    b = spmv_blocks(jcht.at.rp, n);
    S->jcth_nblk = static_cast<int>(b.size()) - 1;
    S->jcth_blk.upload(b);
    b = spmv_blocks(jch.rp, m);
    S->jch_nblk = static_cast<int>(b.size()) - 1;
    S->jch_blk.upload(b);
  }

  // ---- the per-system arena: slots in 256-byte units ----
  Slots& z = S->z;
  int64_t at = 0;
  auto slot = [&](int64_t len) {
    const int64_t o = at;
    at += (std::max<int64_t>(len, 1) + 31) / 32 * 32;
    return o;
  };
  z.in[IN_H] = slot(S->nnz_h);
  z.in[IN_DS] = slot(d);
  z.in[IN_JC] = slot(S->nnz_jc);
  z.in[IN_JD] = slot(S->nnz_jd);
  z.in[IN_RX] = slot(n);
  z.in[IN_RS] = slot(d);
  z.in[IN_RY] = slot(m);
  z.in[IN_RYD] = slot(d);
  z.in[IN_Y0] = slot(m);
  z.gam = slot(1);
  z.jd_vs = slot(S->nnz_jd);
  z.ryd_s = slot(d);
  z.rx_til = slot(n);
  z.htil = slot(S->htp.e.nnz());
  z.jcs = slot(S->nnz_jc);
  z.ry_s = slot(m);
  z.max_d = slot(n + m);
  z.scale = slot(n + m);
  z.scale2 = slot(n + m);
  z.jch_v = slot(S->nnz_jc);
  z.jcth_v = slot(S->nnz_jc);
  z.rxp = slot(n);
  z.t1 = slot(n);
  z.t2 = slot(n);
  z.h0 = slot(n);
  z.cq = slot(n);
  z.cz = slot(n);
  z.cx = slot(m);
  z.cr = slot(m);
  z.cw = slot(m);
  z.cp = slot(m);
  z.cs = slot(m);
  z.schur = slot(m);
  z.sc = slot(dev::CG_SLOTS);
  z.part = slot(dev::reduce_blocks(m));
  z.part2 = slot(S->jch_nblk);
  z.rpart = slot(dev::residual_partials(n, m, d));
  z.dx = slot(n);
  z.dsv = slot(d);
  z.dyc = slot(m);
  z.dyd = slot(d);
  for (Rows& e : z.e) e = Rows{slot(n), slot(d), slot(m), slot(d)};
  z.e_rxt = slot(n);
  z.e_ysc = slot(m);
  z.e_rxp = slot(n);
  z.e_schur = slot(m);
  z.e_cx = slot(m);
  z.c_dx = slot(n);
  z.c_dsv = slot(d);
  z.c_dyc = slot(m);
  z.c_dyd = slot(d);
  const CholEngine::Sizes cz = S->chol->sizes();
  z.L = slot(cz.L);
  z.U = slot(cz.U);
  z.dinv = slot(cz.dinv);
  z.y = slot(cz.y);
  z.ubuf = slot(cz.ubuf);
  z.exch = slot(cz.exch);
  z.stride = at;
  S->cap = cap_;
  S->arena.alloc(static_cast<size_t>(z.stride) * cap_);
  S->flags.alloc(static_cast<size_t>(FL_COUNT) * cap_);
  S->fin.ensure(static_cast<size_t>(dev::FIN_SLOTS) * cap_);
  S->flag_host.ensure(2 * static_cast<size_t>(cap_));
  double* base = S->arena.p;
  S->chol->bind(CholEngine::Storage{base + z.L, base + z.U, base + z.dinv, base + z.y,
                                    base + z.ubuf, base + z.exch, S->flags.p + FL_PIVOT * cap_},
                z.stride, cap_);
  HIPCHK(hipStreamSynchronize(st_));

  for (hykkt_stats& st : st_k_) {
    st.n = n;
    st.m = m;
    st.d = d;
    st.nnz_htil = S->htp.e.nnz();
    st.nnz_hgam = HG.nnz();
    st.nnz_l = pl.nnz_l_stored;
    st.n_supernodes = pl.ns;
    st.n_levels = static_cast<int>(pl.level_ptr.size()) - 1;
    st.max_front = pl.max_front;
    st.factor_flops = pl.flops;
    st.t_symbolic_ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  }
  last_iters_ = last_ref_iters_ = -1;
  sym_ = std::move(S);
}

// ------------------------------------------------------------------ values
// Copy each system's values into its arena slots: a copy kernel over the systems
// from device pointers, or host-to-device copies from host arrays.
void Solver::upload_values(int count)
{
  Sym& S = *sym_;
  const Slots& z = S.z;
  const dev::Batch b{count, z.stride, nullptr};
  const int64_t len[IN_COUNT] = {S.nnz_h, S.d, S.nnz_jc, S.nnz_jd, S.n, S.d, S.m, S.d, S.m};
  bool any_y0 = false;
  std::vector<double> gam(count);
  for (int k = 0; k < count; k++) {
    gam[k] = sys_in_[k].gamma;
    any_y0 = any_y0 || sys_in_[k].v[IN_Y0] != nullptr;
  }
  if (opts.inputs_on_device) {
    static_assert(IN_COUNT == dev::COPY_ARRAYS, "one copy per input array");
    double* dst[IN_COUNT];
    bool zero[IN_COUNT] = {};
    zero[IN_Y0] = any_y0;   // a system without its own start y begins at zero
    std::vector<const double*> src(static_cast<size_t>(IN_COUNT) * count);
    for (int j = 0; j < IN_COUNT; j++) {
      dst[j] = P(z.in[j]);
      for (int k = 0; k < count; k++) src[static_cast<size_t>(k) * IN_COUNT + j] = sys_in_[k].v[j];
    }
    dev::copy_in(dst, len, zero, src.data(), P(z.gam), gam.data(), b, st_, ev_[0]);
  } else {
    HIPCHK(hipEventRecord(ev_[0], st_));
    if (any_y0) dev::fill(P(z.in[IN_Y0]), 0.0, S.m, b, st_);
    for (int k = 0; k < count; k++) {
      double* base = P(static_cast<int64_t>(k) * z.stride);
      for (int j = 0; j < IN_COUNT; j++)
        if (sys_in_[k].v[j] && len[j])
          HIPCHK(hipMemcpyAsync(base + z.in[j], sys_in_[k].v[j], sizeof(double) * len[j],
                                hipMemcpyHostToDevice, st_));
      HIPCHK(hipMemcpyAsync(base + z.gam, &gam[k], sizeof(double), hipMemcpyHostToDevice, st_));
    }
    HIPCHK(hipStreamSynchronize(st_));   // gam is read by the copies
  }
}

// compute_spgemm_hgamma + apply_permutation + add_diag (HykktSolver.cpp:370-395):
// the lower triangle of P*Hg*P^T, each value evaluated from the Ruiz-scaled
// H~ and Jc and written straight to its slot in the factor storage, then the
// diagonal shift.
void Solver::assemble_hgamma(const dev::Batch& b)
{
  Sym& S = *sym_;
  const Slots& z = S.z;
  CholEngine& ch = *S.chol;
  ch.zero_L(b);
  timed(PK_SPGEMM_SCATTER, S.hg_flops, S.hg_bytes, b, [&] {
    dev::spgemm_scatter(ch.n_assembled(), S.ent_src.p, ch.a_dst(), S.hg_dsrc.p, P(z.htil),
                        S.hg_tp.p, S.hg_ta.p, S.hg_tb.p, P(z.jcs), P(z.jcs), P(z.gam), ch.L(), b,
                        st_);
  });
  ch.shift_diag(opts.delta, b);   // add_diag(delta) hook (HykktSolver.cpp:392)
}

// Each candidate factorizes the batch's assembled matrices once (the factor
// is in place, so every run assembles first); the first run, with the default
// shapes, also loads the kernels' code and is not timed.  Patterns whose
// factorization would take more than ~1e13 flops are left at the defaults:
// their trailing updates fill the device whatever the shapes.
void Solver::autotune(const dev::Batch& b)
{
  Sym& S = *sym_;
  CholEngine& ch = *S.chol;
  using T = CholEngine::Tuning;
  tuning_ = hykkt_tuning{};
  const T def;
  tuning_.short_max = def.short_max;
  tuning_.group_max = def.group_max;
  tuning_.pair_min = def.pair_min;
  tuning_.count = b.count;
  if (ch.tuning_pinned()) {
    const T pin = ch.tuning();
    ch.set_tuning(pin, b.count);
    tuning_.short_max = pin.short_max;
    tuning_.group_max = pin.group_max;
    tuning_.pair_min = pin.pair_min;
    return;
  }
  if (ch.plan().flops * b.count > 1e13) {
    ch.set_tuning(def, b.count);
    return;
  }
  const T cand[] = {def,           T{0, 8, 512},   T{1024, 8, 512}, T{128, 4, 512},
                    T{128, 8, 256}, T{128, 8, 2048}, T{128, 1, 512}};
  hipEvent_t e0 = ev_[3], e1 = ev_[4];   // free until the solve phase
  // the tuning runs are neither profiled nor counted in the pass's times
  prof.pause(true);
  HIPCHK(hipEventRecord(ev_[5], st_));
  auto run_one = [&](const T& t) {
    ch.set_tuning(t, b.count);
    assemble_hgamma(b);
    HIPCHK(hipEventRecord(e0, st_));
    ch.factor(opts.pivot_tol, b);
    HIPCHK(hipEventRecord(e1, st_));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    return static_cast<double>(ms);
  };
  run_one(def);   // code loading and first touches
  double best = 0.0;
  int bi = 0;
  for (int i = 0; i < static_cast<int>(sizeof(cand) / sizeof(cand[0])); i++) {
    const double ms = run_one(cand[i]);
    if (i == 0) tuning_.default_ms = ms;
    if (i == 0 || ms < best) {
      best = ms;
      bi = i;
    }
    tuning_.candidates++;
  }
  ch.set_tuning(cand[bi], b.count);
  HIPCHK(hipEventRecord(ev_[6], st_));
  HIPCHK(hipEventSynchronize(ev_[6]));
  HIPCHK(hipEventElapsedTime(&tune_ms_, ev_[5], ev_[6]));
  prof.pause(false);
  tuning_.short_max = cand[bi].short_max;
  tuning_.group_max = cand[bi].group_max;
  tuning_.pair_min = cand[bi].pair_min;
  tuning_.factor_ms = best;
}

// ------------------------------------------------------------------ execute
int Solver::execute()
{
  // HykktSolver.cpp:243-250: a changed Jd emptiness on the file path is an error
  if (file_path_ && !status_ && sym_) {
    if (opts.verbose) std::printf("\n\nERROR: USING HYKKT WITH NEW NONZERO STRUCTURE\n\n");
    return HYKKT_RESIDUAL_FAIL;
  }
  const std::vector<int> rc = run(1, true);
  stats = st_k_[0];
  if (opts.verbose) {
    std::printf("||Ax-b||/||b|| = %32.32g\n\n", stats.resid2);
    std::printf(stats.resid2 < opts.norm_tol ? "Residual test passed\n" : "Residual test failed\n");
  }
  return rc[0];
}

std::vector<int> Solver::execute_batch(int count)
{
  HYKKT_REQUIRE(count >= 1 && count <= cap_, HYKKT_E_ARG, "batch count outside 1 .. capacity");
  for (int k = 0; k < count; k++)
    HYKKT_REQUIRE(sys_in_[k].set, HYKKT_E_STATE,
                  "batch system " + std::to_string(k) + " has no bound values");
  std::vector<int> rc = run(count, false);
  stats = st_k_[0];
  return rc;
}

const hykkt_stats& Solver::stats_of(int k) const
{
  HYKKT_REQUIRE(k >= 0 && k < cap_, HYKKT_E_ARG, "system index beyond the batch capacity");
  return st_k_[k];
}

std::vector<int> Solver::run(int count, bool from_setters)
{
  for (int k = 0; k < 4; k++)
    HYKKT_REQUIRE(blk_[k].set, HYKKT_E_STATE, "a matrix block was not set");
  if (from_setters) {
    auto need = [&](int which, int len, const char* name) {
      HYKKT_REQUIRE(vecs_[which] != nullptr, HYKKT_E_STATE, std::string(name) + " not set");
      HYKKT_REQUIRE(vec_n_[which] == 0 || vec_n_[which] >= len, HYKKT_E_ARG,
                    std::string(name) + " too short");
    };
    need(VEC_RX, blk_[BLK_H].n, "rx");
    need(VEC_RS, blk_[BLK_DS].n, "rs");
    need(VEC_RY, blk_[BLK_JC].n, "ry");
    need(VEC_RYD, blk_[BLK_DS].n, "ryd");
    SystemIn& s0 = sys_in_[0];
    s0.v[IN_H] = blk_[BLK_H].v;
    s0.v[IN_DS] = blk_[BLK_DS].v;
    s0.v[IN_JC] = blk_[BLK_JC].v;
    s0.v[IN_JD] = blk_[BLK_JD].v;
    s0.v[IN_RX] = vecs_[VEC_RX];
    s0.v[IN_RS] = vecs_[VEC_RS];
    s0.v[IN_RY] = vecs_[VEC_RY];
    s0.v[IN_RYD] = vecs_[VEC_RYD];
    s0.v[IN_Y0] = vecs_[VEC_Y];
    s0.gamma = gamma_;
    s0.set = false;   // the batch binding of system 0 is not kept
  }
  const bool fresh = !sym_ || !pattern_matches() || sym_->has_jd != (blk_[BLK_JD].nnz > 0);
  if (fresh) analyze();
  Sym& S = *sym_;
  const Slots& z = S.z;
  const int n = S.n, m = S.m, d = S.d;
  const dev::Batch b{count, z.stride, nullptr};
  tune_ms_ = 0.f;
  upload_values(count);
  bool any_y0 = false;
  for (int k = 0; k < count; k++) any_y0 = any_y0 || sys_in_[k].v[IN_Y0] != nullptr;
  const double* in[IN_COUNT];
  for (int j = 0; j < IN_COUNT; j++) in[j] = P(z.in[j]);

  // ---- compute_spgemm_htil (HykktSolver.cpp:289-337) ----
  if (S.has_jd) {
    dev::row_scale(d, S.jd_rp.p, in[IN_JD], in[IN_DS], in[IN_RYD], in[IN_RS], P(z.jd_vs),
                   P(z.ryd_s), b, st_, S.flag(FL_ZERO_ROW), S.flag(FL_PIVOT));
    timed(PK_SPMV, 2.0 * S.nnz_jd, spmv_bytes(n, d, S.nnz_jd, true, true, false), b, [&] {
      dev::spmv(n, S.jdt_rp.p, S.jdt_ci.p, S.jdt_map.p, in[IN_JD], 1.0, nullptr, P(z.ryd_s), 1.0,
                in[IN_RX], P(z.rx_til), S.jdt_blk.p, S.jdt_nblk, b, st_);
    });
    timed(PK_SPGEMM_VALUES, S.ht_flops, S.ht_bytes, b, [&] {
      dev::spgemm_values(S.htp.e.nnz(), S.ht_dsrc.p, in[IN_H], S.ht_tp.p, S.ht_ta.p, S.ht_tb.p,
                         in[IN_JD], P(z.jd_vs), 1.0, P(z.htil), b, st_);
    });
  } else {
    dev::copy(P(z.rx_til), in[IN_RX], n, b, st_);
    dev::copy(P(z.htil), in[IN_H], S.nnz_h, b, st_);
    dev::fill_i(S.flag(FL_ZERO_ROW), INT_MAX, count, st_);
    dev::fill_i(S.flag(FL_PIVOT), INT_MAX, count, st_);
  }

  // ---- compute_ruiz_scaling (HykktSolver.cpp:340-349; RuizClass.cpp:54-98):
  // each pass applies the last sweep's scale and forms the next one's ----
  if (opts.ruiz_its <= 0) {
    dev::copy(P(z.jcs), in[IN_JC], S.nnz_jc, b, st_);
    dev::copy(P(z.ry_s), in[IN_RY], m, b, st_);
    dev::fill(P(z.max_d), 1.0, n + m, b, st_);
  } else {
    dev::RuizPass r{};
    r.n = n;
    r.m = m;
    r.h_rp = S.ht_rp.p;
    r.h_ci = S.ht_ci.p;
    r.h_v = P(z.htil);
    r.jt_rp = S.jct_rp.p;
    r.jt_ci = S.jct_ci.p;
    r.jt_map = S.jct_map.p;
    r.j_rp = S.jc_rp.p;
    r.j_ci = S.jc_ci.p;
    r.j_src = in[IN_JC];
    r.rhs1 = P(z.rx_til);
    r.rhs2_src = in[IN_RY];
    r.rhs2 = P(z.ry_s);
    r.max_d = P(z.max_d);
    r.zero_row = S.flag(FL_ZERO_ROW);
    double* const scale[2] = {P(z.scale), P(z.scale2)};
    // the passes in between alternate Jc's scaled values between jch_v (free
    // until the factorization is done) and jcs, where the last one leaves them
    double* const jbuf[2] = {P(z.jcs), P(z.jch_v)};
    for (int k = 0; k <= opts.ruiz_its; k++) {
      const bool last = k == opts.ruiz_its;
      r.scale_in = k > 0 ? scale[(k - 1) & 1] : nullptr;
      r.scale_out = last ? nullptr : scale[k & 1];
      r.j_dst = k == 0 ? nullptr : jbuf[last ? 0 : (k & 1)];
      r.first = k == 1;
      dev::ruiz_pass(r, b, st_);
      if (k > 0) {
        r.j_src = r.j_dst;
        r.rhs2_src = r.rhs2;
      }
    }
  }

  // ---- launch shapes of the factorization, once per pattern ----
  if (fresh && opts.autotune) autotune(b);

  // ---- H_gamma straight into the factor storage (HykktSolver.cpp:370-395) ----
  CholEngine& ch = *S.chol;
  ch.set_sweep_share(opts.sweep_share);
  assemble_hgamma(b);

  // ---- compute_hgamma_factorization (HykktSolver.cpp:398-401) ----
  ch.factor(opts.pivot_tol, b, !(fresh && opts.autotune));   // the tuning runs record pivots, too

  // permuted Jc and Jc^T values (apply_permutation, HykktSolver.cpp:386-395).  A
  // system whose factorization met a failing pivot (reported with status 1, as the
  // reference's) gets a zero solution and skips the solve phase, so a batch does
  // not run its CG to the iteration limit on a broken factor.
  dev::AfterFactor af{};
  af.pivot = S.flag(FL_PIVOT);
  af.ok = S.flag(FL_OK);
  af.jcs = P(z.jcs);
  af.jh_map = S.jch_map.p;
  af.jth_map = S.jcth_map.p;
  af.jh_v = P(z.jch_v);
  af.jth_v = P(z.jcth_v);
  af.nnz = S.nnz_jc;
  af.n = n;
  af.m = m;
  af.d = d;
  af.dx = P(z.dx);
  af.dsv = P(z.dsv);
  af.dyc = P(z.dyc);
  af.dyd = P(z.dyd);
  dev::after_factor(af, b, st_, ev_[1]);

  // ---- first pass: the reference's solve (HykktSolver.cpp:404-457) and its
  // check_error (:846-930), with rows 2 and 4 ----
  // CG start y_host, or zero when none is bound (then no start-residual solve)
  const Solution sol{z.dx, z.dsv, z.dyc, z.dyd}, none{-1, -1, -1, -1};
  solve_pass(Pass{z.rxp, z.schur, z.cx}, z.rx_til, z.ry_s, z.in[IN_RS], z.in[IN_RYD], any_y0, sol,
             none, z.e[0], dev::masked(b, S.flag(FL_OK)), b, last_iters_, true);
  std::vector<int> zrow(count), piv(count);
  std::vector<int> rc(count, HYKKT_OK);
  std::vector<double> nb(count);
  auto fin = [&](int k) { return S.fin.p + static_cast<size_t>(k) * dev::FIN_SLOTS; };
  int it_max = 0;
  for (int k = 0; k < count; k++) {
    hykkt_stats& st = st_k_[k];
    const double* h = fin(k) + dev::FIN_RES;
    const CgResult cg = cg_result(fin(k));
    it_max = std::max(it_max, cg.iters);
    nb[k] = h[4] + h[5] + h[6] + h[7];
    st.resid2 = std::sqrt(h[0] + h[1]) / std::sqrt(nb[k]);
    st.resid4 = std::sqrt(h[0] + h[1] + h[2] + h[3]) / std::sqrt(nb[k]);
    st.resid4_first = st.resid4;
    st.refine_steps = 0;
    st.cg_iters = cg.iters;
    st.cg_status = cg.status;
    st.cg_final_norm = cg.final_norm;
    zrow[k] = static_cast<int>(fin(k)[dev::FIN_ZERO_ROW]);
    piv[k] = static_cast<int>(fin(k)[dev::FIN_PIVOT]);
    if (piv[k] == INT_MAX) piv[k] = -1;
    st.pivot = piv[k];
    // matrix_vector_ops.cu:258-264 scales a zero row by 1/sqrt(0) = inf and
    // the solve turns to NaN; here it is an argument error of that system
    if (zrow[k] != INT_MAX) rc[k] = HYKKT_E_ARG;
  }
  last_iters_ = it_max;

  // ---- iterative refinement on the 4x4 block KKT system (an addition: the
  // reference stops after one pass).  The signed residual rows go through the
  // right-hand-side half of formation (r~x = ex + Jd^T (Ds ed + es), then the
  // Ruiz scaling max_d) and the same solve phase with a zero CG start; a
  // correction is kept only if it lowers resid4.  Each system decides for
  // itself, as it would alone; the pass covers the systems still refining. ----
  std::vector<int> act(count), stopped(count, 0);
  int* const act_h = S.flag_host.p;
  int* const keep_h = S.flag_host.p + S.cap;
  const Pass corr{z.e_rxp, z.e_schur, z.e_cx};
  const Solution csol{z.c_dx, z.c_dsv, z.c_dyc, z.c_dyd};
  bool refined = false;
  for (int pass = 0; pass < opts.refine_max; pass++) {
    int nact = 0;
    for (int k = 0; k < count; k++) {
      act[k] = (rc[k] == HYKKT_OK && piv[k] < 0 && !stopped[k] &&
                st_k_[k].resid4 > opts.refine_tol) ? 1 : 0;
      act_h[k] = act[k];
      nact += act[k];
    }
    if (nact == 0) break;
    refined = true;
    dev::Batch ba = b;
    if (nact < count) {   // else every system takes part: no mask
      HIPCHK(hipMemcpyAsync(S.flag(FL_ACT), act_h, sizeof(int) * count, hipMemcpyHostToDevice,
                            st_));
      ba = dev::masked(b, S.flag(FL_ACT));
    }
    const Rows& e = z.e[pass & 1];
    if (S.has_jd) {
      dev::row_scale(d, S.jd_rp.p, in[IN_JD], in[IN_DS], P(e.d), P(e.s), nullptr, P(z.ryd_s), ba,
                     st_);
      timed(PK_SPMV, 2.0 * S.nnz_jd, spmv_bytes(n, d, S.nnz_jd, true, true, false), ba, [&] {
        dev::spmv(n, S.jdt_rp.p, S.jdt_ci.p, S.jdt_map.p, in[IN_JD], 1.0, nullptr, P(z.ryd_s),
                  1.0, P(e.x), P(z.e_rxt), S.jdt_blk.p, S.jdt_nblk, ba, st_);
      });
    } else {
      dev::copy(P(z.e_rxt), P(e.x), n, ba, st_);
    }
    dev::vec_scale(P(z.e_rxt), P(z.max_d), n, ba, st_);
    dev::copy(P(z.e_ysc), P(e.y), m, ba, st_);
    dev::vec_scale(P(z.e_ysc), P(z.max_d) + n, m, ba, st_);
    // the correction's right-hand side is small: its CG usually stops within
    // an iteration or two, so its first look at the live flags comes from
    // the last refinement pass, not the first pass
    solve_pass(corr, z.e_rxt, z.e_ysc, e.s, e.d, false, csol, sol, z.e[(pass + 1) & 1], ba, ba,
               last_ref_iters_, false);
    int rit = 0;
    for (int k = 0; k < count; k++)
      if (act[k]) rit = std::max(rit, cg_result(fin(k)).iters);
    last_ref_iters_ = rit;
    int nkeep = 0;
    for (int k = 0; k < count; k++) {
      keep_h[k] = 0;
      if (!act[k]) continue;
      const double* h = fin(k) + dev::FIN_RES;
      const double c4 = std::sqrt(h[0] + h[1] + h[2] + h[3]) / std::sqrt(nb[k]);
      if (!(c4 < st_k_[k].resid4)) {   // keep the better solution; its rows in e_* are stale
        stopped[k] = 1;
        continue;
      }
      keep_h[k] = 1;
      nkeep++;
      st_k_[k].resid2 = std::sqrt(h[0] + h[1]) / std::sqrt(nb[k]);
      st_k_[k].resid4 = c4;
      st_k_[k].refine_steps++;
    }
    if (nkeep == 0) break;
    if (nkeep < count)
      HIPCHK(hipMemcpyAsync(S.flag(FL_KEEP), keep_h, sizeof(int) * count, hipMemcpyHostToDevice,
                            st_));
    dev::Keep kp{{P(z.c_dx), P(z.c_dsv), P(z.c_dyc), P(z.c_dyd)},
                 {P(z.dx), P(z.dsv), P(z.dyc), P(z.dyd)},
                 {n, d, m, d}};
    dev::keep_where(kp, nkeep < count ? S.flag(FL_KEEP) : nullptr, b, st_);
  }
  if (refined) {
    HIPCHK(hipEventRecord(ev_[4], st_));
    HIPCHK(hipEventSynchronize(ev_[4]));
  }
  prof.collect();
  // the factor is done with: zero its storage for the next execute now, on
  // the factorization's second stream, while the caller reads the results
  S.chol->prezero_L(count);

  float ms[4] = {};
  HIPCHK(hipEventElapsedTime(&ms[0], ev_[0], ev_[refined ? 4 : 3]));
  HIPCHK(hipEventElapsedTime(&ms[1], ev_[0], ev_[1]));
  HIPCHK(hipEventElapsedTime(&ms[2], ev_[1], ev_[2]));
  if (refined) HIPCHK(hipEventElapsedTime(&ms[3], ev_[3], ev_[4]));
  ms[0] -= tune_ms_;   // the autotuning runs sit between ev_[0] and ev_[1]
  ms[1] -= tune_ms_;
  for (int k = 0; k < count; k++) {
    hykkt_stats& st = st_k_[k];
    st.t_solve_ms = ms[0];
    st.t_factor_ms = ms[1];
    st.t_cg_ms = ms[2];
    st.t_refine_ms = ms[3];
    st.n_solves++;
    if (rc[k] != HYKKT_OK) continue;
    if (st.pivot >= 0) rc[k] = HYKKT_RESIDUAL_FAIL;
    else rc[k] = (st.resid2 < opts.norm_tol) ? HYKKT_OK : HYKKT_RESIDUAL_FAIL;
  }
  if (from_setters && zrow[0] != INT_MAX)
    throw Error(HYKKT_E_ARG, zrow[0] < n ? "row " + std::to_string(zrow[0]) +
                                              " of [H~ Jc^T] has no nonzero value (Ruiz scale 1/sqrt(0))"
                                        : "row " + std::to_string(zrow[0] - n) +
                                              " of Jc has no nonzero value (Ruiz scale 1/sqrt(0))");
  return rc;
}

// setup_conjugate_gradient (HykktSolver.cpp:814-843), the Schur CG
// (SchurComplementConjugateGradient.cpp:89-194), recover_solution
// (HykktSolver.cpp:410-457) and the residual rows, for Ruiz-scaled right-hand sides
// rxt (n, natural order) and ysc (m); rs, ryd are the unscaled d-rows used by the
// recovery.  All arguments are arena offsets; the systems of bs take part in the
// solve, those of br in the recovery's and residual's results.
//
// The host looks at the systems after as many iterations as the last pass of the
// kind took (`hint`; below 0: not known), then after each one; or every
// cg_check_every.  The first look that comes no sooner than that pass's end has
// recovery, residual and their results enqueued with it, as if every system stopped
// there, so the usual pass has one host round trip and no iteration that nobody
// needs.  The other looks read the live flags alone, and where that look was too
// early the two run again once every system has stopped (1,000 buses, 13 iterations
// with a look after each: 2158 us a solve, 2472 with both at every look; 1988 with
// the iterations known).
void Solver::solve_pass(const Pass& w, int64_t rxt, int64_t ysc, int64_t rs, int64_t ryd, bool x0,
                        const Solution& out, const Solution& base, const Rows& rows,
                        const dev::Batch& bs, const dev::Batch& br, int hint, bool first)
{
  Sym& S = *sym_;
  const Slots& z = S.z;
  const int n = S.n, m = S.m, d = S.d;
  CholEngine& ch = *S.chol;
  // r^x = r~x + gamma Jc^T ry in the factor's internal order, A^{-1} r^x (kept for
  // the recovery) and the Schur right-hand side Jc A^{-1} r^x - ry
  const double fl = 2.0 * S.nnz_jc;
  timed(PK_SPMV, fl, spmv_bytes(n, m, S.nnz_jc, false, true, false), bs, [&] {
    dev::spmv(n, S.jcth_rp.p, S.jcth_ci.p, nullptr, P(z.jcth_v), 0.0, P(z.gam), P(ysc), 1.0,
              P(rxt), P(w.rxp), S.jcth_blk.p, S.jcth_nblk, bs, st_, nullptr, nullptr, S.phat_d.p,
              ch.sweep_fill(P(z.h0)));
  });
  ch.solve(P(w.rxp), P(z.h0), bs, true);
  timed(PK_SPMV, fl, spmv_bytes(m, n, S.nnz_jc, false, true, false), bs, [&] {
    dev::spmv(m, S.jch_rp.p, S.jch_ci.p, nullptr, P(z.jch_v), 1.0, nullptr, P(z.h0), -1.0,
              P(ysc), P(w.schur), S.jch_blk.p, S.jch_nblk, bs, st_);
  });

  SchurOps ops;
  ops.jh_rp = S.jch_rp.p;
  ops.jh_ci = S.jch_ci.p;
  ops.jh_blk = S.jch_blk.p;
  ops.jh_nblk = S.jch_nblk;
  ops.jh_v = P(z.jch_v);
  ops.jth_rp = S.jcth_rp.p;
  ops.jth_ci = S.jcth_ci.p;
  ops.jth_v = P(z.jcth_v);
  ops.chol = &ch;
  ops.st = st_;
  ops.v = dev::CgVecs{m,       n,       P(w.cx), P(z.cr), P(z.cw),   P(z.cp),    P(z.cs),
                      P(z.t1), P(z.t2), P(z.cq), P(z.cz), P(z.sc),   P(z.part),  P(z.part2),
                      S.jch_nblk};
  ops.f = dev::CgFlags{S.flag(FL_LIVE), S.flag(FL_CG_IT), S.flag(FL_CG_ST)};
  ops.prof = &prof;
  ops.nnz = S.nnz_jc;
  if (x0) dev::copy(P(w.cx), P(z.in[IN_Y0]), m, bs, st_);
  cg_start(ops, P(w.schur), bs, !x0);

  dev::Recover rec{};
  rec.n = n;
  rec.m = m;
  rec.d = d;
  rec.has_jd = S.has_jd ? 1 : 0;
  rec.h0 = P(z.h0);
  rec.z = P(z.cz);
  rec.x = P(w.cx);
  rec.max_d = P(z.max_d);
  rec.ipos = S.ipos_d.p;
  rec.jd_rp = S.jd_rp.p;
  rec.jd_ci = S.jd_ci.p;
  rec.jd_v = P(z.in[IN_JD]);
  rec.ryd = P(ryd);
  rec.ds = P(z.in[IN_DS]);
  rec.rs = P(rs);
  rec.dx = P(out.dx);
  rec.dsv = P(out.dsv);
  rec.dyc = P(out.dyc);
  rec.dyd = P(out.dyd);
  if (base.dx >= 0) {
    rec.base_dx = P(base.dx);
    rec.base_dsv = P(base.dsv);
    rec.base_dyc = P(base.dyc);
    rec.base_dyd = P(base.dyd);
  }
  dev::Residual res{};
  res.n = n;
  res.m = m;
  res.d = d;
  res.has_jd = rec.has_jd;
  res.h_rp = S.h_rp.p;
  res.h_ci = S.h_ci.p;
  res.ct_rp = S.jct_rp.p;
  res.ct_ci = S.jct_ci.p;
  res.ct_map = S.jct_map.p;
  res.dt_rp = S.jdt_rp.p;
  res.dt_ci = S.jdt_ci.p;
  res.dt_map = S.jdt_map.p;
  res.jc_rp = S.jc_rp.p;
  res.jc_ci = S.jc_ci.p;
  res.jd_rp = S.jd_rp.p;
  res.jd_ci = S.jd_ci.p;
  res.h_v = P(z.in[IN_H]);
  res.jc_v = P(z.in[IN_JC]);
  res.jd_v = P(z.in[IN_JD]);
  res.ds = P(z.in[IN_DS]);
  res.rx = P(z.in[IN_RX]);
  res.rs = P(z.in[IN_RS]);
  res.ry = P(z.in[IN_RY]);
  res.ryd = P(z.in[IN_RYD]);
  res.dx = rec.dx;
  res.dsv = rec.dsv;
  res.dyc = rec.dyc;
  res.dyd = rec.dyd;
  res.e_x = P(rows.x);
  res.e_s = P(rows.s);
  res.e_y = P(rows.y);
  res.e_d = P(rows.d);
  res.part = P(z.rpart);
  dev::Finish fin{};
  fin.out = S.fin.p;
  fin.zero_row = S.flag(FL_ZERO_ROW);
  fin.pivot = S.flag(FL_PIVOT);
  fin.sweep_err = ch.solve_error_dev();
  // algorithmic: the recovery's Jd dx; H, Jc twice and Jd twice of the residual
  const double rec_by = spmv_bytes(d, n, S.nnz_jd, false, true, false);
  const double res_fl = 2.0 * (S.nnz_h + 2.0 * S.nnz_jc + 2.0 * S.nnz_jd);
  const double res_by = spmv_bytes(n, n, S.nnz_h, false, true, false) +
                        spmv_bytes(n, m, S.nnz_jc, true, false, false) +
                        spmv_bytes(n, d, S.nnz_jd, true, false, false) +
                        spmv_bytes(m, n, S.nnz_jc, false, true, false) +
                        spmv_bytes(d, n, S.nnz_jd, false, true, false);
  int todo = opts.cg_check_every > 0 ? opts.cg_check_every : std::max(1, hint);
  bool guess = hint >= 0, stopped = false;
  for (;;) {
    cg_iterate(ops, todo, opts.cg_tol, opts.cg_itmax, bs);
    const bool results = stopped || (guess && ops.k >= std::min(hint, opts.cg_itmax));
    if (results) {
      guess = false;
      timed(PK_SPMV, 2.0 * S.nnz_jd, rec_by, bs,
            [&] { dev::recover(rec, bs, st_, first ? ev_[2] : nullptr); });
      timed(PK_SPMV, res_fl, res_by, br, [&] { dev::residual(res, br, st_); });
    }
    dev::finish(fin, results ? &res : nullptr, ops.v, ops.k, opts.cg_tol, opts.cg_itmax, ops.f, br,
                st_, first && results ? ev_[3] : nullptr);
    HIPCHK(hipStreamSynchronize(st_));
    bool live = false, bad = false;
    for (int k = 0; k < br.count; k++) {
      const double* h = S.fin.p + static_cast<size_t>(k) * dev::FIN_SLOTS;
      live = live || h[dev::FIN_LIVE] != 0.0;
      bad = bad || h[dev::FIN_SWEEP_ERR] != 0.0;
    }
    if (bad) {
      ch.clear_solve_error();
      throw Error(HYKKT_E_STATE, "triangular-solve sweep exceeded its wait bound (results invalid)");
    }
    stopped = !live || ops.k >= opts.cg_itmax;
    if (stopped && results) return;
    todo = stopped ? 0 : opts.cg_check_every > 0 ? opts.cg_check_every : 1;
  }
}

void Solver::get_solution(int k, double* dx, double* ds, double* dyc, double* dyd)
{
  HYKKT_REQUIRE(sym_ && st_k_[0].n_solves > 0, HYKKT_E_STATE, "no solution yet");
  HYKKT_REQUIRE(k >= 0 && k < sym_->cap, HYKKT_E_ARG, "system index beyond the batch capacity");
  Sym& S = *sym_;
  const Slots& z = S.z;
  const int64_t o = static_cast<int64_t>(k) * z.stride;
  auto d2h = [&](double* dst, int64_t off, int cnt) {
    if (dst && cnt)
      HIPCHK(hipMemcpy(dst, P(o + off), cnt * sizeof(double), hipMemcpyDeviceToHost));
  };
  d2h(dx, z.dx, S.n);
  d2h(ds, z.dsv, S.d);
  d2h(dyc, z.dyc, S.m);
  d2h(dyd, z.dyd, S.d);
}

void Solver::get_solution_device(int k, const double** dx, const double** ds,
                                 const double** dyc, const double** dyd) const
{
  HYKKT_REQUIRE(sym_ && st_k_[0].n_solves > 0, HYKKT_E_STATE, "no solution yet");
  HYKKT_REQUIRE(k >= 0 && k < sym_->cap, HYKKT_E_ARG, "system index beyond the batch capacity");
  const Slots& z = sym_->z;
  const int64_t o = static_cast<int64_t>(k) * z.stride;
  if (dx) *dx = P(o + z.dx);
  if (ds) *ds = P(o + z.dsv);
  if (dyc) *dyc = P(o + z.dyc);
  if (dyd) *dyd = P(o + z.dyd);
}

void Solver::get_perm(int* perm, int n) const
{
  HYKKT_REQUIRE(sym_, HYKKT_E_STATE, "no analysis yet");
  HYKKT_REQUIRE(n == sym_->n, HYKKT_E_ARG, "wrong permutation length");
  std::memcpy(perm, sym_->perm.data(), sizeof(int) * n);
}

long long Solver::debug_copy(int what, void* out, long long cap)
{
  HYKKT_REQUIRE(sym_, HYKKT_E_STATE, "no analysis yet");
  Sym& S = *sym_;
  const Slots& z = S.z;
  const dev::Batch one{1, z.stride, nullptr};
  HIPCHK(hipStreamSynchronize(st_));
  auto dcopy = [&](const double* src, long long cnt) -> long long {
    HYKKT_REQUIRE(cnt <= cap, HYKKT_E_ARG, "debug_copy: buffer too small");
    if (cnt) HIPCHK(hipMemcpy(out, src, cnt * sizeof(double), hipMemcpyDeviceToHost));
    return cnt;
  };
  auto icopy = [&](const std::vector<int>& v) -> long long {
    HYKKT_REQUIRE(static_cast<long long>(v.size()) <= cap, HYKKT_E_ARG,
                  "debug_copy: buffer too small");
    std::memcpy(out, v.data(), v.size() * sizeof(int));
    return static_cast<long long>(v.size());
  };
  DevBuf<double> tmp;
  switch (what) {
    case 1: return dcopy(P(z.htil), S.htp.e.nnz());
    case 2: return icopy(S.htp.e.rp);
    case 3: return icopy(S.htp.e.ci);
    case 4: return dcopy(P(z.max_d), S.n + S.m);
    case 5: return dcopy(P(z.jcs), S.nnz_jc);
    case 6: return dcopy(P(z.rx_til), S.n);
    case 7: return dcopy(P(z.ry_s), S.m);
    case 8: return icopy(S.hgp.e.rp);
    case 9: return icopy(S.hgp.e.ci);
    case 10: {
      // The assembly of the last execute, run again into the factor storage
      // (the factor itself is recomputed by every execute), and read back
      // from there through the assembly map: entry a_src[e] of P*Hg*P^T is
      // at L[a_dst[e]]; upper-triangle positions are NaN.
      const long long nz = S.hgp_pat.nnz();
      HYKKT_REQUIRE(nz <= cap, HYKKT_E_ARG, "debug_copy: buffer too small");
      CholEngine& ch = *S.chol;
      const int na = ch.n_assembled();
      tmp.alloc(std::max(1, na));
      assemble_hgamma(one);
      dev::gather64(tmp.p, ch.L(), ch.a_dst(), na, st_);
      std::vector<double> got(std::max(1, na));
      HIPCHK(hipMemcpyAsync(got.data(), tmp.p, sizeof(double) * na, hipMemcpyDeviceToHost, st_));
      HIPCHK(hipStreamSynchronize(st_));
      double* o = static_cast<double*>(out);
      std::fill(o, o + nz, std::nan(""));
      const std::vector<int>& src = ch.plan().a_src;
      for (int e = 0; e < na; e++) o[src[e]] = got[e];
      return nz;
    }
    case 11:   // H~ before Ruiz, recomputed from the current inputs
      tmp.alloc(std::max(1, S.htp.e.nnz()));
      if (S.has_jd)
        dev::spgemm_values(S.htp.e.nnz(), S.ht_dsrc.p, P(z.in[IN_H]), S.ht_tp.p, S.ht_ta.p,
                           S.ht_tb.p, P(z.in[IN_JD]), P(z.jd_vs), 1.0, tmp.p, one, st_);
      else
        dev::copy(tmp.p, P(z.in[IN_H]), S.nnz_h, one, st_);
      HIPCHK(hipStreamSynchronize(st_));
      return dcopy(tmp.p, S.htp.e.nnz());
    case 12: {  // r^x in natural order
      std::vector<double> a(S.n), b(S.n);
      HIPCHK(hipMemcpy(a.data(), P(z.rxp), S.n * sizeof(double), hipMemcpyDeviceToHost));
      for (int k = 0; k < S.n; k++) b[S.phat[k]] = a[k];
      HYKKT_REQUIRE(S.n <= cap, HYKKT_E_ARG, "debug_copy: buffer too small");
      std::memcpy(out, b.data(), S.n * sizeof(double));
      return S.n;
    }
    case 13: return dcopy(P(z.schur), S.m);
    case 14: return dcopy(P(z.cx), S.m);
    case 15: return icopy(S.hgp_pat.rp);
    case 16: return icopy(S.hgp_pat.ci);
    case 17: return icopy(S.hgp_map);
    case 18: return icopy(S.jcp_pat.ci);
    case 19: return icopy(S.jcp_map);
    case 20: return icopy(S.jctp_pat.rp);
    case 21: return icopy(S.jctp_pat.ci);
    case 22: return icopy(S.jctp_map);
    case 23: {
      DevBuf<int> words;
      words.alloc(2);
      return icopy({S.chol->second_stream_overlaps() ? 1 : 0,
                    dev::streams_overlap(st_, st_, words.p) ? 1 : 0});
    }
    default: throw Error(HYKKT_E_ARG, "debug_copy: unknown selector");
  }
}

}  // namespace hykkt
