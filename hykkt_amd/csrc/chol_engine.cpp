// chol_engine.cpp -- host orchestration of the device multifrontal Cholesky.
//
// Numeric factorization, per tree level (leaves first):
//   narrow supernodes (front_panel): children added, diagonal block, TRSM in one
//   launch; the others:
//   extend-add of the children's update matrices into the panels,
//   blocked right-looking panel factorization in 128-column steps
//     (factor + invert the diagonal block; TRSM of the rows below with the
//      inverted block on the matrix cores -- for 128-wide blocks by blocked
//      substitution with the inverses of the 16x16 diagonal blocks; MFMA
//      update of the panel's trailing columns),
//   U = -L21 L21^T on the matrix cores plus the children's update matrices;
// after the last level the inverses of groups of columns, for the solves.
// Solves: one forward and one backward sweep over the whole tree.
#include <algorithm>
#include <queue>
#include <climits>
#include <cstdio>
#include <cstdlib>

#include "device.hpp"

namespace hykkt {

namespace {
constexpr int NB = 128;   // panel step, MFMA tile edge, solve block
constexpr int SR = 32;    // rows of a short tile
constexpr int TR = 64;    // rows of a short tile of the blocked TRSM
constexpr int GMAX = 8;   // most steps one grouped trailing update can cover
constexpr int XCD_BLOCK = 1024;   // rows and columns of a block of tiles of one XCD
constexpr int U_SMALL_NC = 512;   // update matrices of at most so many columns take 64 x 64 tiles
static_assert(CholOptions{}.index_narrow == dev::FRONT_NC, "front_panel's index has the columns' rows");
inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// Tiles `from` .. of a launch's list (by supernode, column, row) in the order that keeps
// their operands in an XCD's own L2: workgroup i runs on XCD i % 8, so a block of `side`
// x `side` tiles, which share their rows of A and B, goes to one XCD, the one with the
// shortest queue.  Blocks of 1024 x 1024 entries: trailing updates and update matrices
// at 40,000 buses 519 -> 509 ms, 10,000 9.67 -> 9.60, eight of 5,000 9.84 -> 9.70 (512:
// 510, 9.77, 9.69; 2048: 510, 9.62, 9.76).
void xcd_order(std::vector<int>& sn, std::vector<int>& tr, std::vector<int>& tc, size_t from,
               int side)
{
  constexpr size_t XCDS = 8, LEAST = 512;   // fewer tiles: all in flight at once, in any order
  const size_t n = sn.size() - from;
  if (n < LEAST) return;
  const std::vector<int> s(sn.begin() + from, sn.end()), r(tr.begin() + from, tr.end()),
      c(tc.begin() + from, tc.end());
  std::vector<int> q[XCDS], at, idx;
  for (auto& v : q) v.reserve(n / XCDS + side * side);
  for (size_t i = 0; i < n;) {
    // a stripe of `side` tile columns, counted out by blocks of rows
    size_t j = i;
    int hi = 0;
    for (; j < n && s[j] == s[i] && c[j] / side == c[i] / side; j++) hi = std::max(hi, r[j] / side);
    at.assign(hi + 2, 0);
    idx.resize(j - i);
    for (size_t k = i; k < j; k++) at[r[k] / side + 1]++;
    for (int k = 0; k <= hi; k++) at[k + 1] += at[k];
    std::vector<int> put(at.begin(), at.end() - 1);
    for (size_t k = i; k < j; k++) idx[put[r[k] / side]++] = static_cast<int>(k);
    for (int k = 0; k <= hi; k++) {
      auto& to = *std::min_element(std::begin(q), std::end(q), [](const auto& x, const auto& y) {
        return x.size() < y.size();
      });
      to.insert(to.end(), idx.begin() + at[k], idx.begin() + at[k + 1]);
    }
    i = j;
  }
  // even lengths, the first n % 8 one longer: the tiles past them fill the short queues
  auto len = [&](size_t x) { return n / XCDS + (x < n % XCDS ? 1 : 0); };
  std::vector<int> spare;
  for (size_t x = 0; x < XCDS; x++)
    for (; q[x].size() > len(x); q[x].pop_back()) spare.push_back(q[x].back());
  for (size_t x = 0; x < XCDS; x++)
    for (; q[x].size() < len(x); spare.pop_back()) q[x].push_back(spare.back());
  for (size_t i = 0; i < n; i++) {
    const int k = q[i % XCDS][i / XCDS];
    sn[from + i] = s[k];
    tr[from + i] = r[k];
    tc[from + i] = c[k];
  }
}
}  // namespace

CholEngine::CholEngine(const Pattern& a, const CholOptions& opt, hipStream_t st) : st_(st)
{
  pick_second_stream();
  // the two streams' events order work on this device only: a device-scope
  // release, no system-scope cache writeback when they are recorded
  HIPCHK(hipEventCreateWithFlags(&ev_main_, hipEventDisableTiming | hipEventReleaseToDevice));
  HIPCHK(hipEventCreateWithFlags(&ev_rest_, hipEventDisableTiming | hipEventReleaseToDevice));
  HIPCHK(hipEventCreateWithFlags(&ev_zero_, hipEventDisableTiming | hipEventReleaseToDevice));
  pl_ = chol_analyze(a, opt);
  if (const char* pm = std::getenv("HYKKT_PAIR_MIN")) {
    tun_.pair_min = std::max(1, std::atoi(pm));
    pinned_ = true;
  }
  if (const char* gm = std::getenv("HYKKT_GROUP_MAX")) {
    tun_.group_max = std::clamp(std::atoi(gm), 1, GMAX);
    pinned_ = true;
  }
  {
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    HIPCHK(hipDeviceGetAttribute(&n_cu_, hipDeviceAttributeMultiprocessorCount, dev));
    n_cu_ = std::max(n_cu_, 1);
  }
  auto upi = [](DevBuf<int>& b, const std::vector<int>& v) {
    if (v.empty()) b.upload(std::vector<int>{0});
    else b.upload(v);
  };
  upi(sn_first_, pl_.sn_first);
  upi(rows_ptr_, pl_.rows_ptr);
  upi(rows_, pl_.rows);
  upi(rel_, pl_.rel);
  l_off_.upload(pl_.l_off);
  u_off_.upload(pl_.u_off);
  upi(a_src_, pl_.a_src);
  a_dst_.upload(pl_.a_dst.empty() ? std::vector<int64_t>{0} : pl_.a_dst);
  std::vector<int64_t> dpos(std::max(pl_.n, 1)), uvo(pl_.ns + 1, 0), dvo(pl_.ns + 1, 0);
  for (int s = 0; s < pl_.ns; s++) {
    int f = pl_.nc(s) + pl_.nr(s);
    for (int j = pl_.sn_first[s]; j < pl_.sn_first[s + 1]; j++) {
      int64_t lj = j - pl_.sn_first[s];
      dpos[j] = pl_.l_off[s] + lj * f + lj;
    }
    uvo[s + 1] = uvo[s] + pl_.nr(s);
    dvo[s + 1] = dvo[s] + dev::inv_size(pl_.nc(s));
  }
  diag_pos_.upload(dpos);
  uvec_off_.upload(uvo);
  dinv_off_.upload(dvo);
  n_ubuf_ = uvo[pl_.ns];
  n_dinv_ = dvo[pl_.ns];
  cd_.n = pl_.n;
  cd_.ns = pl_.ns;
  cd_.sn_first = sn_first_.p;
  cd_.rows_ptr = rows_ptr_.p;
  cd_.rows = rows_.p;
  cd_.rel = rel_.p;
  cd_.l_off = l_off_.p;
  cd_.u_off = u_off_.p;
  cd_.dinv_off = dinv_off_.p;
  build_fronts();
  build_tasks();
  build_solve();
}

// The look-ahead needs its stream on another hardware queue than the solver's.
// The runtime spreads streams over a few queues (4 by default) and, once all
// are in use, may give both of a solver's streams the same one, which runs
// their kernels one after the other: a 5,000-bus factorization took 4.37 ms
// there, 3.36 on two queues.  So candidates are tried until one's kernel runs
// while the solver's stream is busy; the rejected ones are kept until then
// (their queue stays counted as used), at most as many as there are queues by
// default.  Streams of default priority, like the solver's.
void CholEngine::pick_second_stream()
{
  constexpr int TRIES = 4;
  DevBuf<int> words;
  words.alloc(2);
  std::vector<hipStream_t> rejected;
  for (int t = 0; t < TRIES; t++) {
    HIPCHK(hipStreamCreate(&st2_));
    overlap_ = dev::streams_overlap(st_, st2_, words.p);
    if (overlap_ || t + 1 == TRIES) break;
    rejected.push_back(st2_);
    st2_ = nullptr;
  }
  for (hipStream_t s : rejected) (void)hipStreamDestroy(s);
}

CholEngine::Sizes CholEngine::sizes() const
{
  auto at_least1 = [](int64_t v) { return std::max<int64_t>(v, 1); };
  return Sizes{at_least1(pl_.l_off[pl_.ns]), at_least1(pl_.u_off[pl_.ns]), at_least1(n_dinv_),
               at_least1(pl_.n), at_least1(n_ubuf_), at_least1(n_exch_)};
}

void CholEngine::set_tuning(const Tuning& t, int count)
{
  HIPCHK(hipStreamSynchronize(st_));   // the task lists of running launches are replaced
  tun_ = t;
  tcount_ = std::max(count, 1);
  build_tasks();
}

void CholEngine::bind(const Storage& s, int64_t vs, int cap)
{
  quiesce();   // a prezero_L of the previous storage may be in flight
  clean_ = 0;
  cd_.L = s.L;
  cd_.U = s.U;
  cd_.dinv = s.dinv;
  cd_.pivot = s.pivot;
  ybuf_ = s.y;
  sd_.ubuf = s.ubuf;
  sd_.exch = s.exch;
  vs_ = vs;
  cap_ = cap;
  // only the lower triangles of the inverses are ever written
  dev::fill(cd_.dinv, 0.0, n_dinv_, dev::Batch{cap, vs, nullptr}, st_);
}

void CholEngine::own(int cap)
{
  const Sizes z = sizes();
  auto al = [](int64_t v) { return (v + 31) / 32 * 32; };   // 256-byte slots
  const int64_t vs = al(z.L) + al(z.U) + al(z.dinv) + al(z.y) + al(z.ubuf) + al(z.exch);
  own_.alloc(static_cast<size_t>(vs) * cap);
  own_piv_.alloc(static_cast<size_t>(cap));
  double* p = own_.p;
  Storage s{};
  s.L = p;
  p += al(z.L);
  s.U = p;
  p += al(z.U);
  s.dinv = p;
  p += al(z.dinv);
  s.y = p;
  p += al(z.y);
  s.ubuf = p;
  p += al(z.ubuf);
  s.exch = p;
  s.pivot = own_piv_.p;
  bind(s, vs, cap);
}

CholEngine::~CholEngine()
{
  if (st2_) quiesce();
  if (ev_main_) (void)hipEventDestroy(ev_main_);
  if (ev_rest_) (void)hipEventDestroy(ev_rest_);
  if (ev_zero_) (void)hipEventDestroy(ev_zero_);
  if (st2_) (void)hipStreamDestroy(st2_);
}

// The supernodes' records.
void CholEngine::build_fronts()
{
  const int ns = pl_.ns;
  std::vector<dev::ChildRec> rec(std::max<size_t>(pl_.child_list.size(), 1));
  for (size_t t = 0; t < pl_.child_list.size(); t++) {
    const int ch = pl_.child_list[t];
    rec[t] = dev::ChildRec{pl_.u_off[ch], pl_.nr(ch), 0};
  }
  std::vector<dev::SnRec> sr(std::max(ns, 1));
  int64_t dinv = 0;
  for (int s = 0; s < ns; s++) {
    const int nc = pl_.nc(s);
    const int nch = pl_.pulls[s] ? pl_.child_ptr[s + 1] - pl_.child_ptr[s] : 0;
    sr[s] = dev::SnRec{pl_.sn_first[s], nc, pl_.nr(s), pl_.child_ptr[s], nch, pl_.inv_rows[s],
                       {0, 0}, pl_.l_off[s], dinv, pl_.u_off[s], pl_.inv_off[s]};
    dinv += dev::inv_size(nc);
  }
  child_rec_.upload(rec);
  sn_rec_.upload(sr);
  if (pl_.inv.empty()) inv_.upload(std::vector<int>{-1});
  else inv_.upload(pl_.inv);
  cd_.child_rec = child_rec_.p;
  cd_.sn_rec = sn_rec_.p;
  cd_.inv = inv_.p;
}

void CholEngine::build_tasks()
{
  // Launch shapes (see Tuning), counted over the tcount_ systems a launch
  // covers: a step whose TRSM has at most short_max tiles of 128 rows runs
  // its TRSM in 64-row tiles and its next-column update in 32-row ones (more
  // workgroups, each with less of the work, for launches on the critical
  // path); up to group_max consecutive steps share one trailing update with
  // K = G * NB (each C tile read and written once for the group) while that
  // update has at least pair_min * G^2 / 4 tiles of 128 x 128 beyond the G
  // block columns next in line (a group's inner steps update their next
  // block column with K up to (G-1) NB on the critical path, which only a big
  // trailing update repays).
  const int64_t tc = std::max(tcount_, 1);
  const int pair_min = std::max(1, tun_.pair_min);
  const int gmax = std::clamp(tun_.group_max, 1, GMAX);
  const int nlev = static_cast<int>(pl_.level_ptr.size()) - 1;
  lv_.assign(nlev, Level{});
  inv_grp_ = Launch{};
  std::vector<int> eap, eacol, eacptr{0}, eacc, eaccol;
  std::vector<int> potrf, trsm_sn, trsm_tr, upd_sn, upd_tr, upd_tc;
  std::vector<int> syrk_sn, syrk_tr, syrk_tc, grp_sn, grp_ix;
  std::vector<int> fp_sn, fp_tile;
  auto narrow = [&](int s) { return pl_.nc(s) <= dev::FRONT_NC; };
  struct Contrib {
    int t, c, r2;
  };
  std::vector<Contrib> con;
  for (int l = 0; l < nlev; l++) {
    Level& L = lv_[l];
    const int b0 = pl_.level_ptr[l], b1 = pl_.level_ptr[l + 1];
    // part 0: panels whose kernels do not add the children themselves; 1: update
    // matrices of the supernodes without an index of their children's rows
    for (int part = 0; part < 2; part++) {
      Launch& la = part == 0 ? L.ea_panel : L.ea_u;
      la.off = static_cast<int>(eap.size());
      for (int q = b0; q < b1; q++) {
        const int p = pl_.level_sn[q], ncp = pl_.nc(p);
        if (pl_.pulls[p] && (part == 1 || narrow(p))) continue;
        con.clear();
        for (int t = pl_.child_ptr[p]; t < pl_.child_ptr[p + 1]; t++) {
          const int c = pl_.child_list[t];
          for (int k = pl_.rows_ptr[c]; k < pl_.rows_ptr[c + 1]; k++) {
            int col = pl_.rel[k];
            if ((col < ncp) == (part == 0)) con.push_back({col, c, k - pl_.rows_ptr[c]});
          }
        }
        std::stable_sort(con.begin(), con.end(),
                         [](const Contrib& x, const Contrib& y) { return x.t < y.t; });
        for (size_t i = 0; i < con.size();) {
          size_t j = i;
          while (j < con.size() && con[j].t == con[i].t) {
            eacc.push_back(con[j].c);
            eaccol.push_back(con[j].r2);
            const double e = pl_.nr(con[j].c) - con[j].r2;   // entries of that U column
            la.flops += e;
            la.bytes += 24.0 * e;   // read the child entry, read + write the parent's
            j++;
          }
          eap.push_back(p);
          eacol.push_back(con[i].t);
          eacptr.push_back(static_cast<int>(eacc.size()));
          i = j;
        }
      }
      la.cnt = static_cast<int>(eap.size()) - la.off;
    }
    int nsteps = 0;
    for (int q = b0; q < b1; q++)
      if (!narrow(pl_.level_sn[q]))
        nsteps = std::max(nsteps, cdiv(pl_.nc(pl_.level_sn[q]), NB));
    // narrow supernodes: one launch for the panel (its flops as a diagonal block's
    // and a TRSM's; the children's entries and the panel read, the panel written)
    L.front.off = static_cast<int>(fp_sn.size());
    for (int q = b0; q < b1; q++) {
      const int s = pl_.level_sn[q];
      if (!narrow(s)) continue;
      const double nc = pl_.nc(s), nr = pl_.nr(s);
      L.front.flops += nc * nc * nc / 3 + nc * nc / 2 + nc / 6 + nr * nc * nc;
      L.front.bytes += 16.0 * (nc * (nc + 1) / 2 + nr * nc);
      for (int t = 0; t < std::max(1, cdiv(pl_.nr(s), NB)); t++) {
        fp_sn.push_back(s);
        fp_tile.push_back(t);
      }
    }
    L.front.cnt = static_cast<int>(fp_sn.size()) - L.front.off;
    L.potrf.resize(nsteps);
    L.trsm.resize(nsteps);
    L.upd_next.resize(nsteps);
    L.upd_rest.resize(nsteps);
    // Groups: steps a .. a+G-1 defer their blocks' updates of the columns
    // after block a+G-1 and apply them together at the group's last step, K =
    // G NB, while that update is big (its tiles beyond the next G block
    // columns).  Step a+i of a group first updates block column a+i+1 by
    // blocks a .. a+i (K = (i+1) NB: the same tiles as a single step's next-
    // column update).  Single steps (G = 1) update after their own block.
    L.gpos.assign(nsteps, 0);
    L.gsize.assign(nsteps, 1);
    L.upd_whole.assign(nsteps, 0);
    for (int j = 0; j < nsteps;) {
      int G = 1;
      for (int g = std::min(gmax, nsteps - j); g >= 2 && G == 1; g--) {
        int64_t rest = 0;
        for (int q = b0; q < b1; q++) {
          const int s = pl_.level_sn[q];
          const int nc = pl_.nc(s), f = nc + pl_.nr(s), k0 = j * NB;
          if (k0 >= nc || narrow(s)) continue;
          const int cs = k0 + std::min(g * NB, nc - k0);
          const int rt = cdiv(f - cs, NB), ct = cdiv(nc - cs, NB);
          for (int tc = g; tc < ct; tc++) rest += rt - tc;
        }
        if (rest * tc >= static_cast<int64_t>(pair_min) * g * g / 4) G = g;
      }
      for (int i = 0; i < G; i++) {
        L.gpos[j + i] = i;
        L.gsize[j + i] = G;
      }
      j += G;
    }
    for (int j = 0; j < nsteps; j++) {
      const int gi = L.gpos[j], G = L.gsize[j];
      const bool last = gi == G - 1;   // the group's update of the columns after it
      L.potrf[j].off = static_cast<int>(potrf.size());
      L.trsm[j].off = static_cast<int>(trsm_sn.size());
      int full_tiles = 0, widest = 0;
      int64_t upd_tiles = 0;   // of 128 x 128
      for (int q = b0; q < b1; q++) {
        const int s = pl_.level_sn[q];
        const int nc = pl_.nc(s), f = nc + pl_.nr(s), k0 = j * NB;
        if (k0 >= nc || narrow(s)) continue;
        const int rt = cdiv(f - (k0 + std::min(NB, nc - k0)), NB);
        const int ct = cdiv(nc - (k0 + std::min(NB, nc - k0)), NB);
        full_tiles += rt;
        upd_tiles += static_cast<int64_t>(ct) * rt - static_cast<int64_t>(ct) * (ct - 1) / 2;
        widest = std::max(widest, std::min(NB, nc - k0));
      }
      const bool shrt = full_tiles * tc <= tun_.short_max;
      const int rows_unit = shrt ? (widest > 64 ? TR : SR) : NB;
      L.trsm[j].short_rows = shrt;
      // A step whose whole update is at most a tile of 128 x 128 per four compute units
      // takes it in one launch on the main stream: beside the diagonal block the rest
      // costs an event on each stream, 11 us a step, more than this update's own time
      // (1,000 buses: 1222 -> 1176 us a solve, 500 1125 -> 1098, 5,000 3738 -> 3707; up
      // to one tile per compute unit 5,000 takes 3797).  32-row tiles up to one per
      // eight (64 x 64 tiles instead: 1185, 1113).
      const bool whole = G == 1 && upd_tiles * tc <= n_cu_ / 4;
      L.upd_whole[j] = whole;
      const bool ushrt = whole ? upd_tiles * tc <= n_cu_ / 8 : shrt && !(last && G > 1);
      L.upd_next[j].short_rows = ushrt;
      for (int q = b0; q < b1; q++) {
        const int s = pl_.level_sn[q];
        const int nc = pl_.nc(s), f = nc + pl_.nr(s);
        const int k0 = j * NB;
        if (k0 >= nc || narrow(s)) continue;
        const int b = std::min(NB, nc - k0);
        potrf.push_back(s);
        L.potrf[j].maxb = std::max(L.potrf[j].maxb, b);
        // Algorithmic (LAPACK) counts: POTRF b^3/3, TRSM r*b^2 for the r rows
        // below the block, and the lower-trapezoid rank-b update of the c
        // trailing panel columns; bytes read each operand and write each
        // result once.
        const double db = b, r = f - (k0 + b), cc = nc - (k0 + b);
        const double tri = db * (db + 1) / 2, pairs = cc * r - cc * (cc - 1) / 2;
        L.potrf[j].flops += db * db * db / 3 + db * db / 2 + db / 6;
        L.potrf[j].bytes += 16.0 * tri;
        L.trsm[j].flops += r * db * db;
        L.trsm[j].bytes += 8.0 * (2 * r * db + tri);
        // the update, unless whole, splits into the next block column (tile column 0) and
        // the rest, so the next step can start before the rest is done.  In a
        // group, an inner step updates the next block column by the group's
        // blocks so far (K = kw) and the last step the columns after the group
        // by all its blocks: the next G block columns, then the rest
        const int ka = k0 - gi * NB;   // the group's first column
        if (last && G > 1) {
          const int kw = std::min(G * NB, nc - ka);
          const double dk = kw, r2 = f - (ka + kw), c2 = nc - (ka + kw);
          const double p2 = c2 * r2 - c2 * (c2 - 1) / 2;
          const double cn = std::min<double>(G * NB, c2);
          const double pn = cn * r2 - cn * (cn - 1) / 2;
          L.upd_next[j].flops += 2.0 * dk * pn;
          L.upd_next[j].bytes += 8.0 * (r2 * dk + 2 * pn);
          L.upd_rest[j].flops += 2.0 * dk * (p2 - pn);
          L.upd_rest[j].bytes += 8.0 * 2 * (p2 - pn);
        } else {
          const double dk = std::min((gi + 1) * NB, nc - ka);
          const double cn = std::min<double>(NB, cc);
          const double pn = cn * r - cn * (cn - 1) / 2;
          L.upd_next[j].flops += 2.0 * dk * pn;
          L.upd_next[j].bytes += 8.0 * (r * dk + 2 * pn);
          if (whole) {
            L.upd_next[j].flops += 2.0 * db * (pairs - pn);
            L.upd_next[j].bytes += 8.0 * 2 * (pairs - pn);
          } else if (G == 1) {
            L.upd_rest[j].flops += 2.0 * db * (pairs - pn);
            L.upd_rest[j].bytes += 8.0 * 2 * (pairs - pn);
          }
        }
        for (int t = 0; t < cdiv(f - (k0 + b), rows_unit); t++) {
          trsm_sn.push_back(s);
          trsm_tr.push_back(t);
        }
      }
      L.potrf[j].cnt = static_cast<int>(potrf.size()) - L.potrf[j].off;
      L.trsm[j].cnt = static_cast<int>(trsm_sn.size()) - L.trsm[j].off;
      for (int part = 0; part < 2; part++) {
        Launch& la = part == 0 ? L.upd_next[j] : L.upd_rest[j];
        la.off = static_cast<int>(upd_sn.size());
        for (int q = b0; q < b1; q++) {
          const int s = pl_.level_sn[q];
          const int nc = pl_.nc(s), f = nc + pl_.nr(s), k0 = j * NB;
          if (k0 >= nc || narrow(s)) continue;
          if (G > 1 && !last && part == 1) continue;   // deferred to the group's update
          if (G > 1 && last) {
            // columns after the group's G blocks, K = all of them: the next G
            // block columns (part 0), then the rest (part 1)
            const int ka = k0 - gi * NB, cs = ka + std::min(G * NB, nc - ka);
            const int rtiles = cdiv(f - cs, NB), ctiles = cdiv(nc - cs, NB);
            for (int tc = part == 0 ? 0 : G; tc < (part == 0 ? std::min(G, ctiles) : ctiles); tc++)
              for (int tr = tc; tr < rtiles; tr++) {
                upd_sn.push_back(s);
                upd_tr.push_back(tr);
                upd_tc.push_back(tc);
              }
            continue;
          }
          const int b = std::min(NB, nc - k0);
          const int ctiles = cdiv(nc - (k0 + b), NB);
          const int tc0 = part == 0 ? 0 : whole ? ctiles : 1;
          const int tc1 = part == 0 && !whole ? std::min(1, ctiles) : ctiles;
          const int unit = part == 0 && ushrt ? SR : NB;   // 32-row tiles
          for (int tc = tc0; tc < tc1; tc++)
            for (int tr = tc * (NB / unit); tr < cdiv(f - (k0 + b), unit); tr++) {
              upd_sn.push_back(s);
              upd_tr.push_back(tr);
              upd_tc.push_back(tc);
            }
        }
        la.cnt = static_cast<int>(upd_sn.size()) - la.off;
        if (part == 1) xcd_order(upd_sn, upd_tr, upd_tc, la.off, XCD_BLOCK / NB);
      }
    }
    // update matrices: tiles of 64 x 64, whose children's entries have four waves a
    // SIMD in flight, unless K is long enough for the operand loads that a 128 x 128
    // tile saves (10,000 buses, K = 404: 424 us against 510; K = 1,468: 1558 against
    // 1512; levels of at most 32 columns: 14-250 us against 27-530)
    L.small_u = true;
    for (int q = b0; q < b1; q++)
      if (pl_.nc(pl_.level_sn[q]) > U_SMALL_NC) L.small_u = false;
    const int ut = L.small_u ? NB / 2 : NB;
    L.syrk.off = static_cast<int>(syrk_sn.size());
    for (int q = b0; q < b1; q++) {
      const int s = pl_.level_sn[q], nt = cdiv(pl_.nr(s), ut);
      const double nr = pl_.nr(s), nc = pl_.nc(s), pairs = nr * (nr + 1) / 2;
      L.syrk.flops += 2.0 * nc * pairs;
      L.syrk.bytes += 8.0 * (nr * nc + pairs);
      for (int t = pl_.child_ptr[s]; pl_.pulls[s] && t < pl_.child_ptr[s + 1]; t++) {
        const int ch = pl_.child_list[t];
        double below = 0;   // the child's rows below s's columns
        for (int k = pl_.rows_ptr[ch]; k < pl_.rows_ptr[ch + 1]; k++) below += pl_.rel[k] >= pl_.nc(s);
        L.syrk.flops += below * (below + 1) / 2;
        L.syrk.bytes += 8.0 * below * (below + 1) / 2;
      }
      for (int tc = 0; tc < nt; tc++)
        for (int tr = tc; tr < nt; tr++) {
          syrk_sn.push_back(s);
          syrk_tr.push_back(tr);
          syrk_tc.push_back(tc);
        }
    }
    L.syrk.cnt = static_cast<int>(syrk_sn.size()) - L.syrk.off;
    xcd_order(syrk_sn, syrk_tr, syrk_tc, L.syrk.off, XCD_BLOCK / ut);
    // the groups' inverses, the longest strips of each first (whole from the 16 x 16
    // ones: (n^3 - 256 n)/3 flops, the triangle read and written).  A block of at most
    // 64 columns that its factorization inverted stays as it is.
    for (int q = b0; q < b1; q++) {
      const int s = pl_.level_sn[q], nc = pl_.nc(s);
      if (narrow(s) || (nc <= 64 && L.potrf[0].maxb <= 64)) continue;
      for (int g0 = 0; g0 < nc; g0 += dev::INV_GROUP) {
        const int n = std::min(dev::INV_GROUP, nc - g0);
        for (int k = 0; k < cdiv(n, 16) - 1; k++) {
          grp_sn.push_back(s);
          grp_ix.push_back(g0 / dev::INV_GROUP * 32 + k);
        }
        const double dn = n;
        inv_grp_.flops += (dn * dn * dn - 256 * dn) / 3;
        inv_grp_.bytes += 16.0 * (dn * dn - 16 * dn) / 2;
      }
    }
  }
  inv_grp_.cnt = static_cast<int>(grp_sn.size());
  auto up = [](DevBuf<int>& b, std::vector<int>& v) {
    if (v.empty()) v.push_back(0);
    b.upload(v);
  };
  up(t_ea_p_, eap);
  up(t_ea_col_, eacol);
  up(t_ea_cptr_, eacptr);
  up(t_ea_cc_, eacc);
  up(t_ea_ccol_, eaccol);
  up(t_fp_sn_, fp_sn);
  up(t_fp_tile_, fp_tile);
  up(t_potrf_, potrf);
  up(t_trsm_sn_, trsm_sn);
  up(t_trsm_tr_, trsm_tr);
  up(t_upd_sn_, upd_sn);
  up(t_upd_tr_, upd_tr);
  up(t_upd_tc_, upd_tc);
  up(t_syrk_sn_, syrk_sn);
  up(t_syrk_tr_, syrk_tr);
  up(t_syrk_tc_, syrk_tc);
  up(t_grp_sn_, grp_sn);
  up(t_grp_ix_, grp_ix);
}

void CholEngine::build_solve()
{
  const int ns = pl_.ns;
  // top of the tree: supernodes wider than FOREST_NC columns or with fronts
  // taller than FOREST_F rows, and all their ancestors; the rest is a forest
  // closed under descendants
  std::vector<char> top(ns, 0);
  for (int s = 0; s < ns; s++)
    if (pl_.nc(s) > dev::FOREST_NC || pl_.nc(s) + pl_.nr(s) > dev::FOREST_F) top[s] = 1;
  for (int s = 0; s < ns; s++)
    if (top[s])
      for (int p = pl_.sn_parent[s]; p >= 0 && !top[p]; p = pl_.sn_parent[p]) top[p] = 1;
  std::vector<int> fwd_top, bwd_top;
  solve_lower_[0] = solve_lower_[1] = 0.0;
  solve_n_[0] = solve_n_[1] = 0;
  for (int s = 0; s < ns; s++) {   // postorder: children first
    const double nc = pl_.nc(s), nr = pl_.nr(s);
    solve_lower_[top[s]] += nc * (nc + 1) / 2 + nr * nc;
    solve_n_[top[s]] += pl_.nc(s);
    if (!top[s]) continue;
    // per group of pivot columns: the group before's chunk of its rows, its values,
    // that chunk of the later groups' rows; then the rows below
    const int n = pl_.nc(s), R = dev::TOP_ROWS, G = dev::INV_GROUP;
    for (int g = 0; g * G < n; g++) {
      const int i0 = g * G / R, i1 = cdiv(std::min(n, (g + 1) * G), R);
      if (g > 0)
        for (int i = i0; i < i1; i++) fwd_top.insert(fwd_top.end(), {s, dev::TOP_CHUNK, i, g - 1});
      for (int i = i0; i < i1; i++) fwd_top.insert(fwd_top.end(), {s, dev::TOP_PIVOT, i, 0});
      if (g > 0)
        for (int i = i1; i < cdiv(n, R); i++)
          fwd_top.insert(fwd_top.end(), {s, dev::TOP_CHUNK, i, g - 1});
    }
    for (int u = 0; u < cdiv(pl_.nr(s), 2048 / dev::top_waves(n)); u++)
      fwd_top.insert(fwd_top.end(), {s, dev::TOP_BELOW, u, 0});
  }
  // forest items, by tree level (leaves first): a tall supernode, or up to four
  // short ones of the level
  std::vector<dev::ForestSn> fsn;
  std::vector<int> fwd, bwd;
  std::vector<int64_t> foff(ns + 1, 0), uvo(ns + 1, 0), dvo(ns + 1, 0);
  for (int s = 0; s < ns; s++) {
    foff[s + 1] = foff[s] + pl_.nc(s) + pl_.nr(s);
    uvo[s + 1] = uvo[s] + pl_.nr(s);
    dvo[s + 1] = dvo[s] + dev::inv_size(pl_.nc(s));
  }
  for (size_t l = 0; l + 1 < pl_.level_ptr.size(); l++) {
    int open = 0;   // waves left in the level's last item
    for (int q = pl_.level_ptr[l]; q < pl_.level_ptr[l + 1]; q++) {
      const int s = pl_.level_sn[q];
      if (top[s]) continue;
      const int i = static_cast<int>(fsn.size());
      fsn.push_back(dev::ForestSn{pl_.sn_first[s], pl_.nc(s), pl_.nr(s), 0, pl_.l_off[s], dvo[s],
                                  uvo[s], foff[s], pl_.rows_ptr[s], 0});
      if (pl_.nc(s) + pl_.nr(s) > dev::FOREST_WAVE_F) {
        // before the level's open item, which stays the last
        fwd.insert(open > 0 ? fwd.end() - 4 : fwd.end(), {i, -2, -2, -2});
      } else {
        if (open == 0) {
          fwd.insert(fwd.end(), {-1, -1, -1, -1});
          open = 4;
        }
        fwd[fwd.size() - open] = i;
        open--;
      }
    }
  }
  for (size_t k = fwd.size(); k >= 4; k -= 4)   // parents first
    bwd.insert(bwd.end(), fwd.begin() + (k - 4), fwd.begin() + k);
  for (int s = ns - 1; s >= 0; s--) {   // parents first
    if (!top[s]) continue;
    const int n = pl_.nc(s), f = n + pl_.nr(s);
    for (int g0 = (n - 1) / dev::INV_GROUP * dev::INV_GROUP; g0 >= 0; g0 -= dev::INV_GROUP) {
      const int g1 = std::min(n, g0 + dev::INV_GROUP);
      for (int kind : {dev::TOP_RHS, dev::TOP_PIVOT}) {
        const int rows = kind == dev::TOP_RHS ? f - g1 : g1 - g0;
        if (rows == 0) continue;
        for (int k = g0; k < g1; k += 16 << dev::top_shape(rows))
          bwd_top.insert(bwd_top.end(), {s, kind, k, 0});
      }
    }
  }
  std::vector<int64_t> exo(ns + 1, pl_.n);
  for (int s = 0; s < ns; s++)
    exo[s + 1] = exo[s] + (top[s] ? static_cast<int64_t>((pl_.nc(s) - 1) / dev::INV_GROUP) * pl_.nc(s) : 0);
  // pull lists: front row of a parent <- entries of its children's update vectors
  std::vector<int> cnt(static_cast<size_t>(foff[ns]) + 1, 0);
  for (int c = 0; c < ns; c++) {
    int p = pl_.sn_parent[c];
    if (p < 0) continue;
    for (int k = pl_.rows_ptr[c]; k < pl_.rows_ptr[c + 1]; k++) cnt[foff[p] + pl_.rel[k] + 1]++;
  }
  for (size_t i = 0; i + 1 < cnt.size(); i++) cnt[i + 1] += cnt[i];
  std::vector<int> src(cnt.back() > 0 ? cnt.back() : 1), fill(cnt.begin(), cnt.end() - 1);
  for (int p = 0; p < ns; p++)
    for (int t = pl_.child_ptr[p]; t < pl_.child_ptr[p + 1]; t++) {
      const int c = pl_.child_list[t];
      for (int k = pl_.rows_ptr[c]; k < pl_.rows_ptr[c + 1]; k++)
        src[fill[foff[p] + pl_.rel[k]]++] =
            static_cast<int>(uvo[c] + (k - pl_.rows_ptr[c]));
    }
  auto upi = [](DevBuf<int>& b, std::vector<int>& v) {
    if (v.empty()) v.push_back(0);
    b.upload(v);
  };
  sd_.n_fwd = static_cast<int>(fwd.size() / 4);
  sd_.n_bwd = static_cast<int>(bwd.size() / 4);
  if (fsn.empty()) fsn.push_back(dev::ForestSn{});
  forest_.upload(fsn);
  sd_.forest = forest_.p;
  sd_.n_fwd_top = static_cast<int>(fwd_top.size() / 4);
  sd_.n_bwd_top = static_cast<int>(bwd_top.size() / 4);
  upi(fwd_items_, fwd);
  upi(bwd_items_, bwd);
  upi(fwd_top_items_, fwd_top);
  upi(bwd_top_items_, bwd_top);
  upi(pull_ptr_, cnt);
  upi(pull_src_, src);
  front_off_.upload(foff);
  exch_off_.upload(exo);
  flags_.alloc(5);   // wait-bound error word, four sweep item counters
  sd_.fwd_items = fwd_items_.p;
  sd_.bwd_items = bwd_items_.p;
  sd_.fwd_items_top = fwd_top_items_.p;
  sd_.bwd_items_top = bwd_top_items_.p;
  sd_.uvec_off = uvec_off_.p;
  sd_.pull_ptr = pull_ptr_.p;
  sd_.pull_src = pull_src_.p;
  sd_.front_off = front_off_.p;
  sd_.exch_off = exch_off_.p;
  n_exch_ = exo[ns];
  sd_.err = flags_.p;
  sd_.ticket = flags_.p + 1;
  forest_full_ = n_cu_ * dev::forest_blocks_per_cu();
  share_ = 1;
  dev::fill_i(flags_.p, 0, 1, st_);
}

// Zeros in the factor storage of b's systems.  The first clean_ ones have them from
// prezero_L, whose fill may still be in flight on the second stream: whatever
// follows waits for it, also when this call has more systems, or it would zero
// entries that were assembled meanwhile.
void CholEngine::zero_L(const dev::Batch& b)
{
  const int have = std::min(clean_, b.count);
  if (clean_ > 0) HIPCHK(hipStreamWaitEvent(st_, ev_zero_, 0));
  if (have < b.count)
    dev::fill(cd_.L + have * b.vs, 0.0, pl_.l_off[pl_.ns],
              dev::Batch{b.count - have, b.vs, b.mask ? b.mask + have : nullptr}, st_);
  clean_ = 0;
}

void CholEngine::prezero_L(int count)
{
  count = std::min(count, cap_);
  dev::fill(cd_.L, 0.0, pl_.l_off[pl_.ns], dev::Batch{count, vs_, nullptr}, st2_);
  HIPCHK(hipEventRecord(ev_zero_, st2_));
  clean_ = count;
}

void CholEngine::assemble(const double* vals, const dev::Batch& b)
{
  zero_L(b);
  dev::scatter(cd_.L, a_dst_.p, vals, a_src_.p, n_assembled(), b, st_);
}

void CholEngine::shift_diag(double delta, const dev::Batch& b)
{
  if (delta != 0.0) dev::add_at(cd_.L, diag_pos_.p, pl_.n, delta, b, st_);
}

void CholEngine::factor(double pivot_tol, const dev::Batch& bt, bool pivots_clear)
{
  HYKKT_REQUIRE(cd_.L && bt.count <= cap_, HYKKT_E_STATE, "factor storage not bound");
  const dev::Batch b{bt.count, vs_, nullptr};
  cd_.pivot_tol = pivot_tol;
  if (!pivots_clear) dev::fill_i(cd_.pivot, INT_MAX, b.count, st_);
  Profiler* pf = prof_ && prof_->on() ? prof_ : nullptr;
  // Bracket one launch (skipped when it has no tasks, like the launchers);
  // charged with the work of all the systems it covers.
  auto timed_on = [&](hipStream_t st, int kind, const Launch& la, auto&& launch) {
    if (la.cnt <= 0) return;
    if (pf) pf->begin(st);
    launch();
    if (pf) pf->end(kind, st, la.flops * b.count, la.bytes * b.count);
  };
  auto timed = [&](int kind, const Launch& la, auto&& launch) { timed_on(st_, kind, la, launch); };
  for (const Level& L : lv_) {
    auto add_children = [&](const Launch& la) {
      timed(PK_EXTEND_ADD, la, [&] {
        dev::extend_add(cd_, la.cnt, t_ea_p_.p + la.off, t_ea_col_.p + la.off, t_ea_cptr_.p + la.off,
                        t_ea_cc_.p, t_ea_ccol_.p, b, st_);
      });
    };
    add_children(L.ea_panel);
    timed(PK_POTRF, L.front, [&] {
      dev::front_panel(cd_, L.front.cnt, t_fp_sn_.p + L.front.off, t_fp_tile_.p + L.front.off, b,
                       st_);
    });
    // Blocked steps with look-ahead.  Main stream: diagonal blocks, TRSM,
    // update of the next block column(s); second stream: the rest of the
    // trailing update, which overlaps the next steps' diagonal blocks and
    // TRSMs.  A main-stream update waits for the pending rests (ev_rest_)
    // only when it writes a block column they write (rest_lo: the lowest
    // such column); a rest waits for its step's TRSM and next-column update
    // (ev_main_).  Both events are re-recorded after their waits were
    // enqueued.
    bool rest_pending = false;
    int rest_lo = INT_MAX;
    // an update of up to five tiles of 128 x 128 per compute unit and K <= 512 takes
    // 64 x 64 ones: more waves cover the loads of C, and the last ones end together
    // (K = 128, 435 tiles: 50 -> 46 us; factor at 5,000 buses 2.99 -> 2.94 ms, 10,000
    // 10.2 -> 9.8, 20,000 49.8 -> 48.8, 40,000 518 -> 516).  A larger one is better
    // off with fewer operand loads (64 x 64 throughout, 20,000 buses: 53.4; for these
    // launches at any K, 40,000: 520)
    auto quarters = [&](const Launch& la, int kblk) {
      return kblk <= 4 && static_cast<int64_t>(la.cnt) * b.count <= 5 * static_cast<int64_t>(n_cu_);
    };
    for (size_t j = 0; j < L.potrf.size(); j++) {
      const int step = static_cast<int>(j);
      // in a group of G starting at step a: step a+i updates block column
      // step+1 by blocks a .. a+i (mode i+2 for K = i+1 blocks from block a,
      // mode 0 for one block); the last step block columns step+1 .. step+G
      // by all G blocks (mode G+1), its rest step+G+1 on
      const int gi = L.gpos[j], G = L.gsize[j], a = step - gi;
      const bool last = gi == G - 1;
      const int kblk = last ? G : gi + 1;
      const int umode = kblk == 1 ? 0 : kblk + 1, ustep = a;
      const int upd_hi = L.upd_whole[j] ? INT_MAX : (last && G > 1) ? step + G : step + 1;
      timed(PK_POTRF, L.potrf[j], [&] {
        dev::potrf_inv(cd_, L.potrf[j].cnt, t_potrf_.p + L.potrf[j].off, step, L.potrf[j].maxb, b,
                       st_);
      });
      if (L.potrf[j].maxb > 64) {
        // 128-wide blocks: blocked substitution, no whole inverse needed yet
        timed(L.trsm[j].short_rows ? PK_TRSM_SHORT : PK_TRSM, L.trsm[j], [&] {
          dev::trsm(cd_, L.trsm[j].cnt, t_trsm_sn_.p + L.trsm[j].off,
                    t_trsm_tr_.p + L.trsm[j].off, step, b, st_, L.trsm[j].short_rows);
        });
      } else {
        timed(L.trsm[j].short_rows ? PK_DENSE_NT_SHORT : PK_DENSE_NT, L.trsm[j], [&] {
          dev::trsm_inv(cd_, L.trsm[j].cnt, t_trsm_sn_.p + L.trsm[j].off,
                        t_trsm_tr_.p + L.trsm[j].off, step, b, st_, L.trsm[j].short_rows);
        });
      }
      if (rest_pending && upd_hi >= rest_lo) {
        HIPCHK(hipStreamWaitEvent(st_, ev_rest_, 0));
        rest_pending = false;
        rest_lo = INT_MAX;
      }
      // the rest waits for this step's next-column update: its event is
      // recorded by that launch's own completion where there is one
      const bool rest = L.upd_rest[j].cnt > 0;
      const bool on_launch = rest && L.upd_next[j].cnt > 0;
      timed(L.upd_next[j].short_rows ? PK_DENSE_NT_SHORT : PK_DENSE_NT, L.upd_next[j], [&] {
        dev::dense_nt(cd_, L.upd_next[j].cnt, t_upd_sn_.p + L.upd_next[j].off,
                      t_upd_tr_.p + L.upd_next[j].off, t_upd_tc_.p + L.upd_next[j].off, umode,
                      ustep, b, st_, L.upd_next[j].short_rows, on_launch ? ev_main_ : nullptr, false,
                      quarters(L.upd_next[j], kblk));
      });
      if (rest) {
        if (!on_launch) HIPCHK(hipEventRecord(ev_main_, st_));
        HIPCHK(hipStreamWaitEvent(st2_, ev_main_, 0));
        // off the diagonal block's compute unit (see dense_nt): up to two tiles of 128 x
        // 128 a compute unit, which are then all resident; as quarters up to eight
        // workgroups, of which the LDS lets five in at a time.  The line at those five
        // takes longer (5,000 buses 3740 -> 3766 us, 10,000 and batches the same)
        timed_on(st2_, PK_DENSE_NT, L.upd_rest[j], [&] {
          dev::dense_nt(cd_, L.upd_rest[j].cnt, t_upd_sn_.p + L.upd_rest[j].off,
                        t_upd_tr_.p + L.upd_rest[j].off, t_upd_tc_.p + L.upd_rest[j].off, umode,
                        ustep, b, st2_, false, ev_rest_,
                        L.upd_rest[j].cnt * b.count <= 2 * n_cu_,
                        quarters(L.upd_rest[j], kblk));
        });
        rest_pending = true;
        rest_lo = std::min(rest_lo, upd_hi + 1);   // the rest starts after the columns just updated
      }
    }
    if (rest_pending) HIPCHK(hipStreamWaitEvent(st_, ev_rest_, 0));
    timed(PK_DENSE_NT, L.syrk, [&] {
      dev::update_matrices(cd_, L.syrk.cnt, t_syrk_sn_.p + L.syrk.off, t_syrk_tr_.p + L.syrk.off,
                           t_syrk_tc_.p + L.syrk.off, L.small_u, b, st_);
    });
    add_children(L.ea_u);
  }
  // the solves' inverses, all levels at once
  timed(PK_INV_GROUP, inv_grp_, [&] {
    dev::inv_groups(cd_, inv_grp_.cnt, t_grp_sn_.p, t_grp_ix_.p, b, st_);
  });
}

std::vector<int> CholEngine::pivots(int count)
{
  std::vector<int> h(std::max(count, 1), INT_MAX);
  HIPCHK(hipMemcpyAsync(h.data(), cd_.pivot, sizeof(int) * count, hipMemcpyDeviceToHost, st_));
  HIPCHK(hipStreamSynchronize(st_));
  for (int& v : h) v = (v == INT_MAX) ? -1 : v;
  h.resize(count);
  return h;
}

void CholEngine::clear_solve_error() { dev::fill_i(sd_.err, 0, 1, st_); }

void CholEngine::set_sweep_share(int share)
{
  share = std::max(share, 1);
  if (share == share_) return;
  share_ = share;
  if (share == 1) {
    sd_.cap_forest = sd_.cap_top = 0;
    return;
  }
  // the forest sweeps: their share of the 256-thread workgroups the device
  // holds; the top of the tree: of two 1024-thread workgroups per CU
  sd_.cap_forest = std::max(1, forest_full_ / share);
  sd_.cap_top = std::max(1, 2 * n_cu_ / share);
}

int CholEngine::solve_error()
{
  int h = 0;
  HIPCHK(hipMemcpyAsync(&h, sd_.err, sizeof(int), hipMemcpyDeviceToHost, st_));
  HIPCHK(hipStreamSynchronize(st_));
  if (h) dev::fill_i(sd_.err, 0, 1, st_);
  return h;
}

dev::SweepFill CholEngine::sweep_fill(double* x) const
{
  dev::SweepFill f;
  f.p[0] = ybuf_;
  f.n[0] = pl_.n;
  f.p[1] = x;
  f.n[1] = pl_.n;
  f.p[2] = sd_.ubuf;
  f.n[2] = n_ubuf_;
  f.p[3] = sd_.exch;
  f.n[3] = n_exch_;
  f.ticket = sd_.ticket;
  return f;
}

void CholEngine::solve(const double* rhs, double* x, const dev::Batch& bt, bool filled)
{
  const dev::Batch b{bt.count, vs_, bt.mask};
  Profiler* pf = prof_ && prof_->on() ? prof_ : nullptr;
  // Algorithmic, per part of the tree: each sweep reads that part's factor
  // entries (lower trapezoids of its panels) once, 2 flops per entry, and
  // reads + writes its vector entries; charged for every system of the
  // launch (those a mask skips included).
  auto sweep = [&](int kind, int part, bool fwd) {
    if ((part == 0 ? (fwd ? sd_.n_fwd : sd_.n_bwd) : (fwd ? sd_.n_fwd_top : sd_.n_bwd_top)) <= 0)
      return;
    if (pf) pf->begin(st_);
    if (fwd)
      (part ? dev::solve_forward_top : dev::solve_forward_forest)(cd_, sd_, rhs, ybuf_, b, st_);
    else
      (part ? dev::solve_backward_top : dev::solve_backward_forest)(cd_, sd_, ybuf_, x, b, st_);
    if (pf)
      pf->end(kind, st_, 2.0 * solve_lower_[part] * b.count,
              8.0 * (solve_lower_[part] + 2.0 * solve_n_[part]) * b.count);
  };
  if (!filled) dev::fill_sentinel(sweep_fill(x), b, st_);
  sweep(PK_SOLVE_FWD_FOREST, 0, true);
  sweep(PK_SOLVE_FWD_TOP, 1, true);
  sweep(PK_SOLVE_BWD_TOP, 1, false);
  sweep(PK_SOLVE_BWD_FOREST, 0, false);
}

}  // namespace hykkt
