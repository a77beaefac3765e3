// cg.cpp -- Schur-complement conjugate gradient on the device, for a batch of
// same-pattern systems.
//
// Same recurrences as SchurComplementConjugateGradient.cpp:102-194
// (Chronopoulos-Gear form: one S-apply and two dots per iteration):
//   p = beta p + r;  s = beta s + w;  x += alpha p;  r -= alpha s;
//   gam1 = r.r;  stop if sqrt(gam1) < tol;  w = S r;  delta = w.r;
//   beta = gam1/gam;  gam = gam1;  alpha = gam/(delta - beta gam/alpha).
// Device-resident: the vector update carries the r.r partials, the second
// SpMV of the S-apply carries the w.r partials, and the kernels that use the
// sums finish them: the start of the next S r takes the stopping test, and
// clears a system's live flag when it stops, the update the scalar recurrences.
// An iteration is cg_apply, the triangular solves, an SpMV and cg_update.
#include <cmath>

#include "device.hpp"

namespace hykkt {

namespace {

template <class F>
void timed_spmv(SchurOps& o, int rows, int cols, bool y_in, bool dot, int count, F&& launch)
{
  if (o.prof) o.prof->begin(o.st);
  launch();
  if (o.prof)
    o.prof->end(PK_SPMV, o.st, 2.0 * o.nnz * count,
                spmv_bytes(rows, cols, o.nnz, false, y_in, dot) * count);
}

}  // namespace

void cg_start(SchurOps& o, const double* b, const dev::Batch& bt, bool x0_zero)
{
  dev::CgVecs& v = o.v;
  dev::cg_start(v, b, x0_zero, o.f, bt, o.st);
  o.k = 0;
  if (x0_zero) return;
  // r = b - S x0 (:104-122), z = A^{-1} Jh^T x0
  const dev::Batch live = dev::masked(bt, o.f.live);
  timed_spmv(o, v.n, v.m, false, false, bt.count, [&] {
    dev::spmv_rows(v.n, o.jth_rp, o.jth_ci, o.jth_v, v.x, v.t1, live, o.st);
  });
  o.chol->solve(v.t1, v.t2, live);
  timed_spmv(o, v.m, v.n, true, false, bt.count, [&] {
    dev::spmv(v.m, o.jh_rp, o.jh_ci, nullptr, o.jh_v, -1.0, nullptr, v.t2, 1.0, b, v.r, o.jh_blk,
              o.jh_nblk, live, o.st);
  });
  if (v.z) dev::copy(v.z, v.t2, v.n, live, o.st);
  dev::dot_partial(v.m, v.r, v.r, v.part, live, o.st);
}

void cg_iterate(SchurOps& o, int count, double tol, int itmax, const dev::Batch& bt)
{
  dev::CgVecs& v = o.v;
  const dev::Batch live = dev::masked(bt, o.f.live);
  for (int i = 0; i < count && o.k < itmax; i++, o.k++) {
    timed_spmv(o, v.n, v.m, false, false, bt.count, [&] {
      dev::cg_apply(v, o.k, tol, itmax, o.jth_rp, o.jth_ci, o.jth_v, o.chol->sweep_fill(v.t2), o.f,
                    bt, o.st);
    });
    o.chol->solve(v.t1, v.t2, live, true);
    timed_spmv(o, v.m, v.n, false, true, bt.count, [&] {
      dev::spmv(v.m, o.jh_rp, o.jh_ci, nullptr, o.jh_v, 1.0, nullptr, v.t2, 0.0, nullptr, v.w,
                o.jh_blk, o.jh_nblk, live, o.st, v.r, v.part2);
    });
    dev::cg_update(v, o.k, o.f, bt, o.st);
  }
}

CgResult cg_result(const double* fin)
{
  return CgResult{static_cast<int>(fin[dev::FIN_ITERS]), static_cast<int>(fin[dev::FIN_STATUS]),
                  std::sqrt(fin[dev::FIN_RR])};
}

}  // namespace hykkt
