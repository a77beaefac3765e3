// profiler.hpp -- optional per-kernel timing with HIP events.
//
// When enabled, every launch of an instrumented kernel is bracketed by two
// events on the stream it runs on; collect() (stream idle) adds each launch's
// duration, and the algorithmic flops / HBM bytes the launch was charged with,
// to its kernel's totals.  Disabled, begin()/end() cost one branch.
#pragma once

#include <hip/hip_runtime_api.h>

#include <vector>

namespace hykkt {

// Groups of launches, each under one name (Profiler::name).  The names are an interface
// that callers look groups up by; several are those of kernels since split or replaced,
// so a group's kernels are listed here.
enum ProfKind {
  PK_DENSE_NT = 0,       // k_dense_nt with tiles of 128 x 128 and 64 x 64 (updates, update
                         // matrices), k_trsm_inv<128>
  PK_DENSE_NT_SHORT,     // k_dense_nt with 32-row tiles, k_trsm_inv<32> (the short launches
                         // on the critical path)
  PK_POTRF,              // k_potrf_inv<128, 64, 32>, k_front_panel
  PK_EXTEND_ADD,         // k_extend_add
  PK_SOLVE_FWD_FOREST,   // k_forest<true, ..>
  PK_SOLVE_FWD_TOP,      // k_solve_fwd
  PK_SOLVE_BWD_TOP,      // k_solve_bwd
  PK_SOLVE_BWD_FOREST,   // k_forest<false, ..>
  PK_SPMV,               // k_spmv, k_spmv_rows, k_cg_apply, k_recover, k_residual
  PK_SPGEMM_VALUES,      // k_spgemm_values
  PK_SPGEMM_SCATTER,     // k_spgemm_scatter
  PK_TRSM,               // k_trsm<128>
  PK_TRSM_SHORT,         // k_trsm<64>
  PK_INV_GROUP,          // k_inv_group
  PK_COUNT
};

// Algorithmic HBM bytes of one y = alpha A x + beta y_in over a CSR A (rows
// x cols, nnz entries): row pointers, column indices and values read once
// (and the value map, when the values are read through one), x and y_in
// once, y written once; with a fused dot, its other operand read once.
inline double spmv_bytes(int rows, int cols, double nnz, bool map, bool y_in, bool dot)
{
  return 4.0 * (rows + 1) + (map ? 16.0 : 12.0) * nnz + 8.0 * cols +
         8.0 * rows * (1 + (y_in ? 1 : 0) + (dot ? 1 : 0));
}

class Profiler {
 public:
  struct Total {
    long long launches = 0;
    double ms = 0.0, flops = 0.0, bytes = 0.0;
  };
  Profiler() = default;
  Profiler(const Profiler&) = delete;
  Profiler& operator=(const Profiler&) = delete;
  ~Profiler();
  void enable(bool on);   // also clears the totals
  bool on() const { return on_ && !paused_; }
  // Leave the launches between pause(true) and pause(false) out.
  void pause(bool p) { paused_ = p; }
  void begin(hipStream_t st);
  void end(int kind, hipStream_t st, double flops, double bytes);
  void collect();
  const Total& total(int k) const { return tot_[k]; }
  static const char* name(int k);

 private:
  struct Pend {
    int kind;
    hipEvent_t a, b;
    double flops, bytes;
  };
  hipEvent_t get();
  bool on_ = false;
  bool paused_ = false;
  hipEvent_t open_ = nullptr;
  std::vector<Pend> pend_;
  std::vector<hipEvent_t> free_, all_;
  Total tot_[PK_COUNT];
};

}  // namespace hykkt
