"""The size of the factorization's index of children's rows: bounded by the children's
rows, whatever their number.  Host code only."""
import os
import subprocess

import numpy as np

from conftest import ROOT

SRC = os.path.join(ROOT, "hykkt_amd", "csrc")

HARNESS = r"""
#include <cstdio>
#include "symbolic.hpp"
using namespace hykkt;
int main(int, char** argv)
{
  std::FILE* f = std::fopen(argv[1], "rb");
  int n = 0;
  if (!f || std::fread(&n, 4, 1, f) != 1) return 1;
  Pattern a;
  a.n = a.m = n;
  a.rp.resize(n + 1);
  if (std::fread(a.rp.data(), 4, n + 1, f) != static_cast<size_t>(n + 1)) return 1;
  a.ci.resize(a.rp[n]);
  if (std::fread(a.ci.data(), 4, a.ci.size(), f) != a.ci.size()) return 1;
  const CholPlan p = chol_analyze(a, CholOptions{});
  int none = 0;
  for (int s = 0; s < p.ns; s++) {
    if (!p.pulls[s]) {
      none++;
      continue;
    }
    // every row of a child at or past inv_first, at its place and nowhere else
    const int first = p.inv_first(s, CholOptions{}.index_narrow);
    const int nch = p.child_ptr[s + 1] - p.child_ptr[s];
    for (int t = 0; t < nch; t++) {
      const int c = p.child_list[p.child_ptr[s] + t];
      int left = 0, found = 0;
      for (int q = p.rows_ptr[c]; q < p.rows_ptr[c + 1]; q++) left += p.rel[q] >= first;
      for (int r = first; r < p.nc(s) + p.nr(s); r++) {
        const int k = p.inv[p.inv_off[s] + static_cast<long long>(t) * p.inv_rows[s] + r];
        if (k < 0) continue;
        if (k >= p.nr(c) || p.rel[p.rows_ptr[c] + k] != r) return 2;
        found++;
      }
      if (found != left) return 3;
    }
  }
  std::printf("%zu %zu %d\n", p.inv.size(), p.rel.size(), none);
  return 0;
}
"""


def many_leaves(mc, nr, leaves):
    """Lower triangle: two dense blocks of mc columns over nr root rows, each with
    `leaves` one-column children of two rows (one in the block, one of the root)."""
    rng = np.random.default_rng(1)
    rows, cols = [], []
    per = leaves + mc
    root = 2 * per
    n = root + nr
    for m in range(2):
        m0 = m * per
        k = np.arange(leaves)
        for r in (m0 + leaves + k % mc, root + rng.integers(0, nr, leaves)):
            rows.append(r)
            cols.append(m0 + k)
        i, j = np.tril_indices(mc)
        rows.append(m0 + leaves + i)
        cols.append(m0 + leaves + j)
        i, j = np.indices((nr, mc)).reshape(2, -1)
        rows.append(root + i)
        cols.append(m0 + leaves + j)
    i, j = np.tril_indices(nr)
    rows.append(root + i)
    cols.append(root + j)
    rows.append(np.arange(n))
    cols.append(np.arange(n))
    key = np.unique(np.concatenate(rows).astype(np.int64) * n + np.concatenate(cols))
    r, c = key // n, key % n
    return np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32), \
        c.astype(np.int32)


def test_index_size(tmp_path):
    exe = tmp_path / "index"
    (tmp_path / "index.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{SRC}", str(tmp_path / "index.cpp")] +
                   [os.path.join(SRC, f) for f in ("cholplan.cpp", "symbolic.cpp", "amd.cpp")] +
                   ["-o", str(exe)], check=True)
    for mc, nr, leaves, indexed in [(20, 40, 12, True), (20, 150, 400, False), (300, 400, 20_000, False)]:
        rp, ci = many_leaves(mc, nr, leaves)
        with open(tmp_path / "p", "wb") as f:
            np.int32(len(rp) - 1).tofile(f)
            rp.tofile(f)
            ci.tofile(f)
        out = subprocess.run([str(exe), str(tmp_path / "p")], check=True, capture_output=True, text=True)
        size, rel, none = map(int, out.stdout.split())
        print(mc, nr, leaves, "index", size, "rows", rel, "without", none)
        assert size <= 64 * rel
        assert (none == 0) == indexed
