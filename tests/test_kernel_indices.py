"""Index rules that kernels and host share, replayed on the CPU: a small program built with the
library's own internal header and linked to the library walks the same loops and checks every
index.  No GPU is used."""
import os
import subprocess

import pytest

import sbdg
from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def run_replay(tmp_path, body):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "replay.cc", tmp_path / "replay"
    src.write_text('#include "sbdg_internal.h"\n#include <cstdio>\n#include <vector>\n#include <algorithm>\n'
                   "using namespace sbdg;\n" + body)
    lib = os.path.dirname(sbdg.LIBPATH)
    subprocess.check_call([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", f"-I{ROOT}/sbd-ykt_amd/csrc",
                           f"-I{ROOT}/include", str(src), "-o", str(exe), f"-L{lib}", "-lsbdg", f"-Wl,-rpath,{lib}"])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr


def test_alpha_beta_staging_stays_inside_the_ket_row(tmp_path):
    """k_ab's staging loads, two neighbouring columns each and none under a condition: every one
    inside its chunk of the ket row, every column of the chunk stored, for one beta string (which
    must not reach the kernel: the second column of its last row lies past the vector), two,
    three, and both sides of each launch geometry."""
    run_replay(tmp_path, r"""
int main() {
  long seen = 0;
  for (int L : {2, 18, 36, 64})
    for (int elem : {4, 8})
      for (int64_t nb : {1, 2, 3, 5, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025, 2047, 6000, 6001, 8193, 24576, 24577, 40705}) {
        if (!ab_any(nb)) continue;  // not launched
        const AbGeometry g = ab_geometry(nb, L, elem);
        const int SR = ab_ket_round(elem, g.m), SV = ab_slice_round(g.nt), NPS = (int)ab_pairs(L);
        for (int64_t j0 = 0; j0 < nb; j0 += g.chunk) {
          const int nj = (int)(std::min(nb, j0 + g.chunk) - j0);
          std::vector<char> stored(nj, 0);
          for (int xt = 0; xt < g.nt; ++xt)
            for (int x0 = 2 * xt, y0 = xt; x0 < nj || y0 < NPS; x0 += SR * g.nt, y0 += SV * g.nt)
              for (int u = 0; u < SR; u += 2) {
                const int x = ab_stage_pair(x0 + u * g.nt, nj);
                if (x < 0 || x + 1 >= nj) {
                  printf("nb %ld L %d: columns %d, %d of %d\n", (long)nb, L, x, x + 1, nj);
                  return 1;
                }
                if (x0 + u * g.nt < nj) stored[x] = stored[x + 1] = 1;
              }
          for (char c : stored)
            if (!c) {
              printf("nb %ld L %d: a column is not staged\n", (long)nb, L);
              return 1;
            }
          ++seen;
        }
      }
  printf("%ld chunks\n", seen);
  return seen > 50 ? 0 : 1;
}
""")


def test_eigenvalue_ranks_are_a_permutation_whatever_the_values(tmp_path):
    """k_jacobi ranks the diagonal by counting the places before each and writes each place to its
    rank: with NaN and infinities too every rank has to occur once (one left out would be an unset
    place, then an index into LDS), and ordinary values come out ascending."""
    run_replay(tmp_path, r"""
int main() {
  const double nan = __builtin_nan(""), inf = __builtin_inf();
  const double pool[] = {nan, -inf, -1.0, -0.0, 0.0, 0.0, 2.5, inf, nan, -1.0};
  unsigned long long r = 12345;
  for (int t = 0; t < 20000; ++t) {
    const int m = 1 + t % 48;
    std::vector<double> a(m);
    for (double& x : a) {
      r = r * 6364136223846793005ull + 1442695040888963407ull;
      x = t % 3 ? pool[(r >> 33) % 10] : (double)(long long)(r >> 20);
    }
    std::vector<int> ord(m, -1);
    for (int k = 0; k < m; ++k) {
      int rank = 0;
      for (int j = 0; j < m; ++j) rank += eigen_before(a[j], j, a[k], k);
      if (rank >= m || ord[rank] >= 0) {
        printf("rank %d of %d twice\n", rank, m);
        return 1;
      }
      ord[rank] = k;
    }
    for (int k = 1; k < m; ++k) {
      const double x = a[ord[k - 1]], y = a[ord[k]];
      if (x > y || (x != x && y == y) || (x == y && ord[k - 1] > ord[k])) return 1;
    }
  }
  return 0;
}
""")
