"""Rules of the kernels (stab_amd/csrc/bounds.h), compiled with g++ and checked
on the host over the sizes and values they meet."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


def _run(tmp_path, body):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "bounds.cpp", tmp_path / "bounds"
    src.write_text('#include "bounds.h"\n#include <cstdio>\nint main() {\n  long long bad = 0;\n' + body +
                   '  std::printf("%lld\\n", bad);\n  return 0;\n}\n')
    r = subprocess.run([cxx, "-O1", "-std=c++17", "-I", os.path.join(ROOT, "stab_amd", "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0
    return int(out.stdout)


def test_l11_staging_stays_in_the_matrix(tmp_path):
    """Every order (multiples of 32 to 1280), every 64-column block, every
    entry: the element read lies in the n x n matrix, and is entry (i, k) of
    the block where the block has one."""
    assert _run(tmp_path, r'''
  for (int n = 32; n <= 1280; n += 32)
    for (int K0 = 0; K0 < n; K0 += 64) {
      const int kb = n - K0 < 64 ? n - K0 : 64;
      for (int i = 0; i < 64; ++i)
        for (int k = 0; k < i; ++k) {
          const long long e = lu_l11_src(K0, kb, i, k, n);
          bad += e < 0 || e >= (long long)n * n;
          if (i < kb) bad += e != (long long)(K0 + k) * n + K0 + i;
        }
    }
''') == 0


def test_schur_reorder_picks_a_row_of_the_matrix(tmp_path):
    """The row brought to the front by k_schur, from the ballot its 64 lanes
    form, over basis sizes, positions and patterns of NaN, infinite, equal and
    ordinary moduli: inside [pos, m), the first of the largest, pos when every
    modulus is NaN."""
    assert _run(tmp_path, r'''
  const double nan = __builtin_nan(""), inf = __builtin_inf();
  unsigned s = 1;
  for (int m = 2; m <= 64; ++m)
    for (int pos = 0; pos < m; ++pos)
      for (int pat = 0; pat < 12; ++pat) {
        double av[64], bv = -1.0;
        for (int l = 0; l < 64; ++l) {
          s = s * 1664525u + 1013904223u;
          const double r = (double)(s >> 8) / 16777216.0;
          double v = pat == 0 ? nan : pat == 1 ? 0.0 : pat == 2 ? 1.0 : pat == 3 ? (r < 0.5 ? nan : 2.0) : r;
          if (pat == 4 && r < 0.1) v = inf;
          if (pat >= 8 && r < 0.9) v = nan;
          av[l] = (l >= pos && l < m) ? v : -1.0;
          if (av[l] > bv) bv = av[l];       // fmax drops NaN
        }
        unsigned long long at = 0;
        int want = pos;
        double wv = -1.0;
        for (int l = 0; l < 64; ++l) at |= (unsigned long long)(av[l] == bv) << l;
        for (int l = pos; l < m; ++l)
          if (av[l] > wv) { wv = av[l]; want = l; }
        const int got = schur_pick(at, pos, m);
        bad += got < pos || got >= m || got != want;
      }
''') == 0


def test_residual_estimate_keeps_nan(tmp_path):
    """The largest estimate of the wanted pairs: the plain maximum of numbers
    and infinities, NaN (neither converged nor a number to improve on) with a
    NaN in any place."""
    assert _run(tmp_path, r'''
  const double nan = __builtin_nan(""), inf = __builtin_inf();
  for (int n = 1; n <= 16; ++n) {
    double e[16];
    for (int i = 0; i < n; ++i) e[i] = 1e-14 * (i + 1);
    bad += est_max(e, n) != 1e-14 * n;
    for (int k = 0; k < n; ++k) {
      const double was = e[k];
      e[k] = inf;
      bad += est_max(e, n) != inf;
      e[k] = nan;
      bad += est_max(e, n) <= 1e-12 || est_max(e, n) > 1e-12;
      e[k] = was;
    }
    for (int i = 0; i < n; ++i) e[i] = nan;
    bad += est_max(e, n) <= 1e-12 || est_max(e, n) > 1e-12;
  }
''') == 0
