"""The device buffers of a network (stab_amd/csrc/mlp_bufs.h) when an
allocation fails, compiled with g++ against a counting hipMalloc / hipFree: no
pointer to freed memory is kept, nothing is freed twice, the loss that every
training call writes stays allocated, and the next call allocates again."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r'''
#include "mlp_bufs.h"
#include <cstdio>
#include <cstdlib>
#include <set>
static std::set<void *> live;
static int bad = 0, fail_at = -1, calls = 0;
static bool pending = false;                          // the error hipGetLastError would still report
extern "C" hipError_t hipMalloc(void **p, size_t n) {
  if (calls++ == fail_at) { pending = true; return hipErrorOutOfMemory; }
  *p = malloc(n < 4096 ? n : 4096);
  live.insert(*p);
  return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
  if (!live.erase(p)) { ++bad; return hipErrorInvalidValue; }
  free(p);
  return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { pending = false; return hipSuccess; }
static void ok(const void *p, bool must) { bad += p ? !live.count((void *)p) : must; }
struct Net {
  DevPool pool;
  MlpRowBufs rows;
  MlpSetBufs set;
  MlpLossBuf loss;
  void check(bool all) {
    for (const void *p : {(void *)rows.actT, (void *)rows.dzT, (void *)rows.act32, (void *)rows.part, (void *)rows.losspart})
      ok(p, all && rows.cap > 0);
    for (const void *p : {(void *)set.X, (void *)set.T, (void *)set.xraw, (void *)set.traw}) ok(p, all && set.cap > 0);
    ok(loss.p, true);
  }
};
int main() {
  for (int which = 0; which < 3; ++which)
    for (int at = 0; at < 5; ++at) {
      Net n;
      fail_at = -1;
      bad += n.loss.reserve(n.pool, 0) != hipSuccess;
      bad += n.rows.reserve(n.pool, 16, 96, 64) != hipSuccess;
      bad += n.set.reserve(n.pool, 5, 16, 2, 64) != hipSuccess;
      n.check(true);
      auto grow = [&](int f) {
        if (which == 0) return n.rows.reserve(n.pool, 16, 96, 64 * f);
        if (which == 1) return n.set.reserve(n.pool, 5, 16, 2, 64 * f);
        return n.loss.reserve(n.pool, 100 * f);
      };
      const int count = which == 0 ? 5 : (which == 1 ? 4 : 1);
      for (int rep = 0; rep < 2; ++rep) {           // fails, and fails again
        calls = 0;
        fail_at = at % count;
        bad += grow(4) == hipSuccess;
        n.check(false);
        bad += pending;
      }
      fail_at = -1;
      bad += grow(2) != hipSuccess;                  // a smaller request than the one that failed
      n.check(true);
      bad += (which == 0 ? n.rows.cap : which == 1 ? n.set.cap : n.loss.cap) != (which == 2 ? 200 : 128);
      n.pool.clear();
      bad += !live.empty();
    }
  std::printf("%d\n", bad);
  return 0;
}
'''


def test_failed_growth_leaves_no_stale_pointer(tmp_path):
    cxx, inc = shutil.which("g++"), "/opt/rocm/include"
    if not cxx or not os.path.isdir(os.path.join(inc, "hip")):
        pytest.skip("g++ or the HIP headers not available")
    src, exe = tmp_path / "bufs.cpp", tmp_path / "bufs"
    src.write_text(SRC)
    r = subprocess.run([cxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", inc, "-I",
                        os.path.join(ROOT, "stab_amd", "csrc"), str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "0", out.stdout
