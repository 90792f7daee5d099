"""Properties of the compiled device code (hipcc for gfx950, no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import ROOT


def test_panel_accesses_are_global(tmp_path):
    """The LU panels reach the matrix through global loads and stores: a flat
    one (an address whose space the compiler lost) also counts as an LDS access
    where a wave waits, so the loads issued ahead would be waited for early."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    src, out = tmp_path / "panel.hip", tmp_path / "panel.s"
    src.write_text('#include "lu.hip"\n' + "".join(
        f"template __global__ void k_lu_panel<{t}>(const PointDev *, cx<{t.split(',')[0]}> *, int *, "
        f"cx<{t.split(',')[0]}> *, int *, const int *, int, int);\n" for t in ("float, 16, 256, 1", "double, 8, 256, 1")))
    r = subprocess.run([hipcc, "-O3", "--offload-arch=gfx950", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I", os.path.join(ROOT, "stab_amd", "csrc"), "--cuda-device-only", "-S",
                        str(src), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    text = out.read_text()
    assert "k_lu_panel" in text and "global_load_dword" in text
    assert not re.findall(r"flat_(?:load|store)\w*", text)
