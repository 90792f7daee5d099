"""Krylov-Schur on FP32 factors without refinement (STAB_IR_MAX = 0): the same
operator from its own factors alone, whatever ran before.

The factors solve a pencil that differs from M by a backward error of about
n u32 = 3e-5 of its norm at n = 480 (partial pivoting, equilibrated; 1e-3
allows for growth and for undoing the scales), which is what the residuals of
the pairs, formed with the FP64 pencil, may show."""
import os

import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", ["0", "256"])
@pytest.mark.parametrize("ny", [48, 96])
def test_unrefined_factors_expand_their_own_basis(gpu_solver, monkeypatch, ny, wide):
    from oracle import stab_oracle as so
    from stab_amd import _lib
    from stab_amd import solver as sv
    inp = sv.read_input(open(os.path.join(GOLDEN, "thesis_TStest", "temporal.inp")).read())
    inp.ny = ny
    gpu_solver.set_profile(0, *so.read_profile(os.path.join(GOLDEN, "TStest", "profile.0")))
    sh = (0.1146788 + 0.0023845j) * (1 + 2e-3j)
    pt, other = sv.make_point(inp, sh, 4), sv.make_point(inp, 0.25 + 0.05j, 4)
    monkeypatch.setenv("STAB_WIDE_POINTS", wide)
    monkeypatch.setenv("STAB_IR_MAX", "0")
    got = []
    for before in (pt, other):                       # the pools hold this point's basis, then another's
        gpu_solver.solve([before], _lib.MODE_PLAIN_F64)
        got.append(gpu_solver.solve([pt], _lib.MODE_MIXED))
    a, b = got
    assert a.info[0] == b.info[0] == _lib.INFO_OK
    assert np.array_equal(a.evals, b.evals) and np.array_equal(a.resid, b.resid)
    assert np.all(a.resid[0, :4] <= 1e-3)
    assert np.max(a.resid[0, :4]) > 1e-13            # the factors alone: no refined answer came back
