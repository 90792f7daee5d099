"""A point whose pencil is not finite (parameters the checks accept, products
that overflow) beside ordinary points: the LU keeps every index in range (its
all-NaN columns take the diagonal as pivot), no entry point reports the point as
solved, and the points around it get what they get alone."""
import os

import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu


def _points(ny):
    from oracle import stab_oracle as so
    from stab_amd import solver as sv
    text = open(os.path.join(GOLDEN, "thesis_TStest", "temporal.inp")).read()
    inp, bad = sv.read_input(text), sv.read_input(text)
    inp.ny = bad.ny = ny
    bad.alpha = 1e200 + 0j                     # alpha^2 overflows: Inf, and NaN where it meets zeros
    sh = 0.1146788 + 0.0023845j
    good = sv.make_point(inp, sh, 4)
    return good, sv.make_point(bad, sh, 4), so.read_profile(os.path.join(GOLDEN, "TStest", "profile.0"))


# 48: n = 240, a 64-wide last block; 64: whole blocks; 96: n = 480, a 32-wide last block and two rows per thread
@pytest.mark.parametrize("ny", [48, 64, 96])
def test_nonfinite_point_is_not_solved(gpu_solver, ny):
    from stab_amd import _lib
    good, bad, prof = _points(ny)
    gpu_solver.set_profile(0, *prof)
    print(f"nonfinite N {ny}: pencil", flush=True)
    assert not np.all(np.isfinite(gpu_solver.pencil(bad, _lib.MAT_SHIFTED)))
    for mode in (_lib.MODE_PLAIN_F64, _lib.MODE_MIXED):
        print(f"nonfinite N {ny} mode {mode}: lu", flush=True)
        lu, perm, dr, dc, info = gpu_solver.lu_factors(bad, mode)
        assert sorted(perm) == list(range(lu.shape[0]))
        # a column that is NaN from its diagonal down had no candidate: the pivot stayed on the diagonal
        nan = np.isnan(lu.real) | np.isnan(lu.imag)
        assert any(nan[k:, k].all() for k in range(lu.shape[0] - 1))
        print(f"nonfinite N {ny} mode {mode}: solve", flush=True)
        r, alone = gpu_solver.solve([good, bad, good], mode), gpu_solver.solve([good], mode)
        assert r.info[1] in (_lib.INFO_NOCONV, _lib.INFO_SINGULAR)
        for k in (0, 2):
            assert r.info[k] == alone.info[0] == _lib.INFO_OK
            assert np.array_equal(r.evals[k], alone.evals[0]) and np.array_equal(r.resid[k], alone.resid[0])
        for method in (_lib.LEAD_KRYLOV, _lib.LEAD_INVIT, _lib.TRACK):
            print(f"nonfinite N {ny} mode {mode}: leading method {method}", flush=True)
            a = gpu_solver.solve_leading([good, bad, good], mode, method)
            b = gpu_solver.solve_leading([good], mode, method)
            assert a["info"][1] in (_lib.INFO_NOCONV, _lib.INFO_SINGULAR)
            for k in (0, 2):
                assert a["info"][k] == b["info"][0] and a["evals"][k] == b["evals"][0]
                assert b["info"][0] in (_lib.INFO_OK, _lib.INFO_FALLBACK)
