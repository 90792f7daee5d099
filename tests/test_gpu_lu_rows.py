"""The panel kernel of the batched LU where its rows change hands: a full last
row per thread, one row more, two and three rows per thread with 256 threads,
and the 512-thread form up to its largest order (parity unpinned: checked
against P (Dr M Dc) = L U and the pivot rule itself).

Tolerances: the factorisation error grows at most with the order, from the
1e-13 (FP64) and 1e-5 (FP32) asked at order 800; a pivot has the largest
|Re| + |Im| of its column, and |x| <= |Re x| + |Im x| <= sqrt(2) |x|, so no
multiplier exceeds sqrt(2), but for the two roundings of a reciprocal and a
product of the factor's precision.  U's rows go through explicit inverses, so
a multiplier is taken from the stored L.
"""
import numpy as np
import pytest

from conftest import golden

pytestmark = pytest.mark.gpu


def _factor(gpu_solver, ts_profile, ny, mode):
    from stab_amd import _lib, solver as sv
    text = open(golden("thesis_TStest", "temporal.inp")).read().replace("96 1.0 0.0", f"{ny} 1.0 0.0")
    gpu_solver.set_profile(0, *ts_profile)
    pt = sv.make_point(sv.read_input(text), 0.2 + 0.05j, 4)
    return gpu_solver.pencil(pt, _lib.MAT_SHIFTED), gpu_solver.lu_factors(pt, mode)


@pytest.mark.parametrize("mode,tol,eps", [(0, 1e-13, 2.0 ** -52), (1, 1e-5, 2.0 ** -23)])
@pytest.mark.parametrize("ny", [51, 52, 103, 153, 154, 205, 256])
def test_rows_per_thread(gpu_solver, ts_profile, ny, mode, tol, eps):
    print(f"lu rows ny {ny} mode {mode}", flush=True)
    M, (lu, perm, dr, dc, info) = _factor(gpu_solver, ts_profile, ny, mode)
    n, npad = M.shape[0], lu.shape[0]
    Ms = np.eye(npad, dtype=complex)
    Ms[:n, :n] = M
    Ms = dr[:, None] * Ms * dc[None, :]
    L = np.tril(lu, -1)
    assert info == 0
    assert sorted(perm) == list(range(npad))
    assert np.abs(L).max() <= np.sqrt(2) * (1 + 16 * eps)
    err = np.linalg.norm(Ms[perm] - (L + np.eye(npad)) @ np.triu(lu)) / np.linalg.norm(Ms)
    assert err < tol * max(1.0, npad / 800)
