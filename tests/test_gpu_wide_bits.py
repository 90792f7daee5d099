"""Wide and four-wave work-groups give the same results to the last bit: every
sum is formed in an order that does not depend on the work-group (Gram-Schmidt
coefficients by one wave each, norms by the first 256 threads), so the Krylov
pairs, vectors and residuals are compared as they are, in both modes, and so is
the inverse iteration with its Krylov fallback, tracked and not.  Every batch has to hold
converged pairs and directly solved points, or nothing would be compared."""
import numpy as np
import pytest

from test_gpu_wide import BATCHES, _points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", BATCHES, ids=lambda b: "-".join(f"{i}x{n}" for i, n in b))
def test_wide_is_bitwise_the_same(gpu_solver, monkeypatch, batch):
    from stab_amd import _lib
    pts, shifts, ym, vt = _points(batch)
    gpu_solver.set_profile(0, ym, vt)
    out = {}
    for wide in ("0", "1000000"):
        monkeypatch.setenv("STAB_WIDE_POINTS", wide)
        out[wide] = [gpu_solver.solve(pts, mode) for mode in (_lib.MODE_PLAIN_F64, _lib.MODE_MIXED)]
        for mode in (_lib.MODE_PLAIN_F64, _lib.MODE_MIXED):
            # near shifts are solved directly; the points' own shifts, one step only, leave the fallback to do it
            out[wide].append(gpu_solver.solve_leading(pts, mode, _lib.LEAD_INVIT, maxit=20, shifts=shifts, want_vectors=True))
            for method in (_lib.LEAD_INVIT, _lib.TRACK):
                out[wide].append(gpu_solver.solve_leading(pts, mode, method, maxit=1, want_vectors=True,
                                                          shifts=[1.2 * s for s in shifts], fallback_shifts=shifts))
    a, b = out["0"], out["1000000"]
    for x, y in zip(a[:2], b[:2]):
        assert np.array_equal(x.info, y.info) and np.array_equal(x.evals, y.evals) and np.array_equal(x.resid, y.resid)
        assert all(np.min(x.resid[p, :4]) < 1e-10 for p in range(len(pts)))
    for x, y in zip(a[2:], b[2:]):
        assert np.array_equal(x["info"], y["info"]) and np.array_equal(x["evals"], y["evals"])
        assert all(np.array_equal(u, v) for u, v in zip(x["evecs"], y["evecs"]))
    for near, far, tracked in (a[2:5], a[5:8]):
        assert np.any(near["info"] == _lib.INFO_OK)
        assert np.any(far["info"] == _lib.INFO_FALLBACK)
        assert np.any(tracked["info"] == _lib.INFO_FALLBACK)
