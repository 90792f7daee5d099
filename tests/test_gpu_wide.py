"""The wide work-groups of the iteration kernels (small batches) against the
four-wave ones: the inverse iteration bitwise, since every sum keeps its order,
and the Krylov leading modes to the residual bound; at orders whose last block
is 32 or 64 wide, the smallest and largest N, spatial and finite-difference
points, and a batch that mixes them."""
import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu

# (itype, N): n = 5 N padded to 32; 64 -> 320 (whole blocks), 96 -> 480, 81 -> 416 (a 32-wide last block)
BATCHES = [[(1, 64)], [(1, 96), (1, 81)], [(1, 12), (1, 33)], [(1, 256)], [(2, 64), (2, 128)], [(3, 101), (4, 64)],
           [(1, 48), (2, 40), (3, 50), (1, 96)]]


def _points(batch):
    import os
    from oracle import stab_oracle as so
    from stab_amd import solver as sv
    pts, shifts = [], []
    for itype, ny in batch:
        kind = "temporal" if itype in (1, 3) else "spatial"
        text = open(os.path.join(GOLDEN, "thesis_TStest", ("fd_" if itype > 2 else "") + kind + ".inp")).read()
        inp = sv.read_input(text)
        inp.ny = ny
        sh = 0.1146788 + 0.0023845j if kind == "temporal" else 0.2280474 - 0.0065163j
        pts.append(sv.make_point(inp, sh, 4))
        shifts.append(sh * (1 + 2e-3j))
    ym, vt = so.read_profile(os.path.join(GOLDEN, "TStest", "profile.0"))
    return pts, shifts, ym, vt


@pytest.mark.parametrize("batch", BATCHES, ids=lambda b: "-".join(f"{i}x{n}" for i, n in b))
def test_wide_matches_four_waves(gpu_solver, monkeypatch, batch):
    from stab_amd import _lib
    pts, shifts, ym, vt = _points(batch)
    gpu_solver.set_profile(0, ym, vt)
    out = {}
    for wide in ("0", "1000000"):
        monkeypatch.setenv("STAB_WIDE_POINTS", wide)
        out[wide] = [gpu_solver.solve_leading(pts, mode, _lib.TRACK, maxit=20, shifts=shifts, want_vectors=True)
                     for mode in (_lib.MODE_MIXED, _lib.MODE_PLAIN_F64)]
        out[wide].append(gpu_solver.solve(pts, _lib.MODE_PLAIN_F64))
    for a, b in zip(out["0"][:2], out["1000000"][:2]):
        direct = (a["info"] == _lib.INFO_OK) & (b["info"] == _lib.INFO_OK)
        assert np.array_equal(a["info"], b["info"])
        for k in np.nonzero(direct)[0]:
            assert a["evals"][k] == b["evals"][k] and a["iters"][k] == b["iters"][k]
            assert np.array_equal(a["evecs"][k], b["evecs"][k])
    a, b = out["0"][2], out["1000000"][2]
    # Gram-Schmidt sums differ in order: pairs converged on both sides agree to what their residuals fix
    for p in range(len(pts)):
        for k in range(4):
            if a.resid[p, k] < 1e-13 and b.resid[p, k] < 1e-13 and batch[p][1] >= 48:
                assert np.min(np.abs(a.evals[p, :4] - b.evals[p, k])) <= 1e-6 * abs(b.evals[p, k])
