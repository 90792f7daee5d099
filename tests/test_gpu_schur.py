"""The projected eigenproblem of the Krylov-Schur iteration at the edges of
its sizes (smallest and largest basis, one wanted pair and the most, a basis
that is a multiple of nothing), through a whole solve: every converged pair
against the ZGGEV spectrum of the oracle's pencil."""
import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,keep,nev", [(6, 2, 1), (17, 8, 4), (24, 12, 3), (40, 20, 8), (64, 32, 16)])
def test_krylov_sizes_match_qz(gpu_solver, monkeypatch, m, keep, nev):
    import os
    from oracle import stab_oracle as so
    from stab_amd import _lib
    from stab_amd import solver as sv
    ym, vt = so.read_profile(os.path.join(GOLDEN, "TStest", "profile.0"))
    text = open(os.path.join(GOLDEN, "thesis_TStest", "temporal.inp")).read().replace("96 1.0 0.0", "48 1.0 0.0")
    A0, B0 = so.temporal_pencil(so.setup(so.parse_input(text), ym, vt, spatial=False))
    wq, yl, xr = so.sla.eig(A0, B0, left=True, right=True, check_finite=False)
    ok = np.isfinite(wq) & (np.abs(wq) > 0)
    wq, yl, xr = wq[ok], yl[:, ok], xr[:, ok]
    # relative condition numbers: a pair of backward error r is defined to about kappa r
    kappa = (np.linalg.norm(yl, axis=0) * np.linalg.norm(xr, axis=0)
             * (np.linalg.norm(A0) + np.abs(wq) * np.linalg.norm(B0))
             / (np.abs(wq) * np.abs(np.einsum("ij,ij->j", yl.conj(), B0 @ xr))))
    monkeypatch.setenv("STAB_KS_M", str(m))
    monkeypatch.setenv("STAB_KS_KEEP", str(keep))
    monkeypatch.setenv("STAB_KS_CYCLES", "40")
    gpu_solver.set_profile(0, ym, vt)
    guess = 0.1146788 + 0.0023845j
    pt = sv.make_point(sv.read_input(text), guess, nev)
    r = gpu_solver.solve([pt, pt], _lib.MODE_PLAIN_F64)
    assert np.array_equal(r.evals[0], r.evals[1])
    found = 0
    for ev, res in zip(r.evals[0, :nev], r.resid[0, :nev]):
        if not res < 1e-10:
            continue
        j = int(np.argmin(np.abs(wq - ev)))
        assert abs(wq[j] - ev) <= max(1e-8, 10.0 * kappa[j] * (res + 1e-14)) * abs(ev)
        found += 1
    assert found >= 1 and abs(r.evals[0, 0] - (0.11467880189410 + 0.0023844535276599j)) <= 1e-7
