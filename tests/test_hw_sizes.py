"""Hill-Wheeler eigensolver and natural-state scan at the sizes where their
routes change (the matrix in LDS, one launch per
rotation step), odd and even, against numpy in 64 bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
# an eigenvalue of a backward stable symmetric solver: a few dim ulp of the norm
TOL = 1e-12


def _ctx():
    from sccm_amd.basis import make_basis
    from sccm_amd.interaction import synthetic_interaction
    from sccm_amd.mesh import make_mesh
    from sccm_amd.pnamp import PNAMP
    b = make_basis("p")
    return PNAMP(b, synthetic_interaction(b, 1.0, 1, 2), make_mesh(1, 2, 1, 1, 0))


def _case(dim):
    r = np.random.default_rng(dim)
    q, _ = np.linalg.qr(r.normal(size=(dim, dim)))
    n = (q * np.linspace(1.0, 0.05, dim)) @ q.T  # every natural state above the cutoff
    h = r.normal(size=(dim, dim))
    h = 0.5 * (h + h.T)
    return 0.5 * (n + n.T), h


@pytest.mark.parametrize("dim", [1, 2, 3, 20, 63, 64, 113, 114, 115, 129, 192, 193, 199, 200, 201, 202, 237])
def test_hw_solve_and_presolve_sizes(dim):
    n, h = _case(dim)
    g = _ctx()
    r = g.hw_solve(n, h, 1e-6)
    w, v = np.linalg.eigh(n)
    w, v = w[::-1], v[:, ::-1]
    R = v / np.sqrt(w)
    G = R.T @ h @ R
    e = np.linalg.eigvalsh(0.5 * (G + G.T))
    scale = np.abs(e).max()
    assert r["ifl"] == 0 and r["m"] == dim
    assert np.abs(r["EN"] - w).max() < TOL
    assert np.abs(r["E"] - e).max() < TOL * scale * 20  # 1 / EN_min amplifies the rounding of N
    F = r["F"]
    assert np.abs(F.T @ n @ F - np.eye(dim)).max() < TOL * 20
    assert np.abs(h @ F - (n @ F) * r["E"]).max() < 20 * TOL * scale * np.abs(F).max()
    s = g.hw_presolve(n, h, 1e-6, 3)
    assert s["m"] == dim
    for nos in (x for x in sorted({1, 2, dim // 2, dim - 1, dim}) if 1 <= x <= dim):
        ee = np.linalg.eigvalsh(0.5 * (G + G.T)[:nos, :nos])[:3]
        assert np.abs(s["E"][nos - 1, :len(ee)] - ee).max() < TOL * scale * 20, nos
    # at all natural states the levels are exact solutions: no variance
    assert s["var"][-1].max() < (TOL * scale * 20 * np.abs(F).max()) ** 2 * dim
    g.close()
