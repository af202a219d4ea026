"""The separable projection takes as many beta nodes at a time as its LDS holds:
all of them, a last pass with fewer, one by one, and one node beyond 48 KB; more
outputs than threads, and a single Euler angle: against the sum itself."""
import numpy as np
import pytest

from sccm_amd.basis import make_basis
from sccm_amd.interaction import synthetic_interaction
from sccm_amd.mesh import make_mesh


@pytest.mark.gpu
@pytest.mark.parametrize("na,nb,ng,jmax", [(1, 10, 1, 6), (1, 1, 1, 0), (6, 7, 5, 9), (2, 3, 9, 1), (30, 3, 30, 8),
                                           (40, 2, 40, 9)])
def test_separable_projection_is_the_sum(oracle_mod, na, nb, ng, jmax):
    from sccm_amd.pnamp import PNAMP
    b = make_basis("p")
    mesh = make_mesh(na, nb, ng, 1, jmax)
    g = PNAMP(b, synthetic_interaction(b, 1.2, 101, 102), mesh)
    r = np.random.default_rng(na + nb)
    z = r.normal(size=(na * nb * ng, 6)) + 1j * r.normal(size=(na * nb * ng, 6))
    kern = g.project_zres(z[None])[0]
    K = np.arange(-jmax, jmax + 1)
    ea, eg = np.exp(1j * K[:, None] * mesh.alp) * mesh.walp, np.exp(1j * K[:, None] * mesh.gam) * mesh.wgam
    s = np.einsum("ka,bago,lg->obkl", ea, z.reshape(nb, na, ng, 6), eg, optimize=True)
    bound = np.abs(mesh.walp).sum() * np.abs(mesh.wgam).sum() * np.abs(mesh.wbet).sum() * np.abs(z).max()
    for J in range(jmax + 1):
        d = np.zeros((nb, 2 * jmax + 1, 2 * jmax + 1))
        for k1 in range(-J, J + 1):
            for k2 in range(-J, J + 1):
                d[:, jmax + k1, jmax + k2] = [oracle_mod.wigner_d(2 * J, 2 * k1, 2 * k2, be) for be in mesh.bet]
        w = (2 * J + 1) / 2.0 if na * ng == 1 else (2 * J + 1) / (8 * np.pi ** 2)
        ref = w * np.einsum("b,bkl,obkl->okl", mesh.wbet, d, s)
        # 2^-53 per term over at most na + nb + ng sequential ones, d to 1e-13
        assert np.abs(kern[:, J] - ref).max() < 2e-13 * w * bound, J
    g.close()
