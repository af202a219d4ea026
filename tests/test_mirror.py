"""Mirrored Euler points and repeated gauge angles: the forms evaluate one of
two points (alpha, gamma) and (2 pi - alpha, 2 pi - gamma), one of two gauge
angles phi, phi + pi, and on axial meshes one of phi, -phi; every form against
the oracle, which evaluates all of them, over the meshes where the pairing
differs (all points paired, a point that is its own mirror among others,
axial, one direction not symmetric, an angle twice) and gauge counts 1 .. 6."""
import numpy as np
import pytest

from sccm_amd.basis import make_basis
from sccm_amd.interaction import synthetic_interaction
from sccm_amd.mesh import make_mesh
from sccm_amd.states import bogoliubov_from_generator, slater_occupations, synthetic_state

REL = 1e-10  # the repository's bar for the FP64 forms (normwise per observable)
ZN = (2, 4)


def _mesh(kind, nphi):
    if kind == "paired":
        return make_mesh(2, 2, 4, nphi, 2)
    if kind == "centre":  # alpha = gamma = pi is its own mirror
        return make_mesh(3, 2, 3, nphi, 2)
    if kind == "axial":
        return make_mesh(1, 3, 1, nphi, 2)
    if kind == "gamma_only":  # alpha = 0 is its own mirror
        return make_mesh(1, 2, 3, nphi, 2)
    m = make_mesh(3, 2, 2, nphi, 2)
    if kind == "shifted":
        m.gam = m.gam + 0.1
    if kind == "twice":
        m.alp = np.array([1.0, 1.0, 2.0 * np.pi - 1.0])
    return m


def _states(b, pn):
    if not pn:
        s = [synthetic_state(b, *ZN, seed=k) for k in (31, 32)]
    else:
        s = []
        for k in (31, 32):
            r = np.random.default_rng(k)
            sk = lambda w: (lambda a: a - a.T)(np.triu(r.normal(0.0, w, (b.n, b.n)), 1))
            s.append(bogoliubov_from_generator(b, sk(0.2), sk(0.1), slater_occupations(b, *ZN)))
    return np.array([x[0] for x in s]), np.array([x[1] for x in s])


def _oracle(oracle_mod, b, it, mesh, U, V):
    return oracle_mod.Oracle(b, it, mesh, *ZN).kernel_pair(U[0], V[0], U[1], V[1])


def test_mirrored_points_are_conjugates(oracle_mod):
    """The identity itself, on the oracle (CPU)."""
    b = make_basis("p")
    it = synthetic_interaction(b, 1.2, 101, 102)
    for pn in (False, True):
        U, V = _states(b, pn)
        for kind in ("paired", "centre", "axial"):
            mesh = _mesh(kind, 3)
            zr, _ = _oracle(oracle_mod, b, it, mesh, U, V)
            z = zr.reshape(mesh.bet.size, mesh.alp.size, mesh.gam.size, -1)
            assert np.abs(z[:, ::-1, ::-1].conj() - z).max() < REL * np.abs(z).max(), (pn, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("nphi", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("kind", ["paired", "centre", "axial", "gamma_only", "shifted", "twice"])
def test_forms_match_oracle_on_mirrored_meshes(oracle_mod, kind, nphi):
    from sccm_amd.pnamp import FORM_FACTORED, FORM_MIXED_FP32, FORM_PLAIN, PNAMP
    b = make_basis("p")
    it = synthetic_interaction(b, 1.2, 101, 102)
    mesh = _mesh(kind, nphi)
    for pn, form, rel in ((True, FORM_PLAIN, REL), (False, FORM_PLAIN, REL), (False, FORM_FACTORED, REL),
                          (False, FORM_MIXED_FP32, 1e-5)):  # FP32 contraction: 2^-24 per term
        U, V = _states(b, pn)
        g = PNAMP(b, it, mesh)
        g.set_states(U, V)
        g.set_form(form)
        zr, kern = g.kernel_pair(0, 1, *ZN, want_zres=True)
        zo, ko = _oracle(oracle_mod, b, it, mesh, U, V)
        for io in range(6):
            assert np.abs(zr[:, io] - zo[:, io]).max() < rel * np.abs(zo[:, io]).max(), (pn, form, io)
            assert np.abs(kern[io] - ko[io]).max() < rel * np.abs(ko[io]).max(), (pn, form, io)
        if form == FORM_FACTORED:  # every gauge point, also those given by symmetry, sums to ZRES
            s = g.mesh_samples([(0, 1)], *ZN)[0]
            n, ne = s[..., 0].mean((1, 2)), (s[..., 0] * s[..., 1]).mean((1, 2))
            assert np.abs(n - zr[:, 0]).max() < 1e-12 * np.abs(zr[:, 0]).max()
            assert np.abs(ne - zr[:, 4]).max() < 1e-12 * np.abs(zr[:, 4]).max()
        g.close()
