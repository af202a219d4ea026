"""k_fac_dens works on one gauge angle per wave for a few Euler points and on
groups of up to 64 / h angles for many: at every species size (h not a multiple
of the 4 x 4 tiles, a last group with fewer angles) the kernels of a
large batch are those of the single pair, which the oracle tests cover."""
import numpy as np
import pytest

from sccm_amd.basis import make_basis
from sccm_amd.interaction import synthetic_interaction
from sccm_amd.mesh import make_mesh
from sccm_amd.states import synthetic_state

ORBITS = {4: [(0, 1, 3)], 6: [(0, 1, 3), (0, 1, 1)], 8: [(0, 3, 7)], 10: [(0, 3, 7), (1, 1, 1)],
          12: [(0, 2, 5), (1, 0, 1), (0, 2, 3)], 14: [(0, 3, 7), (1, 1, 3), (1, 1, 1)],
          16: [(0, 3, 7), (0, 3, 5), (1, 1, 1)], 18: [(0, 3, 7), (0, 3, 5), (1, 1, 3)],
          20: [(0, 3, 7), (1, 1, 3), (0, 3, 5), (1, 1, 1)], 22: [(1, 1, 3), (0, 3, 5), (1, 1, 1), (0, 4, 9)]}


@pytest.mark.gpu
@pytest.mark.parametrize("h", list(ORBITS))
def test_grouped_angles_equal_single_ones(h):
    from sccm_amd.pnamp import FORM_FACTORED, PNAMP
    b = make_basis(f"h{h}", ORBITS[h])
    assert b.n == 2 * h
    zn = (2, 2)
    it = synthetic_interaction(b, 1.2, 301, 302)
    g = PNAMP(b, it, make_mesh(2, 2, 3, 7, 2))
    U, V = zip(*[synthetic_state(b, *zn, seed=s) for s in (71, 72)])
    g.set_states(np.array(U), np.array(V))
    g.set_form(FORM_FACTORED)
    z1, k1 = g.kernels_batched([(0, 1)], *zn, want_zres=True)   # 6 Euler points, 12 blocks of 7 angles
    zb, kb = g.kernels_batched([(0, 1)] * 180, *zn, want_zres=True)
    for i in (0, 91, 179):
        # the same sums in the same order per angle: equal to the last bits
        assert np.abs(zb[i] - z1[0]).max() <= 1e-14 * np.abs(z1[0]).max()
        assert np.abs(kb[i] - k1[0]).max() <= 1e-14 * np.abs(k1[0]).max()
    g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["none", "pp", "nn", "pn", "one"])
def test_lists_with_empty_species_parts(kind):
    """Tables without groups, of one species only, of a single tile: against the plain form."""
    from sccm_amd.interaction import Interaction
    from sccm_amd.pnamp import FORM_FACTORED, FORM_PLAIN, PNAMP
    b = make_basis("sd")
    it = synthetic_interaction(b, 1.2, 301, 302)
    h = b.n // 2
    pa, pb = it.ka <= h, it.kb <= h
    keep = {"none": pa & ~pa, "pp": pa & pb, "nn": ~pa & ~pb, "pn": pa & ~pb, "one": np.arange(it.nme) == 3}[kind]
    it = Interaction(it.ka[keep], it.kb[keep], it.kc[keep], it.kd[keep], it.me[keep], it.t1b, it.e0)
    g = PNAMP(b, it, make_mesh(2, 2, 3, 3, 2))
    U, V = zip(*[synthetic_state(b, 2, 2, seed=s) for s in (71, 72)])
    g.set_states(np.array(U), np.array(V))
    out = []
    for form in (FORM_PLAIN, FORM_FACTORED):
        g.set_form(form)
        out.append(g.kernels_batched([(0, 1)], 2, 2, want_zres=True)[0])
    assert np.abs(out[0] - out[1]).max() <= 1e-10 * np.abs(out[0]).max()  # the repository's bar for the FP64 forms
    g.close()
