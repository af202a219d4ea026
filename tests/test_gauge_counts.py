"""The factored and mixed forms at the gauge counts whose gauge sum evaluates the
most angles (odd counts above eight: eleven and more take the wide variants, 15
the most LDS), against the plain form, at the smallest and the largest species."""
import numpy as np
import pytest

from sccm_amd.basis import make_basis
from sccm_amd.interaction import synthetic_interaction
from sccm_amd.mesh import make_mesh
from sccm_amd.states import synthetic_state

ORBITS = {4: [(0, 1, 3)], 12: [(0, 2, 5), (1, 0, 1), (0, 2, 3)], 22: [(1, 1, 3), (0, 3, 5), (1, 1, 1), (0, 4, 9)]}


@pytest.mark.gpu
@pytest.mark.parametrize("h", list(ORBITS))
@pytest.mark.parametrize("nphi", [9, 10, 11, 13, 14, 15])
def test_forms_agree_at_large_gauge_counts(h, nphi):
    from sccm_amd.pnamp import FORM_FACTORED, FORM_MIXED_FP32, FORM_PLAIN, PNAMP
    b = make_basis(f"h{h}", ORBITS[h])
    U, V = zip(*[synthetic_state(b, 2, 2, seed=s) for s in (71, 72)])
    for na in (1, 2):  # axial (half of the angles), triaxial
        g = PNAMP(b, synthetic_interaction(b, 1.2, 301, 302), make_mesh(na, 2, na, nphi, 2))
        g.set_states(np.array(U), np.array(V))
        ref = None
        # the repository's bars: FP64 forms 1e-10, FP32 contraction 2^-24 per term
        for form, rel in ((FORM_PLAIN, 0.0), (FORM_FACTORED, 1e-10), (FORM_MIXED_FP32, 1e-5)):
            g.set_form(form)
            z = g.kernels_batched([(0, 1), (1, 1)], 2, 2, want_zres=True)[0]
            if ref is None:
                ref = z
            for io in range(z.shape[-1]):
                assert np.abs(z[..., io] - ref[..., io]).max() <= rel * np.abs(ref[..., io]).max(), (na, form, io)
        g.close()
