"""E2 observables of a batch that takes more than one chunk of pairs: the second
chunk of an E2 call computed the gauge-sample pointer from a null base, so the
gauge sum stored through it.  At the pf mesh a pair needs 182 MB of scratch, the
chunk divisor 4 leaves 6 GiB: 35 pairs, then one."""
import numpy as np
import pytest

from sccm_amd import configs
from sccm_amd.operators import q2_matrices

pytestmark = pytest.mark.gpu


def test_e2_over_two_chunks_equals_one():
    from sccm_amd.pnamp import FORM_FACTORED, PNAMP
    w = configs.pf_gcm(nstates=3, jmax=2)
    g = PNAMP(w.basis, w.inter, w.mesh)
    g.set_states(w.U, w.V)
    g.set_q2(q2_matrices(w.basis))
    g.set_form(FORM_FACTORED)
    pairs = np.tile(w.pairs, (6, 1))
    assert len(pairs) == 36
    out, nodes = [], []
    for div in (1, 4):
        g.set_tune(0, 0, div)
        g.kernels_batched(pairs, w.zval, w.nval, want_kern=False)
        nodes.append(g.graph_info()[2])
        out.append(g.kernels_e2(pairs, w.zval, w.nval))
    assert nodes == [4, 8]  # setup, Pfaffian, densities, gauge sum per chunk
    for name, a, b in zip(("zres", "kern", "ze2", "qred", "rho1b"), *out):
        # the chunks differ in the pairs they hold only: the same sums in the same order
        assert np.abs(a - b).max() <= 1e-14 * np.abs(a).max(), name
        for k in range(0, 30):  # each pair as its first occurrence
            assert np.abs(b[k + 6] - b[k]).max() <= 1e-14 * np.abs(a).max(), (name, k)
    g.close()
