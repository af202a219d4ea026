"""The workspace that the Hill-Wheeler calls leave with a context is bounded in
all, whatever sizes were called: a scan over 480 natural states takes 0.5 GB of
rotation log and 0.6 GB of matrices, of which 640 MiB may stay."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEEP = 640 << 20
SLACK = 32 << 20  # the runtime's own allocations are made in blocks of a few MiB


def _free_bytes():
    from sccm_amd.pnamp import load_library
    a, b = C.c_size_t(), C.c_size_t()
    # (found through the library's own HIP runtime)
    assert load_library().hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def test_context_keeps_a_bounded_workspace():
    from test_hw_sizes import _case, _ctx
    g = _ctx()
    n, h = _case(20)
    g.hw_solve(n, h, 1e-6)  # everything that a first call sets up
    g.hw_presolve(n, h, 1e-6, 3)
    before = _free_bytes()
    ref = None
    for dim in (60, 480, 60):
        n, h = _case(dim)
        s = g.hw_presolve(n, h, 1e-6, 3)
        assert before - _free_bytes() <= KEEP + SLACK, dim
        if dim == 60:
            assert ref is None or np.array_equal(ref["E"], s["E"])
            ref = s
    g.close()
    assert before - _free_bytes() <= SLACK
