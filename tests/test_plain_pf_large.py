"""The plain Pfaffian's layout at its largest size class (2n = 128: 16 x 16
threads, eight slot rows) and the sizes that fall into it, emulated on the CPU."""
import numpy as np
import pytest

from test_pf_layout import pf_ref
from test_plain_pf_layout import _skew, emulate


@pytest.mark.parametrize("n2", [100, 112, 124, 128])
def test_largest_layout_matches_explicit_exchanges(n2):
    S = _skew(n2, np.random.default_rng(n2))
    ref = pf_ref(S)
    assert abs(emulate(S, 16, 8) - ref) < 1e-11 * abs(ref)
    assert abs(emulate(S, 16, 8, "position c") - ref) > 1e-3 * abs(ref)
