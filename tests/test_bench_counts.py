"""The benchmark's operation counts name what the kernels evaluate, and its HBM
bytes the Pfaffian route that ran."""
import json
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("nphi", range(1, 17))
def test_gauge_pairs_of_the_plain_form(nphi):
    """Classes of (phi_p, phi_n) under the shift of both angles by pi, counted one by one."""
    seen = set()
    n = 0
    for a in range(nphi):
        for b in range(nphi):
            if (a, b) in seen:
                continue
            n += 1
            seen.add((a, b))
            if nphi % 2 == 0:
                seen.add(((a + nphi // 2) % nphi, (b + nphi // 2) % nphi))
    assert bench.plain_gauge_pairs(nphi) == n


def test_traffic_is_the_measured_route():
    t = json.load(open(os.path.join(ROOT, "profiles", "traffic.json")))
    for schur in (False, True):
        for form in ("factored_fp64", "mixed_fp32", "mixed_bf16"):
            e = t.get(form + ("_schur" if schur else ""))
            b = bench.traffic_per_launch(form, 210, schur)
            assert (b is None) == (e is None)
            if e is not None:
                assert e["pfaffian"] == ("h x h" if schur else "2h x 2h")
                assert b == 1024.0 * 210 / e["pairs_per_launch"] * (
                    e["fetch_kib_per_launch"] * e["fetch_factor"] + e["write_kib_per_launch"] * e["write_factor"])
    assert bench.traffic_per_launch("plain_fp64", 1) is None or "plain_fp64" in t
