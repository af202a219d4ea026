"""CPU emulation of k_plain_pf's elimination, thread by thread in its 2D
block-cyclic layout (G x G threads, vectors R, A, C that start as NaN, the two
barriers of a step as the order of whole-grid phases), against the
explicit-exchange Pfaffian, at sizes around the layouts' block edges."""
import numpy as np
import pytest

from test_pf_layout import pf_ref


def emulate(S, G, T, plant=None):
    N2 = S.shape[0]
    a, b = np.divmod(np.arange(G * G), G)
    sv = {}
    for p in range(T):
        for q in range(p, T):
            i, j = a + G * p, b + G * q
            v = np.zeros(G * G, complex)
            ok = (i < N2) & (j < N2)
            v[ok] = S[i[ok], j[ok]]
            sv[p, q] = v
    nan = np.full(G * T, np.nan + 0j)
    vR, vA, C = [nan.copy(), nan.copy()], [nan.copy(), nan.copy()], nan.copy()
    pf = 1.0 + 0j
    for P in range(T):
        for t in range(G // 2):
            r = G * P + 2 * t
            if r >= N2 - 2:
                break
            R, A = vR[t & 1], vA[t & 1]
            row, row1 = np.nonzero(a == 2 * t)[0], np.nonzero(a == 2 * t + 1)[0]
            cand = [(abs(sv[P, q][x]), -(b[x] + G * q)) for x in row for q in range(P, T) if r < b[x] + G * q < N2]
            c = -max(cand)[1]
            Q, cg = divmod(c, G)
            s = sv[P, Q][2 * t * G + cg]
            for q in range(P, T):
                R[b[row] + G * q] = sv[P, q][row] / s
                A[b[row1] + G * q] = sv[P, q][row1]
            R[c] = sv[P, P][2 * t * G + 2 * t + 1] / s
            # barrier; every thread knows c, s
            if not abs(s) ** 2 > 1e-26:
                big = any(abs(sv[p, q][x]) ** 2 > 1e-26 for p in range(P, T) for q in range(p, T)
                          for x in range(G * G) if a[x] + G * p >= r and a[x] + G * p < b[x] + G * q < N2)
                if not big or not abs(s) ** 2 > 1e-290:
                    return 0j
            swap = c != r + 1
            pf *= -s if swap else s
            cb, ca = np.nonzero(b == cg)[0], np.nonzero(a == cg)[0]
            for pp in range(P, Q + 1):
                x = a[cb] + G * pp
                C[x] = np.where((x == c) & (plant != "position c"), A[c], sv[pp, Q][cb])
            for q in range(Q + 1, T):
                C[b[ca] + G * q] = -sv[Q, q][ca]
            if swap:
                for pp in range(P, Q + 1):
                    sv[pp, Q][cb] = -A[a[cb] + G * pp]
                for q in range(Q, T):
                    sv[Q, q][ca] = A[b[ca] + G * q]
            # barrier
            for pp in range(P, T):
                for q in range(pp, T):
                    i, j = a + G * pp, b + G * q
                    sv[pp, q] = sv[pp, q] - C[i] * R[j] + R[i] * C[j]
    return pf * sv[(N2 - 2) // G, (N2 - 1) // G][((N2 - 2) % G) * G + (N2 - 1) % G]


def _skew(n2, rng):
    m = rng.normal(size=(n2, n2)) + 1j * rng.normal(size=(n2, n2))
    return m - m.T


@pytest.mark.parametrize("G,T,n2", [(8, 4, 16), (8, 4, 28), (8, 6, 36), (8, 6, 48), (16, 4, 52), (16, 4, 64),
                                    (16, 5, 68), (16, 5, 80), (16, 6, 88)])
def test_layout_matches_explicit_exchanges(G, T, n2):
    rng = np.random.default_rng(n2)
    for _ in range(2):
        S = _skew(n2, rng)
        ref = pf_ref(S)
        assert abs(emulate(S, G, T) - ref) < 1e-11 * abs(ref)
        assert abs(emulate(S, G, T, "position c") - ref) > 1e-3 * abs(ref)  # the emulation sees a planted mistake


def test_small_pivots():
    """A row with nothing above 1e-13 ends the elimination only if no other
    entry is larger (ZPfaffianF's rule on the whole remaining matrix)."""
    rng = np.random.default_rng(5)
    S = _skew(16, rng)
    S[:2] *= 1e-14
    S[:, :2] *= 1e-14
    ref = pf_ref(S)
    assert ref != 0 and abs(emulate(S, 8, 4) - ref) < 1e-11 * abs(ref)
    assert emulate(1e-14 * _skew(16, rng), 8, 4) == 0
    S[0] = 0
    S[:, 0] = 0
    assert emulate(S, 8, 4) == 0
