"""Measured cases of the PNAMP projected-kernel framework: what its users run.

A case is one call chain through the public Python front end (``PNAMP``,
``MLP``), on this repository's model spaces with its seeded states and
interactions: projected kernels of one or many pairs of HFB states in each
evaluation form, the E2 observables, the Hill-Wheeler step on projected norm
and Hamiltonian matrices, and the surrogate network.  ``exact`` recomputes the
outputs in 64 bits with plain torch and numpy from the inputs alone.
"""
from __future__ import annotations

import math
from functools import lru_cache

import numpy as np
import torch

from sccm_amd.basis import make_basis
from sccm_amd.configs import gcm_grid, make_states
from sccm_amd.interaction import synthetic_interaction
from sccm_amd.mesh import make_mesh
from sccm_amd.operators import q2_matrices
from sccm_amd.pnamp import FORM_FACTORED, FORM_MIXED_BF16, FORM_MIXED_FP32, FORM_PLAIN, PNAMP
from sccm_amd.states import bogoliubov_from_generator, slater_occupations
from sccm_amd.surrogate import MLP

FORMS = {"plain": FORM_PLAIN, "factored": FORM_FACTORED, "mixed-fp32": FORM_MIXED_FP32, "mixed-bf16": FORM_MIXED_BF16}
# (TBME width in MeV, interaction seeds) per space; sd and pf are the benchmark's
INTER = {"sd": (1.5, 1001, 1002), "pf": (1.2, 1011, 1012), "f5pg9": (1.5, 1031, 1032), "sdpf": (1.2, 1041, 1042)}


def _kernels(name, space, form, nstates, mesh, zval, nval, jmax=8, pairs=0, mixed_pn=False, schur=False,
             out="kern", zn=False):
    """pairs = 0: all q <= q'; out: kern, zres+kern, or e2."""
    return {"name": name, "kind": "kernels", "space": space, "form": form, "nstates": nstates, "nalp": mesh[0],
            "nbet": mesh[1], "ngam": mesh[2], "nphi": mesh[3], "jmax": jmax, "zval": zval, "nval": nval,
            "pairs": pairs, "mixed_pn": mixed_pn, "schur": schur, "out": out, "zn": zn}


def listed():
    return [
        # one pair of an axial sd calculation, the smallest call: latency and launches
        _kernels("pair_sd_axial", "sd", "factored", 2, (1, 10, 1, 7), 2, 2, jmax=6, pairs=1, out="zres+kern"),
        # one pair on the triaxial sd mesh in the general form (the drop-in's default form)
        _kernels("pair_sd_plain", "sd", "plain", 1, (8, 16, 8, 7), 2, 2, out="zres+kern"),
        # axial GCM of states with proton-neutron mixing, as constrained HFB gives them
        _kernels("axial_pf_plain", "pf", "plain", 8, (1, 12, 1, 9), 2, 4, mixed_pn=True),
        # triaxial pairs of proton-neutron mixed states, f5pg9 (n = 44, the Ge isotopes' space)
        _kernels("triaxial_f5pg9_plain", "f5pg9", "plain", 2, (6, 7, 6, 7), 4, 4, jmax=6, pairs=2, mixed_pn=True),
        # the largest space (sd-pf, n = 64), a few axial pairs
        _kernels("axial_sdpf_plain", "sdpf", "plain", 3, (1, 9, 1, 5), 4, 6, jmax=6, pairs=5, mixed_pn=True),
        # the benchmark GCM: 20 pf states, all 210 pairs, its default Pfaffian route; the largest
        _kernels("gcm_pf_factored", "pf", "factored", 20, (10, 20, 10, 9), 2, 4, schur=True),
        # a smaller pf GCM at the drop-in's accuracy (2h x 2h Pfaffian), Euler-point sums kept
        _kernels("gcm_pf_exact", "pf", "factored", 5, (10, 20, 10, 9), 2, 4, out="zres+kern"),
        # uneven batch of GCM instances in f5pg9, valence numbers per pair
        _kernels("batch_f5pg9_zn", "f5pg9", "factored", 7, (9, 14, 9, 8), 2, 4, zn=True),
        # split-BF16 contraction on the matrix units
        _kernels("gcm_pf_mixed", "pf", "mixed-bf16", 5, (8, 16, 8, 9), 2, 4, schur=True),
        # E2 observables of an sd GCM
        _kernels("e2_sd", "sd", "factored", 6, (8, 12, 8, 7), 2, 4, jmax=6, out="e2"),
        # Hill-Wheeler step of one J block (20 configurations x 2J + 1 values of K, J = 4):
        # natural-state selection, then the levels at the chosen number of natural states
        {"name": "hill_wheeler", "kind": "hw", "nconf": 20, "nk": 9, "decay": 0.22, "eps": 1e-6, "kmax": 3},
        # the surrogate network: two epochs of training, then inference on a mesh
        {"name": "surrogate", "kind": "mlp", "width": 128, "hidden": 3, "ntrain": 20000, "batch": 4096, "epochs": 2,
         "npredict": 162000},
    ]


def draw(rng):
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["plain", "plain", "factored", "factored", "factored", "mixed", "e2", "hw", "hw", "mlp"])
    if kind == "hw":
        return {"kind": "hw", "nconf": log_int(4, 20), "nk": 2 * rng.randint(0, 5) + 1,
                "decay": rng.uniform(0.12, 0.4), "eps": 1e-6, "kmax": rng.randint(1, 5)}
    if kind == "mlp":
        return {"kind": "mlp", "width": 32 * rng.randint(1, 6), "hidden": rng.randint(1, 4),
                "ntrain": log_int(2000, 60000), "batch": rng.choice([1000, 2048, 4096]), "epochs": rng.randint(1, 2),
                "npredict": log_int(1000, 300000)}
    zval, nval = 2 * rng.randint(1, 2), 2 * rng.randint(1, 3)
    nphi, jmax = rng.randint(5, 12), rng.randint(3, 8)
    if kind == "plain":
        space = rng.choice(["sd", "pf", "f5pg9", "sdpf"])
        budget = {"sd": 160000, "pf": 60000, "f5pg9": 50000, "sdpf": 8000}[space]  # mesh points
    else:
        space = rng.choice(["sd", "pf", "f5pg9"])
        budget = 4000000
    mixed_pn = kind == "plain" and rng.random() < 0.7
    axial = rng.random() < 0.4
    nbet = rng.randint(6, 20)
    na, ng = (1, 1) if axial else (rng.randint(4, 10), rng.randint(4, 10))
    while na * nbet * ng * nphi * nphi > budget:  # the larger spaces are run on coarser meshes
        na, nbet, ng, nphi = max(1, na - (na > 4)), max(6, nbet - 1), max(1, ng - (ng > 4)), max(5, nphi - 1)
        if (nbet, nphi) == (6, 5) and max(na, ng) <= 4:
            break
    points = na * nbet * ng * nphi * nphi
    npairs = max(1, min(210, log_int(1, max(1, budget // points) + 1)))
    nstates = 1
    while nstates * (nstates + 1) // 2 < npairs:
        nstates += 1
    form = kind if kind in ("plain", "factored") else (rng.choice(["mixed-fp32", "mixed-bf16"]) if kind == "mixed"
                                                       else rng.choice(["plain", "factored"]))
    if kind == "e2" and form == "plain":
        npairs = min(npairs, max(1, {"sd": 160000, "pf": 60000, "f5pg9": 50000}[space] // points))
    c = _kernels("", space, form, nstates, (na, nbet, ng, nphi), zval, nval, jmax, npairs, mixed_pn,
                 kind != "plain" and rng.random() < 0.5, "e2" if kind == "e2" else rng.choice(["kern", "zres+kern"]),
                 kind == "factored" and rng.random() < 0.3)
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs
@lru_cache(maxsize=None)
def _interaction(space):
    return synthetic_interaction(make_basis(space), *INTER[space])


def _states(case, seed):
    b = make_basis(case["space"])
    z, n = case["zval"], case["nval"]
    ns = case["nstates"]
    if not case["mixed_pn"]:
        return make_states(b, z, n, gcm_grid(ns), seed=2000 + seed)
    # the same recipe without the species blocks: real generators that mix
    # protons and neutrons, a smooth offset between the configurations
    rng = np.random.default_rng(7000 + seed)

    def skew(sigma):
        a = np.triu(rng.normal(0.0, sigma, size=(b.n, b.n)), 1)
        return a - a.T

    X, Y, Xc, Yc = skew(0.2), skew(0.04), skew(0.2), skew(0.04)
    occ = slater_occupations(b, z, n)
    Us, Vs = [], []
    for q in range(ns):
        t = 0.5 * q / max(1, ns - 1)
        U, V = bogoliubov_from_generator(b, X + t * Xc, Y + t * Yc, occ)
        Us.append(U)
        Vs.append(V)
    return np.array(Us), np.array(Vs)


def _pairs(case):
    ns = case["nstates"]
    pairs = np.array([(q, r) for q in range(ns) for r in range(q, ns)], dtype=np.int32)
    return pairs[-case["pairs"]:] if case["pairs"] else pairs


def _valence(case, npairs):
    """Valence numbers per pair of an uneven batch: instances of ten pairs."""
    k = np.arange(npairs) // 10
    return (np.full(npairs, case["zval"]) + 2 * (k % 2)).astype(np.int32), \
        (np.full(npairs, case["nval"]) + 2 * ((k // 2) % 2)).astype(np.int32)


def _mesh(case):
    return make_mesh(case["nalp"], case["nbet"], case["ngam"], case["nphi"], case["jmax"])


def _hw_matrices(case, seed):
    """Norm and Hamiltonian of one J block as projected overlaps make them:
    smooth in the coordinates of the configurations, so the norm spectrum
    falls off over many decades."""
    rng = np.random.default_rng(9000 + seed)
    x = rng.uniform(-1.0, 1.0, size=(case["nconf"], 2))
    g = np.exp(-((x[:, None] - x[None]) ** 2).sum(-1) / (2.0 * case["decay"]))
    k = np.arange(case["nk"])
    gk = np.exp(-0.8 * np.abs(k[:, None] - k[None]))
    N = np.kron(g, gk)
    dim = N.shape[0]
    a = rng.normal(size=(dim, dim))
    L = np.linalg.cholesky(N + 1e-10 * np.eye(dim))
    H0 = -20.0 * np.eye(dim) + 1.5 * (a + a.T) / math.sqrt(2.0 * dim)
    H = L @ H0 @ L.T
    return N, 0.5 * (H + H.T)


def _mlp_data(case, seed):
    rng = np.random.default_rng(5000 + seed)
    n = max(case["ntrain"], case["npredict"])
    X = rng.normal(size=(n, 14)).astype(np.float32)
    Wt = rng.normal(size=(14, 5)) / math.sqrt(14.0)
    Y = np.sin(X[:case["ntrain"]].astype(np.float64) @ Wt).astype(np.float32)
    return X, Y


def prepare(case, seed):
    if case["kind"] == "hw":
        ctx = PNAMP(make_basis("sd"), _interaction("sd"), make_mesh(1, 4, 1, 3, 2))
        N, H = _hw_matrices(case, seed)
        return {"case": case, "ctx": ctx, "N": N, "H": H}
    if case["kind"] == "mlp":
        X, Y = _mlp_data(case, seed)
        net = MLP([14] + [case["width"]] * case["hidden"] + [5], seed=seed)
        net.set_data(X[:case["ntrain"]], Y)
        return {"case": case, "net": net, "start": net.get_params(), "X": X[:case["npredict"]]}
    ctx = PNAMP(make_basis(case["space"]), _interaction(case["space"]), _mesh(case))
    ctx.set_states(*_states(case, seed))
    ctx.set_form(FORMS[case["form"]])
    if case["form"] != "plain":
        ctx.set_schur_pfaffian(case["schur"])
    if case["out"] == "e2":
        ctx.set_q2(q2_matrices(make_basis(case["space"]), 1.0))
    pairs = _pairs(case)
    return {"case": case, "ctx": ctx, "pairs": pairs, "zn": _valence(case, len(pairs))}


def run(state):
    case = state["case"]
    if case["kind"] == "hw":
        ctx, N, H = state["ctx"], state["N"], state["H"]
        sel = ctx.hw_presolve(N, H, case["eps"], case["kmax"])
        lev = ctx.hw_solve(N, H, case["eps"], nos=int(sel["nos"][0]), want_f=False)
        return {"EN": sel["EN"], "E_nos": sel["E"], "e_best": sel["e_best"], "E": lev["E"]}
    if case["kind"] == "mlp":
        net = state["net"]
        net.set_params(state["start"])
        loss = net.train(case["epochs"], case["batch"], 2e-3, 0.96, 1)
        return {"loss": loss, "params": net.get_params(), "Y": net.predict(state["X"], bf16=True)}
    ctx, pairs, z, n = state["ctx"], state["pairs"], case["zval"], case["nval"]
    if case["out"] == "e2":
        return list(ctx.kernels_e2(pairs, z, n))
    want = case["out"] == "zres+kern"
    if case["zn"]:
        return ctx.kernels_batched_zn(pairs, *state["zn"], want_zres=want)
    if len(pairs) == 1:
        return ctx.kernel_pair(pairs[0, 0], pairs[0, 1], z, n, want_zres=want)
    return ctx.kernels_batched(pairs, z, n, want_zres=want)


# ---------------------------------------------------------------- work
def work(case):
    if case["kind"] == "hw":
        dim = case["nconf"] * case["nk"]
        # two symmetric eigenproblems with vectors (9 n^3) and the reduction
        return {"bytes": 8 * (2 * dim * dim + dim * (2 + case["kmax"])), "flops": 22 * dim ** 3}
    if case["kind"] == "mlp":
        sz = [14] + [case["width"]] * case["hidden"] + [5]
        mm = sum(2 * a * b for a, b in zip(sz, sz[1:]))
        npar = sum((a + 1) * b for a, b in zip(sz, sz[1:]))
        steps = case["epochs"] * case["ntrain"]
        return {"bytes": 4 * (19 * case["ntrain"] + 2 * npar + 19 * case["npredict"]),
                "flops": 3 * mm * steps + mm * case["npredict"]}
    b, it = make_basis(case["space"]), _interaction(case["space"])
    n, h, jm = b.n, b.n // 2, case["jmax"]
    npairs, f = len(_pairs(case)), case["nphi"]
    ne = case["nalp"] * case["nbet"] * case["ngam"]
    # the states are real, so the points (alpha, gamma, phi) and (-alpha,
    # -gamma, -phi) are complex conjugates: half of the points stand for all
    units = npairs * ne / 2
    if case["form"] == "plain":
        # per gauge point: Pfaffian 2n x 2n, T^-1 on 2n right-hand sides,
        # densities, the regrouped list; per Euler point the products
        per = f * f * ((32 / 3 + 56 / 3 + 12) * n ** 3 + 26.0 * it.nme) + 8 * n ** 3
    else:
        same = (b.t[it.ka - 1] == b.t[it.kb - 1]).sum()
        pf = (4 / 3 if case["schur"] else 32 / 3) * h ** 3
        per = 2 * (f * (pf + (56 / 3 + 12) * h ** 3 + 13.0 * same) + 8 * h ** 3) \
            + 4 * f * (it.nme - same) + 8 * f * f * h * h
    kern = 6 * (jm + 1) * (2 * jm + 1) ** 2
    out = kern + (6 * ne if case["out"] != "kern" else 0)
    if case["out"] == "e2":
        out += 10 * ne + 10 * (jm + 1) * (2 * jm + 5) * (2 * jm + 1)
    return {"bytes": 8 * 2 * n * n * case["nstates"] + 24 * it.nme + 16 * npairs * out, "flops": float(per * units)}


# ---------------------------------------------------------------- exact values
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _skew_pfaffian(S):
    """Pfaffian of a batch [B, m, m] of skew matrices (overwritten):
    elimination with the largest entry of the row as pivot."""
    B, m, _ = S.shape
    ar = torch.arange(B, device=S.device)
    pf = torch.ones(B, dtype=S.dtype, device=S.device)
    for k in range(0, m - 1, 2):
        c = S[:, k, k + 1:].abs().argmax(1) + k + 1
        row = S[ar, c].clone()
        S[ar, c] = S[:, k + 1]
        S[:, k + 1] = row
        col = S[ar, :, c].clone()
        S[ar, :, c] = S[:, :, k + 1]
        S[:, :, k + 1] = col
        p = S[:, k, k + 1].clone()
        pf = pf * torch.where(c == k + 1, p, -p)
        if k + 2 < m:
            u, v = S[:, k, k + 2:], S[:, k + 1, k + 2:] / p[:, None]
            S[:, k + 2:, k + 2:] += v[:, :, None] * u[:, None, :] - u[:, :, None] * v[:, None, :]
    return pf


def _solve_right(W, T):
    """W T^-1 for batches [B, r, n], [B, n, n]: column elimination with row
    pivots on the stacked matrix."""
    M = torch.cat([T, W], 1)
    B, _, n = M.shape
    ar = torch.arange(B, device=M.device)
    for k in range(n):
        c = M[:, k, k:].abs().argmax(1) + k
        col = M[ar, :, c].clone()
        M[ar, :, c] = M[:, :, k]
        M[:, :, k] = col / col[:, k, None]
        f = M[:, k].clone()
        f[:, k] = 0.0
        M -= M[:, :, k, None] * f[:, None, :]
    return M[:, n:]


class _Exact:
    """Mesh-point quantities of one state pair on a set of single-particle
    states (a species, or all of them)."""

    def __init__(self, case, idx):
        b, it = make_basis(case["space"]), _interaction(case["space"])
        dev = _dev()
        self.idx, self.n, self.dev = idx, len(idx), dev
        m, n = self.n, b.n
        tw, tj, orb = b.twom[idx] / 2.0, b.twoj[idx] / 2.0, b.orbit[idx] + 100 * b.t[idx]
        same = orb[:, None] == orb[None]
        jp = np.where(same & (np.abs(tw[:, None] - tw[None] - 1) < 0.1),
                      np.sqrt(np.maximum(tj * (tj + 1) - tw * (tw + 1), 0.0))[None], 0.0)
        t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.complex128, device=dev)
        self.jz, self.jx, self.jk = t(np.diag(tw)), t(0.5 * (jp + jp.T)), t(0.5 * (jp - jp.T))
        self.jj = t(tj * (tj + 1))
        self.m, self.same = tw, same
        # small d matrices of the rotation: exp(-i beta J_y), J_y = (J_+ - J_-) / 2i
        self.wy, self.vy = np.linalg.eigh((jp - jp.T) / 2j)
        self.t1 = t(it.t1b[np.ix_(idx, idx)])
        # the eight-term list sum as two bilinear forms, rho W rho + A01 Q A10
        loc = np.full(n, -1)
        loc[idx] = np.arange(m)
        a, bb, c, d = (loc[x - 1] for x in (it.ka, it.kb, it.kc, it.kd))
        keep = (a >= 0) & (bb >= 0) & (c >= 0) & (d >= 0)
        cross = keep & (it.ka + it.kb != it.kc + it.kd)
        W, Q = np.zeros((m * m, m * m)), np.zeros((m * m, m * m))
        for sel, (i, j, k, l) in ((keep, (a, bb, c, d)), (cross, (c, d, a, bb))):
            i, j, k, l, v = i[sel], j[sel], k[sel], l[sel], it.me[sel]
            np.add.at(W, (k * m + i, l * m + j), v)
            np.add.at(W, (l * m + i, k * m + j), -v)
            np.add.at(Q, (i * m + j, k * m + l), 0.25 * v)
        self.W = torch.tensor(W, device=dev)
        self.Q = torch.tensor(Q, device=dev)

    def rotation(self, al, be, ga):
        d = ((self.vy * np.exp(-1j * be[:, None, None] * self.wy)) @ self.vy.conj().T).real
        R = np.exp(-1j * al[:, None, None] * self.m[:, None]) * d * np.exp(-1j * ga[:, None, None] * self.m[None])
        return torch.tensor(R, device=self.dev)

    def points(self, U0, V0, U1, V1, R, ph):
        """R [B, n, n], ph [B, n] = e^{i phi} per state: Pfaffian, rho and the
        energy, trace and J^2 parts."""
        t = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.complex128, device=self.dev)
        n = self.n
        Z0, Z1 = V0 @ np.linalg.inv(U0), V1 @ np.linalg.inv(U1)
        A = ph[:, :, None] * R
        B = A.shape[0]
        S = torch.zeros(B, 2 * n, 2 * n, dtype=torch.complex128, device=self.dev)
        S[:, :n, :n] = (A @ t(Z1)) @ A.transpose(1, 2).contiguous()
        S[:, :n, n:] = -torch.eye(n, dtype=torch.complex128, device=self.dev)
        S[:, n:, :n] = torch.eye(n, dtype=torch.complex128, device=self.dev)
        S[:, n:, n:] = -t(Z0)
        pf = _skew_pfaffian(S)
        del S
        AV, AU = A @ t(V1), A.conj() @ t(U1)
        T = t(V0.T) @ AV + t(U0.T) @ AU
        W = _solve_right(torch.cat([AV, AU], 1), T)
        rho, k10, k01 = W[:, :n] @ t(V0.T), W[:, :n] @ t(U0.T), -(W[:, n:] @ t(V0.T))
        a01, a10 = k01 - k01.transpose(1, 2), k10 - k10.transpose(1, 2)
        e2 = self._bilinear(rho, self.W, rho) + self._bilinear(a01, self.Q, a10)
        tr = lambda M, X: (M.T.contiguous()[None] * X).sum((1, 2))
        two = lambda M, s: s * ((M @ rho) * (M @ rho).transpose(1, 2)).sum((1, 2))
        kap = lambda M: ((M @ k10 @ M) * k01).sum((1, 2))
        aj = (self.jj * rho.diagonal(dim1=1, dim2=2)).sum(1) - two(self.jz, 1) - two(self.jx, 1) - two(self.jk, -1) \
            + kap(self.jz) + kap(self.jx) + kap(self.jk)
        ts = torch.stack([tr(self.jz, rho), tr(self.jx, rho), tr(self.jk, rho)], 1)
        return {"pf": pf, "rho": rho, "e2": e2, "ek": tr(self.t1, rho), "aj": aj, "ts": ts}

    @staticmethod
    def _bilinear(x, W, y):
        B = x.shape[0]
        y = y.reshape(B, -1)
        w = W.T.contiguous()
        g = torch.complex(y.real.contiguous() @ w, y.imag.contiguous() @ w)
        return (x.reshape(B, -1) * g).sum(1)


def _j2(p):
    return p["aj"] + p["ts"][:, 0] ** 2 + p["ts"][:, 1] ** 2 - p["ts"][:, 2] ** 2


def _angles(mesh):
    b, a, g = np.meshgrid(mesh.bet, mesh.alp, mesh.gam, indexing="ij")
    return a.ravel(), b.ravel(), g.ravel()


def _orbit_traces(b, orbs, rho_diag):
    """sum_m rho(k_a(m), k_b(m)) per species and orbit pair, [.., 2, norb, norb]."""
    out = []
    for sp in range(2):
        for (oa, na, la, ja) in orbs:
            for (ob, nb, lb, jb) in orbs:
                if la != lb or ja != jb:
                    out.append(torch.zeros_like(rho_diag(sp, 0, 0)))
                else:
                    out.append(sum(rho_diag(sp, oa + k, ob + k) for k in range(ja + 1)))
    return torch.stack(out, -1)


def _exact_pair(case, ex, s0, s1, zval, nval, q2):
    """ZRES [NE, 6] and, with q2, the E2 traces [NE, 10] and orbit traces.
    s0, s1: (U, V) of the bra and the ket, per species where no state mixes
    protons and neutrons."""
    b, mesh = make_basis(case["space"]), _mesh(case)
    it = _interaction(case["space"])
    n, h, f = b.n, b.n // 2, case["nphi"]
    al, be, ga = _angles(mesh)
    NE = al.size
    phi = 2.0 * np.pi * np.arange(f) / f
    sgn = -1.0 if (n * (n + 1) // 2) % 2 else 1.0
    logdet = 0.0
    for U, V in s0 + s1:
        Z = V @ np.linalg.inv(U)
        logdet += np.linalg.slogdet(np.eye(len(Z)) + Z.T @ Z)[1]
    vac = sgn * math.exp(-0.25 * logdet)
    dev = _dev()
    pp, pn = np.meshgrid(phi, phi, indexing="ij")
    gph = torch.tensor(np.exp(-1j * (pp * zval + pn * nval)).ravel(), device=dev)
    zres = np.zeros((NE, 6), dtype=complex)
    orbs, k = [], 0
    for (nq, l, tj) in b.orbits:
        orbs.append((k, nq, l, tj))
        k += tj + 1
    norb = len(orbs)
    ze2, zrho = np.zeros((NE, 10), dtype=complex), np.zeros((NE, 2 * norb * norb), dtype=complex)
    if q2 is not None:
        qt = torch.tensor(q2, dtype=torch.complex128, device=dev)
    sep = len(s0) == 2
    step = max(1, (2 ** 31 if sep else 2 ** 30) // (16 * (f * 5 * h * h if sep else f * f * 5 * n * n)))
    for e0 in range(0, NE, step):
        sl = slice(e0, min(NE, e0 + step))
        ne = sl.stop - sl.start
        if sep:
            # states without proton-neutron mixing: every matrix is block
            # diagonal by species, a species depends on its own gauge angle
            P = []
            for s in range(2):
                x = ex[s]
                R = x.rotation(al[sl], be[sl], ga[sl]).repeat_interleave(f, 0)
                ph = torch.tensor(np.exp(1j * np.tile(phi, ne)), device=dev)[:, None].expand(-1, h)
                P.append(x.points(*s0[s], *s1[s], R, ph))
            ff = lambda a, s: (a.reshape(ne, f, 1) if s == 0 else a.reshape(ne, 1, f)).expand(ne, f, f).reshape(-1)
            add = lambda key: ff(P[0][key], 0) + ff(P[1][key], 1)
            r = [P[s]["rho"].reshape(ne, f, h * h) for s in range(2)]
            w = ex[2].T.contiguous()
            g = torch.complex(r[1].real.contiguous() @ w, r[1].imag.contiguous() @ w)
            epn = (r[0] @ g.transpose(1, 2).contiguous()).reshape(-1)
            pf = ((-1) ** h) * ff(P[0]["pf"], 0) * ff(P[1]["pf"], 1)
            ts = torch.stack([ff(P[0]["ts"][:, k], 0) + ff(P[1]["ts"][:, k], 1) for k in range(3)], 1)
            zp = ff(P[0]["rho"].diagonal(dim1=1, dim2=2).sum(1), 0)
            zn = ff(P[1]["rho"].diagonal(dim1=1, dim2=2).sum(1), 1)
            q = {"e2": add("e2") + epn, "ek": add("ek"), "aj": add("aj"), "ts": ts}
            if q2 is not None:
                tq = torch.stack([ff(torch.einsum("ij,bji->b", qt[mu, s * h:(s + 1) * h, s * h:(s + 1) * h],
                                                  P[s]["rho"]), s) for s in range(2) for mu in range(5)], 1)
                to = _orbit_traces(b, orbs, lambda s, i, j: ff(P[s]["rho"][:, i, j], s))
        else:
            x = ex[0]
            R = x.rotation(al[sl], be[sl], ga[sl]).repeat_interleave(f * f, 0)
            hp = np.concatenate([np.repeat(np.exp(1j * pp.ravel())[:, None], h, 1),
                                 np.repeat(np.exp(1j * pn.ravel())[:, None], h, 1)], 1)
            q = x.points(*s0[0], *s1[0], R, torch.tensor(np.tile(hp, (ne, 1)), device=dev))
            d = q["rho"].diagonal(dim1=1, dim2=2)
            zp, zn, pf = d[:, :h].sum(1), d[:, h:].sum(1), q["pf"]
            if q2 is not None:
                tq = torch.stack([torch.einsum("ij,bji->b", qt[mu, s * h:(s + 1) * h, s * h:(s + 1) * h],
                                               q["rho"][:, s * h:(s + 1) * h, s * h:(s + 1) * h])
                                  for s in range(2) for mu in range(5)], 1)
                to = _orbit_traces(b, orbs, lambda s, i, j: q["rho"][:, s * h + i, s * h + j])
        nrm = vac * pf * gph.repeat(ne)
        obs = torch.stack([nrm, nrm * zp, nrm * zn, nrm * q["ek"], nrm * (q["e2"] + q["ek"] + it.e0), nrm * _j2(q)], 1)
        red = lambda a: a.reshape(ne, f * f, -1).mean(1).cpu().numpy()
        zres[sl] = red(obs)
        if q2 is not None:
            ze2[sl], zrho[sl] = red(nrm[:, None] * tq), red(nrm[:, None] * to)
    return zres, ze2, zrho


def _wigner(J, be):
    m = np.arange(J, -J - 1, -1.0)
    jp = np.diag(np.sqrt(J * (J + 1) - m[1:] * (m[1:] + 1)), 1)
    w, v = np.linalg.eigh((jp - jp.T) / 2j)
    d = ((v * np.exp(-1j * be[:, None, None] * w)) @ v.conj().T).real
    return d[:, ::-1, ::-1]  # K from -J to J


def _project(mesh, z):
    """J-projection of z [P, NE, nobs] -> [P, nobs, J+1, 2jmax+1, 2jmax+1]."""
    P, _, nobs = z.shape
    jm, na, nb, ng = mesh.jmax, mesh.alp.size, mesh.bet.size, mesh.gam.size
    zz = z.reshape(P, nb, na, ng, nobs)
    K = np.arange(-jm, jm + 1)
    ea, eg = np.exp(1j * K[:, None] * mesh.alp) * mesh.walp, np.exp(1j * K[:, None] * mesh.gam) * mesh.wgam
    s = np.einsum("ka,pbago,lg->pobkl", ea, zz, eg, optimize=True)
    out = np.zeros((P, nobs, jm + 1, 2 * jm + 1, 2 * jm + 1), dtype=complex)
    for J in range(jm + 1):
        wJ = (2 * J + 1) / 2.0 if na * ng == 1 else (2 * J + 1) / (8 * np.pi ** 2)
        k = slice(jm - J, jm + J + 1)
        out[:, :, J, k, k] = wJ * np.einsum("b,bkl,pobkl->pokl", mesh.wbet, _wigner(J, mesh.bet), s[..., k, k],
                                            optimize=True)
    return out


def _threej(j1, j2, j3, m1, m2, m3):
    if m1 + m2 + m3 or not abs(j1 - j2) <= j3 <= j1 + j2 or abs(m1) > j1 or abs(m2) > j2 or abs(m3) > j3:
        return 0.0
    F = math.factorial
    s = 0.0
    for k in range(j1 + j2 + j3 + 1):
        d = (k, j1 + j2 - j3 - k, j1 - m1 - k, j2 + m2 - k, j3 - j2 + m1 + k, j3 - j1 - m2 + k)
        if min(d) >= 0:
            s += (-1) ** k / math.prod(F(x) for x in d)
    pre = F(j1 + j2 - j3) * F(j1 - j2 + j3) * F(-j1 + j2 + j3) / F(j1 + j2 + j3 + 1)
    pre *= math.prod(F(x) for x in (j1 + m1, j1 - m1, j2 + m2, j2 - m2, j3 + m3, j3 - m3))
    return (-1) ** (j1 - j2 - m3) * math.sqrt(pre) * s


def _reduced_e2(jm, I):
    """<J1 K1 || Q2_s || J2 K2> from the projected traces I [P, 10, J2, K', K2]."""
    P = I.shape[0]
    out = np.zeros((P, 2, 5, jm + 1, 2 * jm + 5, 2 * jm + 1), dtype=complex)
    for dJ in range(-2, 3):
        for J2 in range(jm + 1):
            J1 = J2 + dJ
            if J1 < 0:
                continue
            for K1 in range(-J1, J1 + 1):
                for mu in range(-2, 3):
                    Kp = K1 - mu
                    if abs(Kp) > J2:
                        continue
                    t = (2 * J1 + 1) * (-1) ** (J1 - K1) * _threej(J1, 2, J2, -K1, mu, Kp)
                    for s in range(2):
                        out[:, s, dJ + 2, J2, K1 + jm + 2] += t * I[:, 5 * s + mu + 2, J2, Kp + jm]
    return out


def _hnd(N, H, eps, nos):
    w, v = np.linalg.eigh(N)
    w, v = w[::-1], v[:, ::-1]
    M = 0
    while M < w.size and w[M] / w[0] >= eps:
        M += 1
    M = min(M, nos) if nos > 0 else M
    R = v[:, :M] / np.sqrt(w[:M])
    G = R.T @ H @ R
    return w, R, 0.5 * (G + G.T)


def exact(case, seed):
    if case["kind"] == "hw":
        # the lowest levels per number of natural states; the choice among them
        # (and the levels at it) rests on variances at the rounding level
        N, H = _hw_matrices(case, seed)
        w, R, G = _hnd(N, H, case["eps"], 0)
        M, km = G.shape[0], case["kmax"]
        E = np.zeros((M, km))
        for b in range(M):
            e = np.linalg.eigvalsh(G[:b + 1, :b + 1])
            E[b, :min(km, b + 1)] = e[:km]
        return {"EN": w.copy(), "E_nos": E, "e_best": None, "E": None}
    if case["kind"] == "mlp":
        return None  # the order of the minibatches is the library's own
    b = make_basis(case["space"])
    n, h, f = b.n, b.n // 2, case["nphi"]
    pairs, mesh = _pairs(case), _mesh(case)
    sep = case["form"] != "plain"  # those forms take states without proton-neutron mixing only
    ne = case["nalp"] * case["nbet"] * case["ngam"]
    cost = len(pairs) * ne * (2 * f * h ** 3 if sep else f * f * n ** 3)
    if cost > 1.2e10:
        return None
    U, V = _states(case, seed)
    zv, nv = _valence(case, len(pairs)) if case["zn"] else ([case["zval"]] * len(pairs), [case["nval"]] * len(pairs))
    q2 = q2_matrices(b, 1.0) if case["out"] == "e2" else None
    if sep:
        it = _interaction(case["space"])
        ex = [_Exact(case, np.arange(h)), _Exact(case, np.arange(h, n))]
        # proton-neutron part: rows (c, a) of the protons, columns (d, b) of the neutrons
        W = np.zeros((h * h, h * h))
        i = [x.astype(int) - 1 for x in (it.ka, it.kb, it.kc, it.kd)]
        pn = (i[0] < h) & (i[1] >= h)
        a, bb, c, d, v = i[0][pn], i[1][pn] - h, i[2][pn], i[3][pn] - h, it.me[pn]
        cross = a + bb != c + d
        np.add.at(W, (c * h + a, d * h + bb), v)
        np.add.at(W, ((a * h + c)[cross], (bb * h + d)[cross]), v[cross])
        ex.append(torch.tensor(W, device=_dev()))
    else:
        ex = [_Exact(case, np.arange(n))]
    parts = [np.arange(h), np.arange(h, n)] if sep else [np.arange(n)]
    state = lambda q: [(U[q][np.ix_(i, i)], V[q][np.ix_(i, i)]) for i in parts]
    outs = [_exact_pair(case, ex, state(p), state(q), int(zv[k]), int(nv[k]), q2) for k, (p, q) in enumerate(pairs)]
    z = np.stack([o[0] for o in outs])
    kern = _project(mesh, z)
    if case["out"] == "e2":
        ze2, zrho = np.stack([o[1] for o in outs]), np.stack([o[2] for o in outs])
        norb = len(b.orbits)
        w = np.einsum("b,a,g->bag", mesh.wbet, mesh.walp, mesh.wgam).ravel()
        w0 = 0.5 if mesh.alp.size * mesh.gam.size == 1 else 1.0 / (8 * np.pi ** 2)
        tj = np.array([o[2] for o in b.orbits])
        rho1b = w0 * np.einsum("e,peo->po", w, zrho).reshape(-1, 2, norb, norb) / np.sqrt(tj + 1.0)[None, None, :, None]
        return [z, kern, ze2.reshape(len(pairs), ne, 2, 5), _reduced_e2(case["jmax"], _project(mesh, ze2)), rho1b]
    if not case["zn"] and len(pairs) == 1:
        z, kern = z[0], kern[0]
    return (z, kern) if case["out"] == "zres+kern" else kern

