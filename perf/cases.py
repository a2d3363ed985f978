"""Performance cases of the CTMRG path, through the package's public calls.

Six kinds of work, each on a 2 x 2 unit cell with physical dimension 2, bond
dimension D = 2..5 and environment dimension chi up to 100:

  ctm            a whole environment run from new site tensors
  projector      one projector pair (corner or up-down blocks)
  renormalise    the absorption of one site row (corners and edge)
  observables    one-site, two-site and norm contractions of every site and bond
  gradient       bond energy and its gradient (forward and backward)
  simple_update  imaginary-time steps on all bonds

Outputs that carry the sign freedom of singular vectors are returned in a form
without it: corner spectra, the product PU PL^T of a projector pair, absolute
values of simple-update tensors.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tenes_amd as ta

SZ = np.diag([0.5, -0.5])
SX = np.array([[0.0, 0.5], [0.5, 0.0]])
_SXSX_SYSY = np.zeros((2, 2, 2, 2))
_SXSX_SYSY[0, 1, 1, 0] = _SXSX_SYSY[1, 0, 0, 1] = 0.5
HEISENBERG = np.einsum("ac,bd->abcd", SZ, SZ) + _SXSX_SYSY


def listed():
    return [
        # the smallest configuration of the tests: launches and waits count
        {"name": "ctm_d2_chi10", "kind": "ctm", "D": 2, "chi": 10, "sweeps": 4},
        # an ordinary run, projector matrices just past the exact SVD's size
        {"name": "ctm_d3_chi27", "kind": "ctm", "D": 3, "chi": 27, "sweeps": 3},
        # the benchmark's configuration: sizes of the headline sweep
        {"name": "ctm_d5_chi100", "kind": "ctm", "D": 5, "chi": 100, "sweeps": 4},
        # a ragged matrix of 333 rows, latency of one projector chain
        {"name": "projector_d3_chi37", "kind": "projector", "D": 3, "chi": 37, "corner": True},
        # up-down blocks: four enlarged corners, three matrix products
        {"name": "projector_d4_chi64", "kind": "projector", "D": 4, "chi": 64, "corner": False},
        # one projector of the headline sweep
        {"name": "projector_d5_chi100", "kind": "projector", "D": 5, "chi": 100, "corner": True},
        # absorption of one row: small, and at the headline size
        {"name": "renormalise_d2_chi21", "kind": "renormalise", "D": 2, "chi": 21},
        {"name": "renormalise_d5_chi100", "kind": "renormalise", "D": 5, "chi": 100},
        # measurement of every site and bond on a finished environment
        {"name": "observables_d3_chi45", "kind": "observables", "D": 3, "chi": 45},
        # energy gradient of all eight bonds (variational optimisation)
        {"name": "gradient_d4_chi64", "kind": "gradient", "D": 4, "chi": 64},
        # imaginary-time evolution: many calls on tiny tensors
        {"name": "simple_update_d4", "kind": "simple_update", "D": 4, "chi": 1, "steps": 5},
    ]


def draw(rng):
    kind = rng.choice(["ctm", "projector", "projector", "renormalise", "renormalise", "observables",
                       "gradient", "simple_update"])
    D = rng.randint(2, 5)
    lo = max(8, D * D)  # an initial environment has D^2 directions
    chi = int(round(math.exp(rng.uniform(math.log(lo), math.log(100)))))
    c = {"kind": kind, "D": D, "chi": chi}
    if kind == "ctm":
        c["sweeps"] = rng.randint(1, 4)
    elif kind == "projector":
        c["corner"] = rng.random() < 0.75
    elif kind == "simple_update":
        c["chi"] = 1
        c["steps"] = rng.randint(1, 5)
    return c


# ---------------------------------------------------------------------------
# Inputs (numpy, from the seed alone)
# ---------------------------------------------------------------------------
def _site_tensors(rng, D):
    """Four site tensors as a simple update leaves them: legs weighted by
    decaying bond spectra, a dominant Neel-like component."""
    g = np.exp(-0.45 * np.arange(D))
    out = []
    for i in range(4):
        T = rng.standard_normal((D, D, D, D, 2))
        for leg in range(4):
            T *= g.reshape([-1 if k == leg else 1 for k in range(5)])
        T[0, 0, 0, 0] += (2.0, 0.4) if i in (0, 3) else (0.4, 2.0)
        out.append(T / np.abs(T).max())
    return out


def _environment(rng, D, chi, decay):
    """C[q][site], E[q][site], q counting clockwise from the top-left corner
    and the top edge: decaying corner weights, edges positive in their ket and
    bra legs as those of a converged environment are."""
    w = np.exp(-decay * np.arange(chi) / chi)
    sw = np.sqrt(w[:, None] * w[None, :])
    mu = np.exp(-0.6 * np.arange(D))
    C = [[sw * (np.eye(chi) + 0.1 * rng.standard_normal((chi, chi))) for _ in range(4)] for _ in range(4)]
    E = []
    for _ in range(4):
        row = []
        for _ in range(4):
            A = 0.2 * rng.standard_normal((chi, chi, D, D)) / math.sqrt(chi)
            A += (np.eye(chi)[:, :, None, None] + 0.02) * np.eye(D)
            A *= mu
            e = np.matmul(A.transpose(0, 1, 3, 2), A) * sw[:, :, None, None] ** 0.25
            row.append(e / np.abs(e).max())
        E.append(row)
    return C, E


def _projector_pair(rng, D, chi):
    """A projector pair (chi, D, D, chi) with orthonormal columns."""
    out = []
    for _ in range(2):
        q, _ = np.linalg.qr(rng.standard_normal((chi * D * D, chi)))
        out.append(q.reshape(chi, D, D, chi))
    return out


def _gate(rng):
    """exp(-tau H) of an Ising bond in tilted fields, with a little disorder
    so that no bond spectrum is degenerate."""
    h = rng.uniform(0.5, 1.0, 4)
    I = np.eye(2)
    H = -4.0 * np.kron(SZ, SZ) - h[0] * np.kron(SX, I) - h[1] * np.kron(I, SX) \
        - 0.3 * h[2] * np.kron(SZ, I) - 0.3 * h[3] * np.kron(I, SZ)
    w, v = np.linalg.eigh(H)
    return ((v * np.exp(-0.05 * w)) @ v.T).reshape(2, 2, 2, 2)


def _inputs(case, seed):
    rng = np.random.default_rng([seed, case["D"], case["chi"]])
    D, chi, kind = case["D"], case["chi"], case["kind"]
    s = {"T": _site_tensors(rng, D)}
    if kind in ("projector", "renormalise", "observables", "gradient"):
        # corner decay for kept singular values of the projector's matrix down
        # to 1e-5 or 1e-6 of the largest at every D (the number of its
        # directions per corner weight grows with D^2, and an up-down matrix
        # multiplies all four corners)
        s["C"], s["E"] = _environment(rng, D, chi, (5.5 if case.get("corner", True) else 1.2) * D)
    if kind == "renormalise":
        s["P"] = _projector_pair(rng, D, chi)
    if kind == "simple_update":
        s["T"] = [t + 0.02 * rng.standard_normal(t.shape) for t in s["T"]]
        s["gates"] = [(site, leg, _gate(rng)) for site in range(4) for leg in (2, 1)]
    return s


_ctx = None


def _context():
    """One library context per process, as a program keeps."""
    global _ctx
    if _ctx is None:
        _ctx = ta.Context(0, seed=7)
    return _ctx


def _up(ctx, v):
    return [_up(ctx, x) for x in v] if isinstance(v, list) else ctx.tensor(v)


CORNERS, EDGES = ("C1", "C2", "C3", "C4"), ("eTt", "eTr", "eTb", "eTl")


def prepare(case, seed):
    ctx = _context()
    h = _inputs(case, seed)
    kind = case["kind"]
    s = {"case": case, "ctx": ctx, "T": _up(ctx, h["T"])}
    if kind == "ctm":
        s["params"] = ta.peps_parameters(CHI=case["chi"], Max_CTM_Iteration=case["sweeps"],
                                         CTM_Convergence_Epsilon=0.0)
    elif kind == "projector":
        s["C"], s["E"] = _up(ctx, h["C"]), _up(ctx, h["E"])
        s["params"] = ta.peps_parameters(CHI=case["chi"])
        n = case["chi"] * case["D"] ** 2
        s["out"] = torch.empty((n, n), dtype=torch.float64, device="cuda")
    elif kind == "renormalise":
        s["C"], s["E"] = _up(ctx, h["C"]), _up(ctx, h["E"])
        s["P"] = _up(ctx, h["P"])
        c, d = case["chi"], case["D"]
        s["out"] = [torch.empty(z, dtype=torch.float64, device="cuda")
                    for z in ((c, c), (c, c), (c, c, d, d))]
    elif kind in ("observables", "gradient"):
        env = ta.Environment(ctx, 2, 2)
        env.set_site_tensors(h["T"])
        for q in range(4):
            for i in range(4):
                env.set(CORNERS[q], i, h["C"][q][i])
                env.set(EDGES[q], i, h["E"][q][i])
        s["env"] = env
        if kind == "gradient":
            s["bonds"] = [(i, dx, dy, HEISENBERG) for i in range(4) for dx, dy in ((1, 0), (0, 1))]
    else:
        s["gates"] = [(i, leg, ctx.tensor(op)) for i, leg, op in h["gates"]]
    ctx.synchronize()
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "ctm":
        env = ta.Environment(ctx, 2, 2)
        for i in range(4):
            env.set("Tn", i, s["T"][i])
        n, _ = env.calc_ctm_environment(s["params"])
        return {"sweeps": n, "spectra": [env.corner_spectrum(k, i) for k in CORNERS for i in range(4)]}
    if kind == "projector":
        C, E, T = s["C"], s["E"], s["T"]
        if case["corner"]:
            PU, PL = ta.calc_projector_left_block(C[0][0], C[3][2], E[0][0], E[2][2], E[3][2], E[3][0],
                                                  T[0], T[2], s["params"])
        else:
            PU, PL = ta.calc_projector_updown_blocks(
                [C[0][0], C[1][1], C[2][3], C[3][2], E[0][0], E[0][1], E[1][1], E[1][3], E[2][3],
                 E[2][2], E[3][2], E[3][0], T[0], T[1], T[3], T[2]], s["params"])
        ta.tensordot(PU, PL, [3], [3]).copy_to_device(s["out"].data_ptr())
        return s["out"]
    if kind == "renormalise":
        C, E, T, (PU, PL) = s["C"], s["E"], s["T"], s["P"]
        new = ta.calc_next_ctm(C[0][0], C[3][2], E[0][0], E[2][2], PU, PL)
        new += (ta.calc_next_et(E[3][0], T[0], PU, PL),)
        for t, o in zip(new, s["out"]):
            t.copy_to_device(o.data_ptr())
        return s["out"]
    if kind == "observables":
        env = s["env"]
        one = [[env.contract_one_site(i, op) for op in (None, SZ, SX)] for i in range(4)]
        two = [[env.contract_two_sites_op12(i, dx, dy, HEISENBERG), env.contract_cluster(i, dx, dy)]
               for i in range(4) for dx, dy in ((1, 0), (0, 1))]
        return {"one": np.array(one), "two": np.array(two)}
    if kind == "gradient":
        e, g = s["env"].bond_energy(s["bonds"], grad=True)
        return {"energy": e, "gradient": g}
    env = ta.Environment(ctx, 2, 2)
    for i in range(4):
        env.set("Tn", i, s["T"][i])
    env.simple_update(s["gates"], case["steps"])
    return {"lambda": [env.get_lambda(i, leg) for i in range(4) for leg in range(4)],
            "site": [np.abs(t) for t in env.site_tensors()]}


def work(case):
    """Inputs read once and outputs written once; multiply-adds of the
    reference's contraction order (a truncated SVD of an n x n matrix as the
    two products that a rank-chi factorisation cannot do without)."""
    D, c, kind = float(case["D"]), float(case["chi"]), case["kind"]
    n = c * D * D
    site = 2 * D ** 4
    edge, corner = c * c * D * D, c * c
    enlarged = 2 * c * c * c * D * D + 2 * c * c * c * D ** 4 + 4 * 2 * c * c * D ** 6
    nextc = 2 * (2 * c ** 3 * D * D + 2 * c ** 3 * D * D)
    nexte = 2 * c ** 3 * D ** 4 + 4 * 2 * c * c * D ** 6 + 2 * c ** 3 * D ** 4
    proj = 2 * enlarged + 2 * n ** 3 + 2 * 2 * n * n * c + 2 * 2 * n * n * c
    if kind == "ctm":
        sweep = 16 * (proj + nextc) + 32 * nexte
        return {"bytes": 8 * (4 * site + 16 * c), "flops": case["sweeps"] * sweep}
    if kind == "projector":
        if case["corner"]:
            return {"bytes": 8 * (2 * site + 4 * edge + 2 * corner + n * n), "flops": proj + 2 * n * n * c}
        return {"bytes": 8 * (4 * site + 8 * edge + 4 * corner + n * n),
                "flops": proj + 2 * enlarged + 2 * 2 * n ** 3 + 2 * n * n * c}
    if kind == "renormalise":
        return {"bytes": 8 * (site + 3 * edge + 2 * corner + 2 * n * c + 2 * corner + edge),
                "flops": nextc + nexte}
    half = 2 * c ** 3 * D * D * 2 + 2 * c ** 3 * D ** 4 * 2 + 4 * 2 * c * c * D ** 6
    env_bytes = 8 * (4 * site + 16 * edge + 16 * corner)
    if kind == "observables":
        return {"bytes": env_bytes, "flops": 12 * half + 8 * 2 * 2 * half}
    if kind == "gradient":
        return {"bytes": env_bytes + 8 * 4 * site, "flops": 8 * 2 * half * 3}
    bond = 2 * 2 * (D ** 3) * (2 * D) ** 2 * 2 + 4 * (2 * D) ** 3 * 4
    return {"bytes": 2 * 8 * 4 * site, "flops": case["steps"] * 8 * bond}


# ---------------------------------------------------------------------------
# The same in numpy / torch, 64 bits
# ---------------------------------------------------------------------------
td = np.tensordot


def _rot(T, q):
    return T.transpose([(q + k) % 4 for k in range(4)] + [4])


def _enlarged(C1, eT1, eT8, T):
    """(t12, e12, tc12, t41, e78, tc41): corner, edges and both layers."""
    X = td(td(td(td(C1, eT1, (1, 0)), eT8, (0, 1)), T, ([2, 5], [1, 0])), T, ([1, 3, 6], [1, 0, 4]))
    # legs e12, e78, t12c, t41c, t12, t41
    return X.transpose(4, 0, 2, 5, 1, 3)


def _enlarged_low(C4, eT7, eT6, T):
    """(t41, e78, tc41, t34, e56, tc34)"""
    X = td(td(td(td(C4, eT7, (1, 0)), eT6, (0, 1)), T, ([2, 5], [0, 3])), T, ([1, 3, 6], [0, 3, 4]))
    return X.transpose(4, 0, 2, 5, 1, 3)


def _truncated(A, B, M, shape, chi, cut=1e-12):
    """PU = B V s^-1/2, PL = A U s^-1/2 as (n, k) matrices."""
    U, s, V = np.linalg.svd(M, full_matrices=False)
    k = min(chi, int(np.sum(s / s[0] > cut)))
    r = 1.0 / np.sqrt(s[:k])
    PU, PL = (B @ V[:k].T) * r, (A @ U[:, :k]) * r
    t, e, b = shape  # stored (t, e, b), wanted (e, t, b, k)
    return [P.reshape(t, e, b, k).transpose(1, 0, 2, 3) for P in (PU, PL)]


def _corner_pair(C1, C4, eT1, eT6, eT7, eT8, T1, T4, chi):
    LT, LB = _enlarged(C1, eT1, eT8, T1), _enlarged_low(C4, eT7, eT6, T4)
    shape = LT.shape[3:]
    n = int(np.prod(shape))
    LT, LB = LT.reshape(-1, n), LB.reshape(n, -1)
    return _truncated(LT.T, LB, LT @ LB, shape, chi)


def _updown_pair(C, e, T, chi):
    LT, LB = _enlarged(C[0], e[0], e[7], T[0]), _enlarged_low(C[3], e[6], e[5], T[3])
    # the right half turned by half a turn has the left half's form
    RB = _enlarged(C[2], e[4], e[3], _rot(T[2], 2))  # (t34, e56, b34, t23, e34, b23)
    RT = _enlarged_low(C[1], e[2], e[1], _rot(T[1], 2))  # (t23, e34, b23, t12, e12, b12)
    shape = LT.shape[3:]
    n = int(np.prod(shape))
    R1 = RT.reshape(n, -1) @ LT.reshape(-1, n)  # (right bond, left bond)
    R2 = RB.reshape(-1, n).T @ LB.reshape(n, -1).T
    return _truncated(R1.T, R2.T, R1 @ R2.T, shape, chi)


def _next_corners(C1, C4, eT1, eT6, PU, PL):
    a = td(PU, td(C1, eT1, (1, 0)), ([0, 1, 2], [0, 2, 3]))
    b = td(td(eT6, C4, (1, 0)), PL, ([3, 1, 2], [0, 1, 2]))
    return a / np.abs(a).max(), b / np.abs(b).max()


def _next_edge(eT8, T, PU, PL):
    X = td(eT8, PL, (1, 0))  # a, k8, b8, t, tc, c
    X = td(X, T, ([2, 4], [0, 1]))  # a, k8, t, c, r', d', p
    X = td(X, T, ([1, 2, 6], [0, 1, 4]))  # a, c, r', d', r, d
    e = td(X, PU, ([0, 3, 5], [0, 2, 1])).transpose(3, 0, 2, 1)  # c, r', r, k -> (k, c, r, r')
    return e / np.abs(e).max()


def _ctm(T, chi, sweeps):
    """Directional CTMRG on the 2 x 2 cell, all four moves as the left move
    seen from a turned lattice."""
    x, y = lambda i: i % 2, lambda i: i // 2
    # neighbours l, u, r, d of the 2 x 2 torus
    step = [lambda i: y(i) * 2 + 1 - x(i), lambda i: (1 - y(i)) * 2 + x(i)] * 2

    def fit(M):
        M = M[:chi, :chi]
        pad = [(0, chi - M.shape[0]), (0, chi - M.shape[1])] + [(0, 0)] * (M.ndim - 2)
        return np.pad(M, pad)

    C, E = [[None] * 4 for _ in range(4)], [[None] * 4 for _ in range(4)]
    for q in range(4):
        for i in range(4):
            A = _rot(T[step[(1 + q) % 4](step[q](i))], q)
            B = td(A, A, ([0, 1, 4], [0, 1, 4]))
            C[q][i] = fit(B.transpose(1, 3, 0, 2).reshape(A.shape[3] ** 2, A.shape[2] ** 2))
            A = _rot(T[step[(1 + q) % 4](i)], q)
            B = td(A, A, ([1, 4], [1, 4])).transpose(0, 3, 1, 4, 2, 5)
            E[q][i] = fit(B.reshape(A.shape[0] ** 2, A.shape[2] ** 2, A.shape[3], A.shape[3]))
    lines = [[[0, 2], [1, 3]], [[2, 3], [0, 1]], [[1, 3], [0, 2]], [[0, 1], [2, 3]]]
    for _ in range(sweeps):
        for q in (0, 2, 1, 3):
            a, b, d = q, (q + 2) % 4, (q + 3) % 4  # edges t, b, l; corners q, d
            dn, up, fwd = step[(q + 3) % 4], step[(q + 1) % 4], step[(q + 2) % 4]
            for line in lines[q]:
                P = {i: _corner_pair(C[q][i], C[d][dn(i)], E[a][i], E[b][dn(i)], E[d][dn(i)], E[d][i],
                                     _rot(T[i], q), _rot(T[dn(i)], q), chi) for i in line}
                new = []
                for i in line:
                    l = dn(i)
                    c1, c4 = _next_corners(C[q][i], C[d][l], E[a][i], E[b][l], P[up(i)][0], P[l][1])
                    new.append((fwd(i), fwd(l), c1, c4,
                                _next_edge(E[d][i], _rot(T[i], q), P[i][0], P[up(i)][1])))
                for j, k, c1, c4, e in new:
                    C[q][j], C[d][k], E[d][j] = c1, c4, e
    return C, E


def _rho(T, C, E, i, j, q):
    """Two-site density matrix (ket i, bra i, ket j, bra j), j one step behind
    direction q + 2 of i (torch, the lattice turned by q)."""
    r = lambda t: t.permute([(q + k) % 4 for k in range(4)] + [4])  # noqa: E731
    Ti, Tj = r(T[i]), r(T[j])
    Cq = lambda k, s: C[(k + q) % 4][s]  # noqa: E731
    Eq = lambda k, s: E[(k + q) % 4][s]  # noqa: E731
    X = torch.einsum("ac,cdkK->adkK", Cq(3, i), Eq(3, i))
    X = torch.einsum("adkK,de->aekK", X, Cq(0, i))
    X = torch.einsum("aekK,etnN->atkKnN", X, Eq(0, i))
    X = torch.einsum("atkKnN,knrmp->atKNrmp", X, Ti)
    X = torch.einsum("atKNrmp,KNRMq->atrmpRMq", X, Ti)
    L = torch.einsum("atrmpRMq,bamM->btrRpq", X, Eq(2, i))
    X = torch.einsum("ef,fgxX->egxX", Cq(1, j), Eq(1, j))
    X = torch.einsum("egxX,gh->ehxX", X, Cq(2, j))
    X = torch.einsum("tenN,ehxX->thnNxX", Eq(0, j), X)
    X = torch.einsum("thnNxX,rnxms->thNXrms", X, Tj)
    X = torch.einsum("thNXrms,RNXMu->thrmsRMu", X, Tj)
    R = torch.einsum("thrmsRMu,hbmM->btrRsu", X, Eq(2, j))
    return torch.einsum("btrRpq,btrRsu->pqsu", L, R)


def _bonds(T, C, E):
    """The density matrices of the bonds (site, +x), (site, +y)."""
    for i in range(4):
        yield _rho(T, C, E, i, i ^ 1, 0)
        yield _rho(T, C, E, i ^ 2, i, 1)  # the upper site first


def _one_site(T, C, E, i):
    X = torch.einsum("ac,cdkK,de->aekK", C[3][i], E[3][i], C[0][i])
    X = torch.einsum("aekK,efnN->afkKnN", X, E[0][i])
    X = torch.einsum("afkKnN,knrmp->afKNrmp", X, T[i])
    X = torch.einsum("afKNrmp,KNRMq->afrmpRMq", X, T[i])
    Y = torch.einsum("fg,ghrR,hj->fjrR", C[1][i], E[1][i], C[2][i])
    Y = torch.einsum("fjrR,jamM->farRmM", Y, E[2][i])
    return torch.einsum("afrmpRMq,farRmM->pq", X, Y)


def _simple_update(T, gates, steps):
    T = list(T)
    lam = [[np.ones(T[i].shape[k]) for k in range(4)] for i in range(4)]
    for _ in range(steps):
        for i, leg, op in gates:
            j = i ^ 1 if leg == 2 else i ^ 2
            back = (leg + 2) % 4
            half, D = [], T[i].shape[leg]
            for s, k in ((i, leg), (j, back)):
                rest = [q for q in range(4) if q != k]
                A = T[s]
                for q in rest:
                    A = A * lam[s][q].reshape([-1 if r == q else 1 for r in range(5)])
                A = A.transpose(rest + [k, 4])
                Q, R = np.linalg.qr(A.reshape(-1, D * 2))
                half.append((rest, A.shape[:3], Q, R.reshape(-1, D, 2)))
            theta = np.einsum("axp,bxq,pqrs->arbs", half[0][3], half[1][3], op)
            m, n = theta.shape[0] * 2, theta.shape[2] * 2
            U, w, V = np.linalg.svd(theta.reshape(m, n), full_matrices=False)
            w = w[:D]
            w = np.sqrt(w / np.sqrt(np.sum(w * w)))
            new = [(U[:, :D] * w).reshape(-1, 2, D), (V[:D].T * w).reshape(-1, 2, D)]
            for (s, k), (rest, shape, Q, _), N in zip(((i, leg), (j, back)), half, new):
                A = np.einsum("xa,apk->xkp", Q, N).reshape(shape + (D, 2))
                for pos, q in enumerate(rest):
                    A = A / lam[s][q].reshape([-1 if r == pos else 1 for r in range(5)])
                order = rest + [k]
                T[s] = A.transpose([order.index(q) for q in range(4)] + [4])
            lam[i][leg] = lam[j][back] = w
    return T, lam


def exact(case, seed):
    D, chi, kind = case["D"], case["chi"], case["kind"]
    n = chi * D * D
    if kind == "ctm" and 16 * case["sweeps"] * n ** 3 > 6e10:
        return None  # minutes of LAPACK SVDs
    h = _inputs(case, seed)
    if kind == "ctm":
        C, _ = _ctm(h["T"], chi, case["sweeps"])
        spec = []
        for q in range(4):
            for i in range(4):
                s = np.linalg.svd(C[q][i], compute_uv=False)
                spec.append(s / np.sqrt(np.sum(s * s)))
        return {"sweeps": None, "spectra": spec}
    if kind == "projector":
        C, E, T = h["C"], h["E"], h["T"]
        if case["corner"]:
            PU, PL = _corner_pair(C[0][0], C[3][2], E[0][0], E[2][2], E[3][2], E[3][0], T[0], T[2], chi)
        else:
            PU, PL = _updown_pair([C[0][0], C[1][1], C[2][3], C[3][2]],
                                  [E[0][0], E[0][1], E[1][1], E[1][3], E[2][3], E[2][2], E[3][2], E[3][0]],
                                  [T[0], T[1], T[3], T[2]], chi)
        return PU.reshape(n, -1) @ PL.reshape(n, -1).T
    if kind == "renormalise":
        C, E, (PU, PL) = h["C"], h["E"], h["P"]
        return [*_next_corners(C[0][0], C[3][2], E[0][0], E[2][2], PU, PL),
                _next_edge(E[3][0], h["T"][0], PU, PL)]
    if kind in ("observables", "gradient"):
        T, C, E = ([torch.from_numpy(t) for t in h["T"]],
                   *([[torch.from_numpy(t) for t in r] for r in h[k]] for k in ("C", "E")))
        op = torch.from_numpy(HEISENBERG)
        norm = lambda rho: torch.einsum("ppss->", rho)  # noqa: E731
        if kind == "observables":
            one = [_one_site(T, C, E, i) for i in range(4)]
            two = [[float(torch.einsum("pqsu,psqu->", r, op)), float(norm(r))] for r in _bonds(T, C, E)]
            return {"one": np.array([[float(torch.trace(r)), float((r * torch.from_numpy(SZ)).sum()),
                                      float((r * torch.from_numpy(SX)).sum())] for r in one]),
                    "two": np.array(two)}
        for t in T:
            t.requires_grad_(True)
        e = sum(torch.einsum("pqsu,psqu->", r, op) / norm(r) for r in _bonds(T, C, E)) / 4
        e.backward()
        return {"energy": e.item(), "gradient": [t.grad.numpy() for t in T]}
    T, lam = _simple_update(h["T"], h["gates"], case["steps"])
    return {"lambda": [lam[i][k] for i in range(4) for k in range(4)], "site": [np.abs(t) for t in T]}
