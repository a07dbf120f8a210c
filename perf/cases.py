"""Performance cases: the calls a DMRG / TDVP program makes, over their sizes.

Every case is one pass through the package's public entry points on a state
that a sweep would hand them: isometric tensors left and right of the centre
(so the environments are true projections of the Hamiltonian), a centre pair
whose weights fall off as an entanglement spectrum does (about five decades
over the kept states), charges distributed as at the middle of a chain.

Paths:
  envs     Lupdate and Rupdate of one site each (the update after a bond step,
           makeEnv, expect, measurements)
  bond     one two-site DMRG bond step (dmrj_twostep: two-vector Lanczos on
           H_eff, truncated SVD), left- or right-moving, in FP64 or with
           split-precision H_eff
  step3s   one single-site step with subspace expansion (step3S)
  tdvp     one real-time TDVP bond step on a ComplexF64 state (Krylov
           exponential, truncated SVD, one-site evolution of the new centre)
  sweep    dmrg() on a whole short chain, one sweep back and forth
  evolve   tdvp_twosite() on a whole short chain, one half-sweep

The SVD is the default one (backend 0, FP64 accuracy).  The Gram-matrix form
(backend 5) is not listed: its small singular values carry an error of
sqrt(eps), so its outputs are not defined to the digits that are compared.

Tensors stay on the device between calls, as in a sweep; a Results entry that
is a tensor comes to the host when it is read.  Where a tensor has a free
gauge (the signs and rotations of singular vectors) the outputs hold the
gauge-free product of the tensors: the two-site state, or the state vector of
a short chain.
"""
import ctypes as C
import math

import numpy as np
import torch

from __graft_entry__ import load_package

pkg = load_package()

# physical charges and the Hamiltonian of the two models
HEISENBERG = np.array([[1], [-1]])                          # 2 Sz
HUBBARD = np.array([[0, 0], [1, 1], [1, -1], [2, 0]])       # N, 2 Sz

# how much more peaked a truncated bond's charges are than the free count, by
# the number of charges: sector sizes as found in converged sweeps (m=1024
# Heisenberg: up to 600; m=2048 Hubbard: up to 1100)
SHARPEN = {0: 0.0, 1: 0.01, 2: 0.1}


class Results(dict):
    """Outputs of a pass by name; entries that are functions read a device
    tensor out when they are asked for."""

    def __getitem__(self, key):
        v = super().__getitem__(key)
        return v() if callable(v) else v


def listed():
    return [
        # the first and last sites of every chain, and product-like states: launches only
        dict(name="envs_dense_m16", path="envs", model="heisenberg", qn=False, m=16, mr=16),
        # the environment update of the Hubbard chain
        dict(name="envs_hubbard_m1024", path="envs", model="hubbard", qn=True, m=1024, mr=1024),
        # early sweeps and weakly entangled bonds: every sector is small
        dict(name="bond_heisenberg_m96", path="bond", model="heisenberg", qn=True, m=96, mr=90, dir=-1,
             precision="f64"),
        # a program that uses no charges: one dense matrix
        dict(name="bond_dense_m200", path="bond", model="heisenberg", qn=False, m=200, mr=187, dir=1,
             precision="f64"),
        # the middle of the L=100 Heisenberg chain at m=1024
        dict(name="bond_heisenberg_m1024", path="bond", model="heisenberg", qn=True, m=1024, mr=1024, dir=1,
             precision="f64"),
        # the ramp of the Hubbard chain, ragged dimensions
        dict(name="bond_hubbard_m510", path="bond", model="hubbard", qn=True, m=510, mr=477, dir=-1,
             precision="f64"),
        # the middle of the L=64 Hubbard chain at m=2048, FP64 throughout
        dict(name="bond_hubbard_m2048", path="bond", model="hubbard", qn=True, m=2048, mr=2048, dir=1,
             precision="f64"),
        # the mixed-precision step of its ramp, moving left
        dict(name="bond_hubbard_m1024_f16x3", path="bond", model="hubbard", qn=True, m=1024, mr=1024, dir=-1,
             precision="f16x3"),
        # 3S with the expansion active: sectors far wider than tall
        dict(name="step3s_heisenberg_m512", path="step3s", model="heisenberg", qn=True, m=512, mr=512, dir=1),
        # a bond of a time evolution that has built up entanglement
        dict(name="tdvp_dense_m96", path="tdvp", model="heisenberg", qn=False, m=96, mr=90, dir=1),
        # a whole call: L=20 at m=64 without charges
        dict(name="sweep_dense_L20_m64", path="sweep", model="heisenberg", qn=False, L=20, m=64),
        # a whole call: a half-sweep of a weakly entangled evolving chain
        dict(name="evolve_L14_m12", path="evolve", model="heisenberg", qn=True, L=14, m=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["envs", "envs", "bond", "bond", "bond", "bond", "step3s", "tdvp", "sweep", "evolve"])
    if path == "sweep":
        return dict(path=path, model="heisenberg", qn=rng.random() < 0.5, L=rng.randint(10, 20),
                    m=_log_int(rng, 12, 64))
    if path == "evolve":
        return dict(path=path, model="heisenberg", qn=rng.random() < 0.7, L=rng.randint(8, 14),
                    m=_log_int(rng, 4, 12))
    if path == "step3s":
        model, qn, m = "heisenberg", True, _log_int(rng, 24, 512)
    elif path == "tdvp":
        # with charges up to the dimension of the first times of an evolution
        # (charge sectors up to 30)
        model, qn = "heisenberg", rng.random() < 0.5
        m = _log_int(rng, 8, 40 if qn else 110)
    else:
        kind = rng.choice(["dense", "heisenberg", "hubbard", "hubbard"])
        model, qn = ("heisenberg", False) if kind == "dense" else (kind, True)
        m = _log_int(rng, 8, {"dense": 200, "heisenberg": 1024, "hubbard": 2048}[kind])
    case = dict(path=path, model=model, qn=qn, m=m, mr=max(4, int(m * rng.uniform(0.8, 1.0))))
    if path != "envs":
        case["dir"] = rng.choice([1, -1])
    if path == "bond":
        case["precision"] = rng.choice(["f64", "f64", "f64", "f16x3", "bf16x3"])
    return case


# ------------------------------------------------------------ host inputs

def _charges(case):
    q = HUBBARD if case["model"] == "hubbard" else HEISENBERG
    return q if case["qn"] else q[:, :0]


def _bulk(case):
    return pkg.hubbardMPO() if case["model"] == "hubbard" else pkg.heisenbergMPO()


def _mpo(case, L):
    d = len(_charges(case))
    H = pkg.makeMPO(_bulk(case), d, L).H
    return pkg.MPO(H, qphys=_charges(case)) if case["qn"] else pkg.MPO(H)


def _groups(q):
    """{charge: indices} of a list of charges, charges ascending."""
    out = {}
    for i, c in enumerate(map(tuple, q.tolist())):
        out.setdefault(c, []).append(i)
    return {c: np.array(out[c]) for c in sorted(out)}


def _pick(avail, m, centre):
    """How many states of each charge a bond of dimension m keeps: all when
    they fit, else in proportion to what there is, weighted to the centre."""
    total = sum(avail.values())
    if total <= m:
        return dict(avail)
    w = {c: n * math.exp(-SHARPEN[len(c)] * sum((x - y) ** 2 for x, y in zip(c, centre))) for c, n in avail.items()}
    keep = {c: 0 for c in avail}
    left = m
    while left > 0:
        open_ = [c for c in avail if keep[c] < avail[c]]
        s = sum(w[c] for c in open_)
        step = {c: min(avail[c] - keep[c], int(left * w[c] / s)) for c in open_}
        if not any(step.values()):
            step = {c: 1 for c in sorted(open_, key=lambda c: -w[c])[:left]}
        for c, n in step.items():
            keep[c] += n
            left -= n
    return {c: n for c, n in keep.items() if n}


def _blocks(qrow, qcol):
    rows, cols = _groups(qrow), _groups(qcol)
    return [(rows[c], cols[c]) for c in rows if c in cols]


def _join(q, qphys):
    """Charges of (a, s) for a left bond a, s running fastest."""
    return (q[:, None, :] + qphys[None, :, :]).reshape(len(q) * len(qphys), qphys.shape[1])


def _cols(q, qphys):
    """Charges of (s, b) for a right bond b, b running fastest."""
    return (q[None, :, :] - qphys[:, None, :]).reshape(len(q) * len(qphys), qphys.shape[1])


def _left_blocks(ql, qphys, qr):
    """Index sets of A[a, s, b] seen as a matrix (a + n s, b)."""
    stacked = (ql[None, :, :] + qphys[:, None, :]).reshape(len(ql) * len(qphys), qphys.shape[1])
    return _blocks(stacked, qr)


def _right_blocks(ql, qphys, qr):
    """Index sets of A[a, s, b] seen as a matrix (a, s + d b)."""
    stacked = (qr[:, None, :] - qphys[None, :, :]).reshape(len(qr) * len(qphys), qphys.shape[1])
    return _blocks(ql, stacked)


def _bond_charges(keep, nq):
    rows = [c for c in sorted(keep) for _ in range(keep[c])]
    return np.array(rows, dtype=np.int64).reshape(len(rows), nq)


def _grow(case, m):
    """Charges of the bonds from a chain's end to a bond of dimension m."""
    qphys = _charges(case)
    d, nq = qphys.shape
    n = max(1, math.ceil(math.log(m) / math.log(d) - 1e-9)) + (1 if case["qn"] else 0)
    q = [np.zeros((1, nq), dtype=np.int64)]
    for k in range(n):
        avail = {c: len(i) for c, i in _groups(_join(q[-1], qphys)).items()}
        q.append(_bond_charges(_pick(avail, m, [x * (k + 1) for x in qphys.mean(axis=0)]), nq))
    return q


def _isometry(rng, ql, qphys, qr, left):
    """A[a, s, b] (column-major) with orthonormal columns (left) or rows."""
    n, d, m = len(ql), len(qphys), len(qr)
    if left:
        M = np.zeros((n * d, m), order="F")
        for r, c in _left_blocks(ql, qphys, qr):
            M[np.ix_(r, c)] = np.linalg.qr(rng.standard_normal((len(r), len(c))))[0]
    else:
        M = np.zeros((n, d * m), order="F")
        for r, c in _right_blocks(ql, qphys, qr):
            M[np.ix_(r, c)] = np.linalg.qr(rng.standard_normal((len(c), len(r))))[0].T
    return M.reshape(n, d, m, order="F")


def _spread(q, centre):
    """Schmidt-like weights of a bond, descending within every charge:
    exp(-a ln^2(1 + r)) of a rank r over the whole bond, eight decades."""
    n = len(q)
    a = 18.4 / math.log(1.0 + max(n, 2)) ** 2
    w = np.zeros(n)
    for c, idx in _groups(q).items():
        r = np.arange(len(idx)) * (n / len(idx)) * 0.5 + 0.5 * sum((x - y) ** 2 for x, y in zip(c, centre))
        w[idx] = np.exp(-a * np.log1p(r) ** 2)
    return w


def _bonds(case):
    """Bond charges: left sites, the centre bond, right sites."""
    qphys = _charges(case)
    nq = qphys.shape[1]
    qL, qR = _grow(case, case["m"]), _grow(case, case["mr"])
    n = len(qL) + len(qR)                            # sites: those of both sides and the centre pair
    # half filling, no magnetisation (one unpaired spin on an odd chain)
    total = np.array([n, n % 2][2 - nq:] if nq else [], dtype=np.int64)
    qB = [_bond_charges({c: len(i) for c, i in _groups(total[None, :] - x).items()}, nq) for x in qR[::-1]]
    # the centre bond: what both neighbours reach
    left = {c: len(i) for c, i in _groups(_join(qL[-1], qphys)).items()}
    right = {c: len(i) for c, i in _groups(_cols(qB[0], qphys)).items()}
    both = {c: min(k, right[c]) for c, k in left.items() if c in right}
    qc = _bond_charges(_pick(both, case["m"], [x * len(qL) for x in qphys.mean(axis=0)]), nq)
    return qL, qc, qB


def _host(case, seed):
    """Left sites, the two centre tensors, right sites and all bond charges."""
    rng = np.random.default_rng([seed, case["m"]])
    qphys = _charges(case)
    d = len(qphys)
    qL, qc, qB = _bonds(case)
    AL = [_isometry(rng, qL[k], qphys, qL[k + 1], True) for k in range(len(qL) - 1)]
    BR = [_isometry(rng, qB[k], qphys, qB[k + 1], False) for k in range(len(qB) - 1)]
    qa, qb = qL[-1], qB[0]
    mean = qphys.mean(axis=0)
    wa, wb, wc = (_spread(q, [x * k for x in mean]) for q, k in
                  ((qa, len(qL) - 1), (qb, len(qL) + 1), (qc, len(qL))))
    cplx = case["path"] == "tdvp"

    def gauss(n, m):
        g = rng.standard_normal((n, m))
        return g + 1j * rng.standard_normal((n, m)) if cplx else g

    kind = np.complex128 if cplx else np.float64
    P = np.zeros((len(qa) * d, len(qc)), dtype=kind, order="F")
    R = np.zeros((len(qc), d * len(qb)), dtype=kind, order="F")
    wrow, wcol = np.tile(wa ** 0.5, d), np.repeat(wb ** 0.5, d)
    gram, pnorm, rnorm, norm = {}, 0.0, 0.0, 0.0
    for r, c in _left_blocks(qa, qphys, qc):
        x = wrow[r][:, None] * gauss(len(r), len(c)) * wc[c] ** 0.3
        P[np.ix_(r, c)] = x
        gram[c[0]] = x.conj().T @ x
        pnorm += np.linalg.norm(x) ** 2
    for r, c in _right_blocks(qc, qphys, qb):
        x = (wc[r] ** 0.3)[:, None] * gauss(len(r), len(c)) * wcol[c]
        R[np.ix_(r, c)] = x
        norm += np.real(np.sum(gram[r[0]] * (x @ x.conj().T).T))
        rnorm += np.linalg.norm(x) ** 2
    # unit norm of the two-site state and of its centre: the right tensor when moving left
    f = math.sqrt(pnorm if case.get("dir", 1) > 0 else norm / rnorm)
    P /= f
    R *= f / math.sqrt(norm)
    return AL, P.reshape(len(qa), d, len(qc), order="F"), R.reshape(len(qc), d, len(qb), order="F"), BR, qL, qc, qB


def _chain(case, seed):
    """A right-canonical state of a short chain and its bond charges."""
    rng = np.random.default_rng([seed, case["m"], case["L"]])
    qphys = _charges(case)
    d, nq = qphys.shape
    L, m = case["L"], case["m"]
    total = np.array([L % 2] * nq, dtype=np.int64)
    fwd, back = [{(0,) * nq: 1}], [{tuple(total): 1}]
    for k in range(L):
        f, b = {}, {}
        for p in map(tuple, qphys.tolist()):
            for c, n in fwd[-1].items():
                t = tuple(x + y for x, y in zip(c, p))
                f[t] = min(f.get(t, 0) + n, m)
            for c, n in back[-1].items():
                t = tuple(x - y for x, y in zip(c, p))
                b[t] = min(b.get(t, 0) + n, m)
        fwd.append(f)
        back.append(b)
    back = back[::-1]
    q = []
    for k in range(L + 1):
        both = {c: min(n, back[k][c]) for c, n in fwd[k].items() if c in back[k]}
        q.append(_bond_charges(_pick(both, m, [0.0] * nq), nq))
    A = [None] * L
    for k in range(L - 1, -1, -1):
        M = np.zeros((len(q[k]), d * len(q[k + 1])))
        qcol = _cols(q[k + 1], qphys)
        for r, c in _blocks(q[k], qcol):
            g = rng.standard_normal((len(c), len(r)))
            M[np.ix_(r, c)] = np.linalg.qr(g)[0].T if len(c) >= len(r) else 0.0
            if len(c) < len(r):
                M[np.ix_(r[:len(c)], c)] = np.linalg.qr(g.T)[0].T[:, :len(c)]
        A[k] = M.reshape(len(q[k]), d, len(q[k + 1]))
    A[0] = A[0] / np.linalg.norm(A[0])
    return A, q


# ------------------------------------------------------------ the passes

def _up(case, A, ql, qr):
    if not case["qn"]:
        return pkg.site_from_dense(pkg.default_context(), A)
    q = _charges(case)
    return pkg.site_from_dense(pkg.default_context(), A, ql, q, qr, q.shape[1])


def prepare(case, seed):
    ctx = pkg.default_context()
    nq = _charges(case).shape[1]
    if case["path"] in ("sweep", "evolve"):
        A, q = _chain(case, seed)
        psi = pkg.MPS(A, oc=1, qphys=_charges(case) if nq else None, qbond=q if nq else None, ctx=ctx,
                      canonical=True)
        return dict(case=case, ctx=ctx, nq=nq, psi=psi, mpo=_mpo(case, case["L"]))
    AL, P, R, BR, qL, qc, qB = _host(case, seed)
    n = len(AL) + len(BR) + 2
    mpo = _mpo(case, n)
    i = len(AL) + 1                                  # the centre pair is (i, i + 1)
    from dmrjtensor_jl_amd.network import makeBoundary
    E = makeBoundary(ctx, True, nq, qL[0] if nq else None)
    for k, A in enumerate(AL):
        E = pkg.Lupdate(E, _up(case, A, qL[k], qL[k + 1]), mpo, k + 1)
    F = makeBoundary(ctx, False, nq, qB[-1] if nq else None)
    for k in range(len(BR) - 1, -1, -1):
        F = pkg.Rupdate(F, _up(case, BR[k], qB[k], qB[k + 1]), mpo, i + 2 + k)
    s = dict(case=case, ctx=ctx, nq=nq, mpo=mpo, i=i, L=E, R=F, P=_up(case, P, qL[-1], qc),
             Q=_up(case, R, qc, qB[0]))
    if case["path"] == "step3s":
        s["Lenv"], s["Renv"] = pkg.environment(n), pkg.environment(n)
        if case["dir"] > 0:                          # the centre i and its right environment
            s["Lenv"][i], s["Renv"][i] = E, pkg.Rupdate(F, s["Q"], mpo, i + 1)
        else:
            s["Lenv"][i + 1], s["Renv"][i + 1] = pkg.Lupdate(E, s["P"], mpo, i), F
    return s


def _theta(ctx, a, b):
    h = C.c_void_p()
    ctx.call("dmrj_theta2", a.h, b.h, C.byref(h))
    return pkg.DeviceTensor(ctx, h)


def _pair(s, a, b):
    """The two-site state of a pair of tensors, read when asked for."""
    def read():
        t = _theta(s["ctx"], a, b)
        return t.to_dense(s["nq"])[0]
    return read


class _Pair:
    """The two sites a single-site step works on, indexed as an MPS."""

    def __init__(self, s):
        self.ctx, self.n = s["ctx"], len(s["mpo"])
        self.t = {s["i"]: s["P"].copy(), s["i"] + 1: s["Q"].copy()}

    def __len__(self):
        return self.n

    def __getitem__(self, i):
        return self.t[i]

    def __setitem__(self, i, v):
        self.t[i] = v


def _vector(psi):
    """The state vector of a short chain."""
    def read():
        A, _ = psi.to_dense()
        v = A[0].reshape(A[0].shape[1], -1)
        for a in A[1:]:
            v = (v @ a.reshape(a.shape[0], -1)).reshape(-1, a.shape[2])
        return v.reshape(-1)
    return read


def _svd(s, AA, m, cutoff, direction):
    l, r, te, k = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
    sv = np.zeros(4 * m + 16)
    s["ctx"].call("dmrj_svd_trunc2", AA.h, m, 2, cutoff, direction, C.byref(l), C.byref(r), C.byref(te),
                  C.byref(k), sv.ctypes.data_as(C.POINTER(C.c_double)), len(sv))
    return pkg.DeviceTensor(s["ctx"], l), pkg.DeviceTensor(s["ctx"], r), te.value, k.value, sv[:k.value]


def run(s):
    case, ctx, nq = s["case"], s["ctx"], s["nq"]
    path = case["path"]
    if path == "envs":
        E = pkg.Lupdate(s["L"], s["P"], s["mpo"], s["i"])
        F = pkg.Rupdate(s["R"], s["Q"], s["mpo"], s["i"] + 1)
        return Results(left=lambda: E.to_dense(nq)[0], right=lambda: F.to_dense(nq)[0])
    if path == "bond":
        m = case["m"]
        sv = np.zeros(4 * m + 16)
        nl, nr, e, te, kept = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_double(), C.c_int64()
        ctx.call("dmrj_twostep", s["L"].h, s["R"].h, s["P"].h, s["Q"].h, s["mpo"].device(ctx, s["i"]),
                 s["mpo"].device(ctx, s["i"] + 1), case["dir"], m, 2, 0.0, PREC[case["precision"]], C.byref(nl),
                 C.byref(nr), C.byref(e), C.byref(te), C.byref(kept), sv.ctypes.data_as(C.POINTER(C.c_double)),
                 len(sv))
        a, b = pkg.DeviceTensor(ctx, nl), pkg.DeviceTensor(ctx, nr)
        return Results(energy=e.value, truncerr=te.value, kept=kept.value, svals=sv[:kept.value],
                       state=_pair(s, a, b))
    if path == "step3s":
        psi = _Pair(s)
        params = pkg.algvars(psi, maxm=case["m"])
        params.method = "3S"
        d = case["dir"]
        i = s["i"] if d > 0 else s["i"] + 1
        pkg.step3S(1, d, i, s["i"], s["i"] + 1, psi, s["mpo"], s["Lenv"], s["Renv"], params)
        return Results(energy=params.energy, truncerr=params.truncerr, kept=params.biggestm,
                       state=_pair(s, psi[s["i"]], psi[s["i"] + 1]))
    if path == "tdvp":
        i, dt, mpo = s["i"], -0.02j, s["mpo"]
        AA = _theta(ctx, s["P"], s["Q"])
        new, _ = pkg.krylovTimeEvol2(s["L"], s["R"], AA, mpo, i, 12, dt, energy=False)
        ctx.call("dmrj_normalize", new.h)
        a, b, te, kept, sv = _svd(s, new, case["m"], 1e-12, case["dir"])
        if case["dir"] > 0:
            E = pkg.Lupdate(s["L"], a, mpo, i)
            ctx.call("dmrj_normalize", b.h)
            b, _ = pkg.krylovTimeEvol1(E, s["R"], b, mpo, i + 1, 12, dt, energy=False)
        else:
            E = pkg.Rupdate(s["R"], b, mpo, i + 1)
            ctx.call("dmrj_normalize", a.h)
            a, _ = pkg.krylovTimeEvol1(s["L"], E, a, mpo, i, 12, dt, energy=False)
        return Results(truncerr=te, kept=kept, state=_pair(s, a, b))
    psi = s["psi"].copy()                            # a pass starts from the same state
    if path == "sweep":
        e = pkg.dmrg(psi, s["mpo"], m=case["m"], sweeps=1, cutoff=1e-12)
        return Results(energy=e, state=_vector(psi))
    e, _, _ = pkg.tdvp_twosite(psi, s["mpo"], m=case["m"], cutoff=1e-12, r=12, prefactor=-0.5j)
    return Results(energy=e, state=_vector(psi))


PREC = {"f64": 0, "bf16x3": 1, "f16x3": 2}


# ------------------------------------------------------------ work and exact values

def _dims(q):
    return {c: len(i) for c, i in _groups(q).items()}


def _add(c, p, sign=1):
    return tuple(x + sign * y for x, y in zip(c, p))


def _env_work(na, nb, qphys, D, deltas):
    """Flops of one environment update: bra and ket blocks of the old bond
    joined to the new one, the cheaper order of the two GEMMs."""
    flops = 0.0
    for w in deltas:
        for c, n in na.items():
            k = na.get(_add(c, w, -1), 0)
            for p in map(tuple, qphys.tolist()):
                flops += 2.0 * n * k * nb.get(_add(c, p), 0)
                flops += 2.0 * k * nb.get(_add(_add(c, w, -1), p), 0) * nb.get(_add(c, p), 0)
    return flops


def work(case):
    """Bytes: every input tensor once, every output once.  Flops: the
    block-sparse contractions, and 8 K^2 N (K <= N the sides of a sector) for
    the singular values and both sets of vectors."""
    qphys = _charges(case)
    d, nq = qphys.shape
    model = case["model"]
    deltas = [(0,) * nq] * (6 if model == "hubbard" else 5)
    if nq == 1:
        deltas = [(0,), (2,), (-2,), (0,), (0,)]
    if nq == 2:
        deltas = [(0, 0), (1, 1), (-1, -1), (1, -1), (-1, 1), (0, 0)]
    phys = list(map(tuple, qphys.tolist()))

    def env_bytes(n):
        return 8.0 * sum(k * n.get(_add(c, w, -1), 0) for w in deltas for c, k in n.items())

    def site_bytes(n, k):
        return 8.0 * sum(x * k.get(_add(c, p), 0) for c, x in n.items() for p in phys)

    def two(na, nb, nb2, steps):
        """H_eff applications on a two-site (or one-site) tensor and its SVD."""
        pairs = [(p, r) for p in phys for r in phys]
        size, heff = 0.0, 0.0
        for c, n in na.items():
            for p, r in pairs:
                cols = nb.get(_add(_add(c, p), r), 0)
                size += n * cols
                for w in deltas:
                    heff += 2.0 * n * na.get(_add(c, w), 0) * cols + 2.0 * n * cols * nb.get(
                        _add(_add(_add(c, p), r), w), 0)
        svd = 0.0
        cent = {}
        for c, n in na.items():
            for p in phys:
                cent[_add(c, p)] = cent.get(_add(c, p), 0) + n
        for q, rows in cent.items():
            cols = sum(nb.get(_add(q, p), 0) for p in phys)
            svd += 8.0 * min(rows, cols) ** 2 * max(rows, cols)
        return size, heff * steps, svd

    if case["path"] in ("sweep", "evolve"):
        q = _chain(case, 0)[1]
        n = [_dims(x) for x in q]
        flops = 0.0
        nbytes = 2.0 * sum(site_bytes(n[k], n[k + 1]) for k in range(case["L"]))
        for k in range(case["L"] - 1):
            _, h, v = two(n[k], n[k + 2], None, 2 if case["path"] == "sweep" else 24)
            e = _env_work(n[k], n[k + 1], qphys, None, deltas)
            if case["path"] == "sweep":
                flops += 2 * (h + v) + 3 * e
            else:
                flops += 4 * (h + v) + 4 * e
        return dict(bytes=nbytes, flops=flops)
    qL, qc, qB = _bonds(case)
    na, nc, nb = _dims(qL[-1]), _dims(qc), _dims(qB[0])
    envs = env_bytes(na) + env_bytes(nb)
    sites = site_bytes(na, nc) + site_bytes(nc, nb)
    if case["path"] == "envs":
        neg = {tuple(-x for x in c): n for c, n in nb.items()}, {tuple(-x for x in c): n for c, n in nc.items()}
        return dict(bytes=envs + sites + 2 * env_bytes(nc),
                    flops=_env_work(na, nc, qphys, None, deltas) + _env_work(neg[0], neg[1], qphys, None, deltas))
    size, heff, svd = two(na, nb, None, 2)
    if case["path"] == "bond":
        return dict(bytes=envs + 2 * sites, flops=heff + svd)
    if case["path"] == "step3s":
        one = heff / (2 * d)
        return dict(bytes=env_bytes(na) + 2 * sites, flops=one + svd * len(deltas) / d)
    return dict(bytes=envs + 4 * sites, flops=4 * (6 * heff * (1 + 1.0 / d) + svd))


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(x):
    return torch.as_tensor(np.ascontiguousarray(x), device=_dev())


def _mul(a, b, ax):
    if a.is_complex() != b.is_complex():
        a, b = a.to(torch.complex128), b.to(torch.complex128)
    return torch.tensordot(a, b, dims=ax)


def _lup(L, A, W, B=None):
    """L'[b', u, b] = sum L[a', w, a] conj(A[a', k, b']) W[w, j, k, u] A[a, j, b]"""
    T = _mul(L, A.conj(), ([0], [0]))
    T = _mul(T, W, ([0, 2], [0, 2]))
    return _mul(T, A, ([0, 2], [0, 1]))


def _rup(R, A, W):
    """R'[a, w, a'] = sum A[a, j, b] W[w, j, k, u] conj(A[a', k, b']) R[b, u, b']"""
    T = _mul(A.conj(), R, ([2], [2]))
    T = _mul(W, T, ([2, 3], [1, 3]))
    return _mul(A, T, ([1, 2], [1, 3]))


def _heff2(L, R, x, W1, W2):
    T = _mul(L, x, ([2], [0]))
    W = torch.tensordot(W1, W2, dims=([3], [0]))            # w j1 k1 j2 k2 u
    T = _mul(T, W, ([1, 2, 3], [0, 1, 3]))
    return _mul(T, R, ([1, 4], [0, 1]))


def _heff1(L, R, x, W):
    T = _mul(L, x, ([2], [0]))
    T = _mul(T, W, ([1, 2], [0, 1]))
    return _mul(T, R, ([1, 3], [0, 1]))


def _dot(x, y):
    return complex(torch.sum(x.conj() * y).item()) if x.is_complex() or y.is_complex() else torch.sum(x * y).item()


def _keep(sv, m, cutoff):
    keep, acc = len(sv), 0.0
    while keep > 0 and acc + sv[keep - 1] ** 2 < cutoff:
        acc += sv[keep - 1] ** 2
        keep -= 1
    return max(min(keep, m), min(2, len(sv)))


def _trunc(x, m, cutoff, direction, qrow, qcol):
    """Truncated SVD by charges: (left, right, weights, truncation error) with
    the weights on the side the centre moves to."""
    a, d1, d2, b = x.shape
    M = x.reshape(a * d1, d2 * b).cpu()
    parts = []
    for r, c in _blocks(qrow, qcol):
        u, v, w = torch.linalg.svd(M[torch.as_tensor(r)][:, torch.as_tensor(c)], full_matrices=False)
        parts.append((r, c, u, v.numpy(), w))
    order = sorted(((-p[3][k], n, k) for n, p in enumerate(parts) for k in range(len(p[3]))))
    sv = np.array([-o[0] for o in order])
    keep = _keep(sv, m, cutoff)
    nk = [0] * len(parts)
    for _, n, _ in order[:keep]:
        nk[n] += 1
    scale = 1.0 / np.linalg.norm(sv[:keep])
    U, V = torch.zeros(a * d1, keep, dtype=M.dtype), torch.zeros(keep, d2 * b, dtype=M.dtype)
    qn, o = [], 0
    for (r, c, u, v, w), k in zip(parts, nk):
        wgt = torch.as_tensor(v[:k] * scale).to(M.dtype)
        U[torch.as_tensor(r), o:o + k] = u[:, :k] * (1.0 if direction > 0 else wgt)
        V[o:o + k, torch.as_tensor(c)] = (wgt[:, None] if direction > 0 else 1.0) * w[:k]
        qn += [qrow[r[0]]] * k
        o += k
    return (U.reshape(a, d1, keep).to(x.device), V.reshape(keep, d2, b).to(x.device), sv[:keep] * scale,
            float(np.sum(sv[keep:] ** 2)), np.array(qn).reshape(keep, qrow.shape[1]))


def _link_charges(Ws, qphys):
    """Charge of every MPO link: u carries w's charge plus q(bra) - q(ket)."""
    out = [np.zeros((Ws[0].shape[0], qphys.shape[1]), dtype=np.int64)]
    for W in Ws:
        nxt = np.zeros((W.shape[3], qphys.shape[1]), dtype=np.int64)
        for w, j, k, u in torch.nonzero(W).tolist():
            nxt[u] = out[-1][w] + qphys[k] - qphys[j]
        out.append(nxt)
    return out


def _lanczos2(L, R, a, b, W1, W2):
    AA = _mul(a, b, ([2], [0]))
    H = _heff2(L, R, AA, W1, W2)
    AA = AA / torch.linalg.norm(AA)
    a1 = _dot(AA, H)
    p2 = H - a1 * AA
    b1 = torch.linalg.norm(p2).item()
    if b1 <= 1e-10:
        return a1, AA
    p2 = p2 / b1
    a2 = _dot(p2, _heff2(L, R, p2, W1, W2))
    e, u = np.linalg.eigh(np.array([[a1, b1], [b1, a2]]))
    if (u[0, 0] < 0) != (a2 >= a1):                  # the sign dmrj_lanczos2 gives the Ritz vector
        u = -u
    return float(e[0]), u[0, 0] * AA + u[1, 0] * p2


def _krylov(apply, x, r):
    """Krylov basis (fully orthogonal) and tridiagonal of r applications."""
    V, al, be = [x / torch.linalg.norm(x)], [], []
    for j in range(r):
        w = apply(V[-1])
        al.append(np.real(_dot(V[-1], w)))
        if j == r - 1:
            break
        for _ in range(2):
            for v in V:
                w = w - _dot(v, w) * v
        b = torch.linalg.norm(w).item()
        if b <= 1e-10:
            break
        be.append(b)
        V.append(w / b)
    n = len(V)
    T = np.diag(al[:n]) + np.diag(be[:n - 1], 1) + np.diag(be[:n - 1], -1)
    return V, np.linalg.eigh(T)


def _evolve(apply, x, dt):
    V, (lam, Z) = _krylov(apply, x.to(torch.complex128), 12)
    c = Z @ (np.exp(dt * lam) * Z[0])
    return sum(complex(ck) * v for ck, v in zip(c, V)), float(lam[0])


def exact(case, seed):
    """The same pass in 64 bits with dense torch tensors."""
    qphys = _charges(case)
    if case["path"] in ("sweep", "evolve"):
        return _exact_chain(case, seed)
    AL, P, R, BR, qL, qc, qB = _host(case, seed)
    n = len(AL) + len(BR) + 2
    Ws = [_t(W) for W in _mpo(case, n).H]
    i = len(AL)
    E = torch.ones((1, 1, 1), dtype=torch.float64, device=_dev())
    F = E
    for k, A in enumerate(AL):
        E = _lup(E, _t(A), Ws[k])
    for k in range(len(BR) - 1, -1, -1):
        F = _rup(F, _t(BR[k]), Ws[i + 2 + k])
    P, R = _t(P), _t(R)
    if case["path"] == "envs":
        return dict(left=_lup(E, P, Ws[i]).cpu(), right=_rup(F, R, Ws[i + 1]).cpu())
    rows, cols = _join(qL[-1], qphys), _cols(qB[0], qphys)
    if case["path"] == "bond":
        e, AA = _lanczos2(E, F, P, R, Ws[i], Ws[i + 1])
        a, b, sv, te, _ = _trunc(AA, case["m"], 0.0, case["dir"], rows, cols)
        return dict(energy=e, truncerr=te, kept=None, svals=sv, state=_mul(a, b, ([2], [0])).cpu())
    if case["path"] == "step3s":
        return _exact_3s(case, E, F, P, R, Ws, i, qphys, qL[-1], qc, qB[0])
    dt = -0.02j
    AA, _ = _evolve(lambda v: _heff2(E, F, v, Ws[i], Ws[i + 1]), _mul(P, R, ([2], [0])), dt)
    AA = AA / torch.linalg.norm(AA)
    a, b, sv, te, _ = _trunc(AA, case["m"], 1e-12, case["dir"], rows, cols)
    if case["dir"] > 0:
        E2 = _lup(E, a, Ws[i])
        b, _ = _evolve(lambda v: _heff1(E2, F, v, Ws[i + 1]), b / torch.linalg.norm(b), dt)
    else:
        F2 = _rup(F, b, Ws[i + 1])
        a, _ = _evolve(lambda v: _heff1(E, F2, v, Ws[i]), a / torch.linalg.norm(a), dt)
    return dict(truncerr=te, kept=None, state=_mul(a, b, ([2], [0])).cpu())


def _exact_3s(case, E, F, P, R, Ws, i, qphys, qa, qc, qb):
    """Single-site Lanczos, the tensor joined with its expansion along the
    moving bond, truncated SVD, the neighbour absorbed."""
    m = case["m"]
    deltas = _link_charges(Ws, qphys)
    if case["dir"] > 0:
        G = _rup(F, R, Ws[i + 1])
        V, (lam, Z) = _krylov(lambda v: _heff1(E, G, v, Ws[i]), P, 2)
        A = sum(float(z) * v for z, v in zip(Z[:, 0], V))
        A = A if _dot(A, P) >= 0 else -A
        X = _mul(_mul(E, A, ([2], [0])), Ws[i], ([1, 2], [0, 1])).permute(0, 2, 3, 1)    # a' k u b
        T = torch.cat([A, X.reshape(A.shape[0], A.shape[1], -1)], dim=2)
        q2 = np.concatenate([qc, (deltas[i + 1][:, None, :] + qc[None, :, :]).reshape(T.shape[2] - len(qc), -1)])
        T = T / torch.linalg.norm(T)
        a, b, sv, te, _ = _trunc(T[:, :, None, :], m, 0.0, 1, _join(qa, qphys), q2)
        b = _mul(b[:, 0, :qc.shape[0]], R, ([1], [0]))
    else:
        G = _lup(E, P, Ws[i])
        V, (lam, Z) = _krylov(lambda v: _heff1(G, F, v, Ws[i + 1]), R, 2)
        A = sum(float(z) * v for z, v in zip(Z[:, 0], V))
        A = A if _dot(A, R) >= 0 else -A
        X = _mul(A, F, ([2], [0]))                                                     # c j u b'
        X = _mul(Ws[i + 1], X, ([1, 3], [1, 2]))                                       # w k c b'
        X = X.permute(0, 2, 1, 3)                                                      # w c k b'
        T = torch.cat([A, X.reshape(-1, A.shape[1], A.shape[2])], dim=0)
        q2 = np.concatenate([qc, (qc[None, :, :] + deltas[i + 1][:, None, :]).reshape(T.shape[0] - len(qc), -1)])
        T = T / torch.linalg.norm(T)
        a, b, sv, te, _ = _trunc(T[:, None, :, :], m, 0.0, -1, q2, _cols(qb, qphys))
        a = _mul(P, a[:qc.shape[0], 0, :], ([2], [0]))
    return dict(energy=float(lam[0]), truncerr=te, kept=None, state=_mul(a, b, ([2], [0])).cpu())


def _exact_chain(case, seed):
    qphys = _charges(case)
    A, q = _chain(case, seed)
    L, m = case["L"], case["m"]
    A = [torch.as_tensor(x) for x in A]
    Ws = [torch.as_tensor(W) for W in _mpo(case, L).H]
    E, F = [None] * L, [None] * L
    E[0] = F[L - 1] = torch.ones((1, 1, 1), dtype=torch.float64)
    for k in range(L - 1, 0, -1):
        F[k - 1] = _rup(F[k], A[k], Ws[k])
    energy = 0.0
    if case["path"] == "sweep":
        for k, d in [(k, 1) for k in range(L - 1)] + [(k, -1) for k in range(L - 2, -1, -1)]:
            c = k if d > 0 else k + 1
            A[c] = A[c] / torch.linalg.norm(A[c])
            energy, AA = _lanczos2(E[k], F[k + 1], A[k], A[k + 1], Ws[k], Ws[k + 1])
            A[k], A[k + 1], _, _, q[k + 1] = _trunc(AA, m, 1e-12, d, _join(q[k], qphys), _cols(q[k + 2], qphys))
            if d > 0:
                E[k + 1] = _lup(E[k], A[k], Ws[k])
            else:
                F[k] = _rup(F[k + 1], A[k + 1], Ws[k + 1])
    else:
        dt = -0.5j / (L - 1) / 2
        for k in range(L - 1):
            AA, _ = _evolve(lambda v: _heff2(E[k], F[k + 1], v, Ws[k], Ws[k + 1]), _mul(A[k], A[k + 1], ([2], [0])), dt)
            AA = AA / torch.linalg.norm(AA)
            A[k], b, _, _, q[k + 1] = _trunc(AA, m, 1e-12, 1, _join(q[k], qphys), _cols(q[k + 2], qphys))
            E[k + 1] = _lup(E[k], A[k], Ws[k])
            b, energy = _evolve(lambda v: _heff1(E[k + 1], F[k + 1], v, Ws[k + 1]), b / torch.linalg.norm(b), dt)
            A[k + 1] = b / torch.linalg.norm(b)
    v = A[0].reshape(A[0].shape[1], -1)
    for a in A[1:]:
        v = _mul(v, a, ([1], [0])).reshape(-1, a.shape[2])
    return dict(energy=energy, state=v.reshape(-1))
