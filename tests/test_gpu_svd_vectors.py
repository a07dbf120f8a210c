"""Singular vectors that carry little or no weight: the canonical factor of the
truncated SVD is an isometry over everything that is kept, and a weak charge
sector is solved to its own scale."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _svd(pkg, ctx, t, nq, direction, m=0):
    l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
    sv = np.zeros(8192)
    ctx.call("dmrj_svd_trunc2", t.h, m, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
             pkg._lib.dptr(sv), len(sv))
    L = pkg.DeviceTensor(ctx, l).to_dense(nq)[0]
    Rt = pkg.DeviceTensor(ctx, r).to_dense(nq)[0]
    return L.reshape(-1, kk.value), Rt.reshape(kk.value, -1), sv[:kk.value]


def _dense(pkg, ctx, M, direction):
    return _svd(pkg, ctx, pkg.site2_from_dense(ctx, M.reshape(M.shape[0], 1, 1, M.shape[1])), 0, direction)


def _isometry(L, Rt, direction):
    Q = L if direction > 0 else Rt.conj().T
    return np.max(np.abs(Q.conj().T @ Q - np.eye(Q.shape[1])))


def _phases(M, rng):
    return np.exp(2j * np.pi * rng.random(M.shape[0]))[:, None] * M * np.exp(2j * np.pi * rng.random(M.shape[1]))[None, :]


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("tiny", [1e-155, 1e-160, 1e-161])
def test_residuals_below_the_range_of_squares(pkg, ctx, tiny, cplx, direction):
    """Columns that equal a multiple of a unit vector up to 1e-155 .. 1e-161 of
    the norm, before columns of order one: the squares of what a reflector
    leaves of them are subnormal numbers of few bits, or vanish."""
    rng = np.random.default_rng(5)
    R, Cc = 40, 33
    M = 0.1 * rng.standard_normal((R, Cc))
    M[0] = 0.0
    M[:, :6] = 0.0
    M[0, :6] = 1.0
    M[1:, 1:6] = tiny * rng.standard_normal((R - 1, 5))
    if cplx:
        M = _phases(M, rng)
    M = M / np.linalg.norm(M)
    if direction < 0:
        M = np.ascontiguousarray(M.T)
    L, Rt, sv = _dense(pkg, ctx, M, direction)
    n = max(R, Cc)
    want = np.linalg.svd(M, compute_uv=False)
    assert np.max(np.abs(sv - want)) <= 2 * n * EPS
    assert np.max(np.abs(L @ Rt - M)) <= 8 * n * EPS
    assert _isometry(L, Rt, direction) <= 1e-13 + 4 * n * EPS


def _charged(cplx, rng, dims, rdims=None, edit=None):
    """A two-site tensor of spins 1/2 whose bonds hold dims[q] (right: rdims[q])
    states of charge q, and the matrix of its centre sectors; edit(Q, sector)
    changes a sector."""
    ql, qr = (np.array([[c] for c in sorted(d) for _ in range(d[c])], dtype=np.int32) for d in (dims, rdims or dims))
    qp = np.array([[1], [-1]], dtype=np.int32)
    row = (ql[:, 0][:, None] + qp[:, 0][None, :]).ravel()
    col = (qr[:, 0][None, :] - qp[:, 0][:, None]).ravel()
    M = np.zeros((len(row), len(col)), dtype=complex if cplx else float)
    sectors = {}
    for Q in sorted(set(row) & set(col)):
        at = np.ix_(np.flatnonzero(row == Q), np.flatnonzero(col == Q))
        S = rng.standard_normal((len(at[0]), at[1].size)) / len(row)
        if cplx:
            S = _phases(S, rng)
        M[at] = S if edit is None else edit(int(Q), S)
        sectors[int(Q)] = at
    return M.reshape(len(ql), 2, 2, len(qr)), (ql, qp, qp, qr, 1), M, sectors


DIMS = {-4: 7, -2: 12, 0: 40, 2: 27, 4: 3}


def _check_sectors(M, sectors, L, Rt, sv, direction):
    """Values, products and the isometry, every sector to its own norm."""
    n = max(at[0].size + at[1].size for at in sectors.values()) // 2
    P = L @ Rt
    norm = np.linalg.norm(M)
    assert np.all(np.isfinite(L)) and np.all(np.isfinite(Rt))
    want = []
    for at in sectors.values():
        w = np.linalg.svd(M[at], compute_uv=False)
        want += [(x, np.linalg.norm(w)) for x in w]
        assert np.max(np.abs(P[at] * norm - M[at])) <= 16 * n * EPS * np.linalg.norm(w)
    want.sort(key=lambda p: -p[0])
    assert len(sv) == len(want)
    for got, (w, scale) in zip(sv, want):
        assert abs(got * norm - w) <= 4 * n * EPS * scale
    assert _isometry(L, Rt, direction) <= 1e-13 + 4 * n * EPS


WIDE = {-4: 15, -2: 30, 0: 90, 2: 55, 4: 8}
TWINS = {-2: 20, 0: 31, 2: 20}   # sectors of 20, 51, 51 and 20 rows


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("bonds", [(DIMS, DIMS), (DIMS, WIDE), (TWINS, TWINS)], ids=["square", "wide", "twins"])
@pytest.mark.parametrize("batching", [0, 1, 2, 3])
@pytest.mark.parametrize("kind", ["real", "gram", "complex"])
def test_eigensolves_of_several_sectors(pkg, ctx, kind, batching, bonds, direction):
    """What the block Jacobi leaves to the eigensolves (all of it here): sectors
    of six sizes, or of two sizes twice, in one call, every way of batching
    them.  The Gram form is accurate to n eps in the squares of the values."""
    A, charges, M, sectors = _charged(kind == "complex", np.random.default_rng(29), *bonds)
    t = pkg.site2_from_dense(ctx, A, *charges)
    ctx.set_jacobi_sweeps(0)
    ctx.set_eig_batching(batching)
    ctx.set_svd_backend(5 if kind == "gram" else 0)
    try:
        L, Rt, sv = _svd(pkg, ctx, t, 1, direction)
    finally:
        ctx.set_jacobi_sweeps(40)
        ctx.set_eig_batching(1)
        ctx.set_svd_backend(0)
    if kind != "gram":
        _check_sectors(M, sectors, L, Rt, sv, direction)
        return
    norm, n = np.linalg.norm(M), max(M.shape)
    want = np.sort(np.concatenate([np.linalg.svd(M[at], compute_uv=False) for at in sectors.values()]))[::-1] / norm
    assert np.max(np.abs(sv ** 2 - want ** 2)) <= 4 * n * EPS
    assert np.max(np.abs(L @ Rt * norm - M)) <= 8 * n * EPS * norm
    assert _isometry(L, Rt, direction) <= 1e-13 + 4 * n * EPS


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("shape", [(40, 33), (33, 70), (130, 257)])
def test_eigensolve_of_sectors_with_zero_rows(pkg, ctx, shape, cplx, direction):
    """Rows and columns of zeros in what is left to the eigensolves: finite
    factors whose product is the tensor."""
    R, Cc = shape
    rng = np.random.default_rng(R + Cc)
    M = np.zeros((R, Cc))
    M[1:1 + R // 3, :Cc // 4] = rng.standard_normal((R // 3, Cc // 4))
    if cplx:
        M = _phases(M, rng)
    M = M / np.linalg.norm(M)
    n = max(R, Cc)
    ctx.set_jacobi_sweeps(0)
    try:
        L, Rt, sv = _dense(pkg, ctx, M, direction)
    finally:
        ctx.set_jacobi_sweeps(40)
    assert np.max(np.abs(sv - np.linalg.svd(M, compute_uv=False))) <= 4 * n * EPS
    assert np.max(np.abs(L @ Rt - M)) <= 16 * n * EPS


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("limit", [1, 2, 4])
def test_sectors_that_do_not_converge(pkg, ctx, limit, cplx, direction):
    """Sweep limits that the diagonal sector keeps and the others do not: what
    has converged stays, the others take the eigensolves."""
    A, charges, M, sectors = _charged(cplx, np.random.default_rng(31), DIMS,
                                      edit=lambda q, S: np.diag(np.linspace(0.3, 1.0, len(S))) if q == -1 else S)
    t = pkg.site2_from_dense(ctx, A, *charges)
    ctx.set_jacobi_sweeps(limit)
    try:
        L, Rt, sv = _svd(pkg, ctx, t, 1, direction)
    finally:
        ctx.set_jacobi_sweeps(40)
    _check_sectors(M, sectors, L, Rt, sv, direction)


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("scale", [1e-170, 3e-154, 1e153])
def test_squared_norm_out_of_range(pkg, ctx, scale, cplx, direction):
    """Norms whose squares are no normal numbers, sectors of 3 .. 67 rows; and the
    weight that a truncation discards, in the tensor's own units."""
    A, charges, M, sectors = _charged(cplx, np.random.default_rng(37), DIMS)
    f = scale / np.linalg.norm(M)
    t = pkg.site2_from_dense(ctx, A * f, *charges)
    L, Rt, sv = _svd(pkg, ctx, t, 1, direction)
    _check_sectors(M, sectors, L, Rt, sv, direction)
    te, kept = C.c_double(), 100
    l, r, kk = C.c_void_p(), C.c_void_p(), C.c_int64()
    ctx.call("dmrj_svd_trunc2", t.h, kept, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
             pkg._lib.dptr(sv), len(sv))
    want = np.sort(np.concatenate([np.linalg.svd(M[at], compute_uv=False) for at in sectors.values()]))[::-1]
    want = want / np.linalg.norm(want) * scale
    # (squares of 1e-154 are subnormal: half a unit of 5e-324)
    assert abs(te.value - np.sum(want[kept:] ** 2)) <= 1e-12 * np.sum(want[kept:] ** 2) + 1e-322


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("weak", [1e-6, 1e-20, 1e-40])
@pytest.mark.parametrize("Q", [5, 1, -1])
def test_weak_sector(pkg, ctx, Q, weak, cplx, direction):
    """One charge sector far below the others: its values and vectors are
    accurate to its own norm (sectors of 3, 43 .. 67 and 19 .. 52 rows)."""
    A, charges, M, sectors = _charged(cplx, np.random.default_rng(23), DIMS,
                                      edit=lambda q, S: S * (weak if q == Q else 1.0))
    assert Q in sectors
    t = pkg.site2_from_dense(ctx, A, *charges)
    L, Rt, sv = _svd(pkg, ctx, t, 1, direction)
    _check_sectors(M, sectors, L, Rt, sv, direction)


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("shape", [(90, 64), (200, 230), (500, 480)])
def test_truncation_inside_a_weak_tail(pkg, ctx, shape, cplx, direction):
    """A flat spectrum and a tail of 1e-10 to 1e-13 of the largest value, cut in its
    middle: what is kept is the best approximation, to the rounding of the
    solver, and the factor an isometry."""
    R, Cc = shape
    rng = np.random.default_rng(R + 3 * Cc)
    K, n = min(R, Cc), max(R, Cc)
    s = np.ones(K)
    s[K // 2:] = np.logspace(-10, -13, K - K // 2)
    U, V = (np.linalg.qr(rng.standard_normal((d, K)) + (1j * rng.standard_normal((d, K)) if cplx else 0.0))[0]
            for d in (R, Cc))
    M = (U * s) @ V.conj().T / np.linalg.norm(s)
    t = pkg.site2_from_dense(ctx, M.reshape(R, 1, 1, Cc))
    keep = 3 * K // 4
    L, Rt, sv = _svd(pkg, ctx, t, 0, direction, keep)
    assert len(sv) == keep
    best = np.linalg.norm(np.linalg.svd(M, compute_uv=False)[keep:])
    assert np.linalg.norm(L @ Rt - M, 2) <= best + 16 * n * EPS
    assert _isometry(L, Rt, direction) <= 1e-13 + 4 * n * EPS


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("sweeps", [40, 0], ids=["jacobi", "eigensolve"])
@pytest.mark.parametrize("shape", [(9, 12), (16, 16), (210, 16), (16, 230), (40, 33), (33, 70), (130, 257), (280, 300)])
def test_vanishing_values_keep_an_isometry(pkg, ctx, shape, sweeps, cplx, direction):
    """Rank-deficient sectors, everything kept: equal columns (singular values
    at the rounding level), zero rows and columns (exact zeros), one element.  The bounds
    are those of the vectors with weight."""
    R, Cc = shape
    n = max(R, Cc)
    for kind in ("equal", "zeros", "one"):
        rng = np.random.default_rng(R * 17 + Cc)
        if kind == "equal":
            M = np.repeat(rng.standard_normal((R, -(-Cc // 4))), 4, axis=1)[:, :Cc]
            M[rng.permutation(R)[:R // 5]] = 0.0
        elif kind == "one":
            M = np.zeros((R, Cc))
            M[R // 2, Cc // 2] = 1.0
        else:
            M = np.zeros((R, Cc))
            M[:R // 3, 1:1 + Cc // 4] = rng.standard_normal((R // 3, Cc // 4))
        if cplx:
            M = _phases(M, rng)
        M = M / np.linalg.norm(M)
        ctx.set_jacobi_sweeps(sweeps)
        try:
            L, Rt, sv = _dense(pkg, ctx, M, direction)
        finally:
            ctx.set_jacobi_sweeps(40)
        assert len(sv) == min(R, Cc)
        assert np.max(np.abs(sv - np.linalg.svd(M, compute_uv=False))) <= 2 * n * EPS
        assert np.max(np.abs(L @ Rt - M)) <= 8 * n * EPS
        assert _isometry(L, Rt, direction) <= 1e-13 + 4 * n * EPS


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("Q", [5, 1])
def test_sector_of_zeros(pkg, ctx, Q, cplx, direction):
    """A charge sector without weight that is kept all the same, and a tensor of
    zeros: the factor is still an isometry."""
    A, charges, M, sectors = _charged(cplx, np.random.default_rng(41), DIMS,
                                      edit=lambda q, S: S * (0.0 if q == Q else 1.0))
    t = pkg.site2_from_dense(ctx, A, *charges)
    L, Rt, sv = _svd(pkg, ctx, t, 1, direction)
    _check_sectors(M, sectors, L, Rt, sv, direction)
    t = pkg.site2_from_dense(ctx, 0.0 * A, *charges)
    L, Rt, sv = _svd(pkg, ctx, t, 1, direction)
    assert np.all(sv == 0.0) and np.all(L @ Rt == 0.0)
    assert _isometry(L, Rt, direction) <= 1e-13


@pytest.mark.parametrize("limit", [-1, 41])
def test_sweep_limit_out_of_range(pkg, ctx, limit):
    with pytest.raises(Exception, match="sweep limit"):
        ctx.set_jacobi_sweeps(limit)
