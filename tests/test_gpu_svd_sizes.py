"""Truncated SVD of single sectors over the sizes its solver treats
differently: remainders of the 16-column panels, one and several register
tiles per wave, the tallest sectors of the register-resident kernels and the
ones above them, wide and tall sectors in both directions."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _matrix(kind, R, Cc, rng):
    K = min(R, Cc)
    if kind == "flat":
        M = rng.standard_normal((R, Cc))
    elif kind == "graded":      # both sides graded, as a two-site tensor is
        M = np.exp(-25.0 * np.arange(R) / R)[:, None] * rng.standard_normal((R, Cc)) * \
            np.exp(-10.0 * np.arange(Cc) / Cc)[None, :]
        M = M[rng.permutation(R)][:, rng.permutation(Cc)]
    elif kind == "equal":       # groups of equal columns and of zero rows
        M = np.repeat(rng.standard_normal((R, -(-Cc // 8))), 8, axis=1)[:, :Cc]
        M[rng.permutation(R)[:R // 5]] = 0.0
    else:                       # isometric: all singular values equal
        Q = np.linalg.qr(rng.standard_normal((max(R, Cc), K)))[0]
        M = Q if R >= Cc else Q.T
    return M / np.linalg.norm(M)


SHAPES = [(16, 20), (20, 17), (17, 40), (33, 32), (65, 65), (66, 150), (150, 67), (127, 129), (256, 255), (257, 300), (500, 513),
          (1024, 80), (70, 1025), (1030, 1027), (2048, 90), (90, 2048), (2049, 72)]


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("kind", ["flat", "graded", "equal", "isometric"])
@pytest.mark.parametrize("shape", SHAPES)
def test_svd_single_sector(pkg, ctx, shape, kind, direction):
    R, Cc = shape
    if max(shape) > 1000 and min(shape) > 1000 and kind != "graded":
        pytest.skip("one large square case is enough")
    M = _matrix(kind, R, Cc, np.random.default_rng(R * 7 + Cc))
    t = pkg.site2_from_dense(ctx, M.reshape(R, 1, 1, Cc))
    l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
    sv = np.zeros(4096)
    ctx.call("dmrj_svd_trunc2", t.h, 0, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
             pkg._lib.dptr(sv), 4096)
    L = pkg.DeviceTensor(ctx, l).to_dense()[0].reshape(R, -1)
    Rt = pkg.DeviceTensor(ctx, r).to_dense()[0].reshape(-1, Cc)
    n = max(R, Cc)
    want = np.linalg.svd(M, compute_uv=False)
    assert kk.value == min(R, Cc)
    # backward-stable factorisations and orthogonal updates: n eps |M| each
    assert np.max(np.abs(sv[:kk.value] - want)) <= 2 * n * EPS
    # (vectors of sigma <= 1e-10 sigma_max are replaced by an orthonormal
    # completion, which leaves their part of M out)
    zero = want[want <= 1e-10 * want[0]]
    assert np.max(np.abs(L @ Rt - M)) <= 8 * n * EPS + np.linalg.norm(zero)
    # columns are orthogonal to the pair tolerance (1e-14 or 4 eps sqrt(n)) on
    # top of the rounding of the back-transformation and the completion
    Q = L if direction > 0 else Rt.T
    assert np.max(np.abs(Q.T @ Q - np.eye(kk.value))) <= 1e-13 + 4 * n * EPS


@pytest.mark.parametrize("scale", [1e-150, 1e-60, 1e60, 1e120])
def test_svd_scaled(pkg, ctx, scale):
    """The tensor's norm enters as a power of two only."""
    M = _matrix("graded", 130, 97, np.random.default_rng(3))
    sv = []
    for f in (1.0, scale):
        t = pkg.site2_from_dense(ctx, (M * f).reshape(130, 1, 1, 97))
        l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
        s = np.zeros(128)
        ctx.call("dmrj_svd_trunc2", t.h, 0, 2, 0.0, 1, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
                 pkg._lib.dptr(s), 128)
        Q = pkg.DeviceTensor(ctx, l).to_dense()[0].reshape(130, -1)
        assert np.max(np.abs(Q.T @ Q - np.eye(97))) <= 1e-13 + 4 * 130 * EPS
        sv.append(s[:97])
    assert np.max(np.abs(sv[0] - sv[1])) <= 2 * 130 * EPS


def _complex_matrix(kind, R, Cc, rng):
    M = rng.standard_normal((R, Cc)) + 1j * rng.standard_normal((R, Cc))
    if kind == "graded":
        M = np.exp(-25.0 * np.arange(R) / R)[:, None] * M * np.exp(-10.0 * np.arange(Cc) / Cc)[None, :]
    return M / np.linalg.norm(M)


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("kind", ["flat", "graded"])
@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (16, 17), (33, 32), (70, 40), (130, 257), (300, 280), (600, 513),
                                   (1024, 40), (1030, 40)])
def test_complex_svd_single_sector(pkg, ctx, shape, kind, direction):
    """ComplexF64 sectors: same bounds; vectors of sigma <= 1e-10 sigma_max keep
    the extracted form (no completion), so their orthogonality is not checked."""
    R, Cc = shape
    M = _complex_matrix(kind, R, Cc, np.random.default_rng(R * 7 + Cc))
    t = pkg.site2_from_dense(ctx, M.reshape(R, 1, 1, Cc))
    l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
    sv = np.zeros(4096)
    ctx.call("dmrj_svd_trunc2", t.h, 0, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
             pkg._lib.dptr(sv), 4096)
    L = pkg.DeviceTensor(ctx, l).to_dense()[0].reshape(R, -1)
    Rt = pkg.DeviceTensor(ctx, r).to_dense()[0].reshape(-1, Cc)
    n = max(R, Cc)
    want = np.linalg.svd(M, compute_uv=False)
    assert kk.value == min(R, Cc)
    assert np.max(np.abs(sv[:kk.value] - want)) <= 2 * n * EPS
    assert np.max(np.abs(L @ Rt - M)) <= 8 * n * EPS
    big = want > 1e-10 * want[0]
    Q = (L if direction > 0 else Rt.conj().T)[:, big]
    assert np.max(np.abs(Q.conj().T @ Q - np.eye(big.sum()))) <= 1e-13 + 4 * n * EPS


@pytest.mark.parametrize("direction", [1, -1])
def test_complex_svd_sectors_of_different_sizes(pkg, ctx, direction):
    """Charge sectors of 3 to 67 rows in one call: every vector is finite and
    the product of the factors is the tensor (a batched Hermitian eigensolve
    of such sectors, padded to one size, has returned NaN vectors)."""
    rng = np.random.default_rng(11)
    dims = {-2: 12, 0: 40, 2: 27, 4: 3}
    q = np.array([[c] for c in sorted(dims) for _ in range(dims[c])], dtype=np.int32)
    m = len(q)
    qp = np.array([[1], [-1]], dtype=np.int32)
    A = rng.standard_normal((m, 2, 2, m)) + 1j * rng.standard_normal((m, 2, 2, m))
    ok = (q[:, None, None, None, 0] + qp[None, :, None, None, 0] + qp[None, None, :, None, 0] == q[None, None, None, :, 0])
    A = np.where(ok, A, 0.0)
    A /= np.linalg.norm(A)
    t = pkg.site2_from_dense(ctx, A, q, qp, qp, q, 1)
    l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
    sv = np.zeros(4096)
    ctx.call("dmrj_svd_trunc2", t.h, 0, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
             pkg._lib.dptr(sv), 4096)
    L = pkg.DeviceTensor(ctx, l).to_dense(1)[0]
    Rt = pkg.DeviceTensor(ctx, r).to_dense(1)[0]
    assert np.all(np.isfinite(L)) and np.all(np.isfinite(Rt))
    assert np.max(np.abs(np.tensordot(L, Rt, axes=(2, 0)) - A)) <= 8 * 2 * m * EPS


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("shape", [(210, 16), (16, 230), (40, 33), (33, 70), (130, 257), (280, 300)])
def test_complex_svd_rank_deficient(pkg, ctx, shape, direction):
    """Groups of equal columns and zero rows: the vectors of the vanishing
    singular values must not bring weight into the product of the factors."""
    R, Cc = shape
    rng = np.random.default_rng(R * 31 + Cc)
    M = np.exp(2j * np.pi * rng.random(R))[:, None] * _matrix("equal", R, Cc, rng)
    M = M * np.exp(2j * np.pi * rng.random(Cc))[None, :]
    n = max(R, Cc)
    want = np.linalg.svd(M, compute_uv=False)
    for scale in (1.0, 1e-150, 1e100):
        t = pkg.site2_from_dense(ctx, (M * scale).reshape(R, 1, 1, Cc))
        l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
        sv = np.zeros(512)
        ctx.call("dmrj_svd_trunc2", t.h, 0, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
                 pkg._lib.dptr(sv), 512)
        L = pkg.DeviceTensor(ctx, l).to_dense()[0].reshape(R, -1)
        Rt = pkg.DeviceTensor(ctx, r).to_dense()[0].reshape(-1, Cc)
        assert kk.value == min(R, Cc)
        assert np.max(np.abs(sv[:kk.value] * np.linalg.norm(want) - want)) <= 2 * n * EPS
        assert np.max(np.abs(L @ Rt * np.linalg.norm(want) - M)) <= 8 * n * EPS

def _factors(pkg, ctx, M, direction):
    R, Cc = M.shape
    t = pkg.site2_from_dense(ctx, M.reshape(R, 1, 1, Cc))
    l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
    sv = np.zeros(64)
    ctx.call("dmrj_svd_trunc2", t.h, 0, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
             pkg._lib.dptr(sv), 64)
    L = pkg.DeviceTensor(ctx, l).to_dense()[0].reshape(R, -1)
    Rt = pkg.DeviceTensor(ctx, r).to_dense()[0].reshape(-1, Cc)
    return L, Rt, sv[:kk.value]


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("kind", ["flat", "graded", "equal", "isometric"])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("shape", [(1, 1), (1, 7), (6, 1), (2, 2), (3, 2), (5, 16), (16, 16), (16, 15), (13, 8), (16, 33),
                                   (31, 7), (16, 200), (210, 16), (16, 440), (452, 16)])
def test_svd_small_sides(pkg, ctx, shape, cplx, kind, direction):
    """Sides up to 16: one launch of cyclic Jacobi while the sector fits into
    LDS.  Pairs are orthogonal to 4 eps, sums over the longer side add their
    rounding; the accumulated factor ends in a Newton-Schulz step."""
    R, Cc = shape
    rng = np.random.default_rng(R * 31 + Cc)
    M = _matrix(kind, R, Cc, rng)
    if cplx:  # unitary phases: the same singular values
        M = np.exp(2j * np.pi * rng.random(R))[:, None] * M * np.exp(2j * np.pi * rng.random(Cc))[None, :]
    n, K = max(R, Cc), min(R, Cc)
    want = np.linalg.svd(M, compute_uv=False)
    for scale in (1.0, 1e-150, 1e100):
        L, Rt, sv = _factors(pkg, ctx, M * scale, direction)
        assert len(sv) == K
        assert np.max(np.abs(sv - want / np.linalg.norm(want))) <= 2 * n * EPS
        zero = want[want <= 1e-10 * want[0]]
        assert np.max(np.abs(L @ Rt * np.linalg.norm(want) - M)) <= 8 * n * EPS + np.linalg.norm(zero)
        big = want > 1e-10 * want[0] if cplx else np.full(K, True)
        Q = (L if direction > 0 else Rt.conj().T)[:, big]
        assert np.max(np.abs(Q.conj().T @ Q - np.eye(big.sum()))) <= (8 + 2 * np.sqrt(n)) * EPS + 4 * K * EPS


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("shape", [(32, 40), (48, 64), (96, 160), (160, 96), (300, 280)])
def test_svd_large_rotations(pkg, ctx, shape, cplx, direction):
    """A step matrix: its panels hold columns of nearly equal norms and inner
    products, whose simultaneous rotations have a spectral norm above the range
    of the inner solve's Newton-Schulz steps; the solve has to notice the
    divergence (overflow to not-a-number included) and shorten them."""
    R, Cc = shape
    rng = np.random.default_rng(R + Cc)
    M = np.tril(np.ones((R, Cc))) + 1e-3 * rng.standard_normal((R, Cc))
    if cplx:
        M = np.exp(2j * np.pi * rng.random(R))[:, None] * M * np.exp(2j * np.pi * rng.random(Cc))[None, :]
    M = M / np.linalg.norm(M)
    n, K = max(R, Cc), min(R, Cc)
    t = pkg.site2_from_dense(ctx, M.reshape(R, 1, 1, Cc))
    l, r, te, kk = C.c_void_p(), C.c_void_p(), C.c_double(), C.c_int64()
    sv = np.zeros(512)
    ctx.call("dmrj_svd_trunc2", t.h, 0, 2, 0.0, direction, C.byref(l), C.byref(r), C.byref(te), C.byref(kk),
             pkg._lib.dptr(sv), 512)
    L = pkg.DeviceTensor(ctx, l).to_dense()[0].reshape(R, -1)
    Rt = pkg.DeviceTensor(ctx, r).to_dense()[0].reshape(-1, Cc)
    assert kk.value == K
    assert np.max(np.abs(sv[:K] - np.linalg.svd(M, compute_uv=False))) <= 2 * n * EPS
    assert np.max(np.abs(L @ Rt - M)) <= 8 * n * EPS
    Q = L if direction > 0 else Rt.conj().T
    assert np.max(np.abs(Q.conj().T @ Q - np.eye(K))) <= 1e-13 + 4 * n * EPS


@pytest.mark.parametrize("direction", [1, -1])
@pytest.mark.parametrize("shape", [(16, 12), (72, 40), (40, 2048), (2049, 20), (20, 2049)])
def test_backend5_routes(pkg, ctx, shape, direction):
    """Backend 5: the block Jacobi up to 2048 rows or columns (as the default),
    the Gram eigensolve, sigma^2 to n eps |M|^2, above."""
    R, Cc = shape
    M = _matrix("flat", R, Cc, np.random.default_rng(R + Cc))
    n, K = max(R, Cc), min(R, Cc)
    ctx.set_svd_backend(5)
    try:
        L, Rt, sv = _factors(pkg, ctx, M, direction)
    finally:
        ctx.set_svd_backend(0)
    want = np.linalg.svd(M, compute_uv=False)
    assert len(sv) == K
    if n > 2048:
        assert np.max(np.abs(sv ** 2 - want ** 2)) <= 4 * n * EPS
    else:
        assert np.max(np.abs(sv - want)) <= 2 * n * EPS
    assert np.max(np.abs(L @ Rt - M)) <= 8 * n * EPS
    Q = L if direction > 0 else Rt.T
    assert np.max(np.abs(Q.T @ Q - np.eye(K))) <= 1e-13 + 4 * n * EPS
