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
