"""The Krylov iteration (algs/time.jl:182-202) and the two-vector Lanczos step
(algs/DMRG.jl:57-90) at the lengths where their kernels change.  Krylov: one work-group up to 4096 stored elements, above that several, whose
pieces hold 1024 elements, up to 512 work-groups; and over the Krylov
dimensions the coefficient kernel takes (1..64).

Environments of canonical chains, so that |H_eff| <= 3 N / 4 and every step of
the iteration is accurate to a few rounding errors: output and Ritz value to
1e-12 relative (r <= 64 steps of about 10 eps each, times pf |H| <= 4).
"""
import ctypes as C

import numpy as np
import pytest

from oracle import dmrg as od
from oracle import tdvp as ot

pytestmark = pytest.mark.gpu


def isometry(rng, rows, cols, cplx):
    a = rng.standard_normal((rows, cols))
    if cplx:
        a = a + 1j * rng.standard_normal((rows, cols))
    return np.linalg.qr(a)[0]


def chain(rng, dl, dr, cplx):
    left, d = [], 1
    while d < dl:
        n = min(2 * d, dl)
        left.append(isometry(rng, 2 * d, n, cplx).reshape(d, 2, n))
        d = n
    right, d = [], 1
    while d < dr:
        n = min(2 * d, dr)
        right.insert(0, np.ascontiguousarray(isometry(rng, 2 * d, n, cplx).T).reshape(n, 2, d))
        d = n
    mid = [rng.standard_normal((dl, 2, 3)), rng.standard_normal((3, 2, dr))]
    if cplx:
        mid = [m + 1j * rng.standard_normal(m.shape) for m in mid]
    return left, mid, right


def environments(pkg, ctx, A, k, mpo):
    """Device and oracle environments around the two sites k, k + 1 (0-based)."""
    N = len(A)
    gL, oL = pkg.network.makeBoundary(ctx, True), np.ones((1, 1, 1))
    for i in range(k):
        gL = pkg.Lupdate(gL, pkg.site_from_dense(ctx, A[i]), mpo, i + 1)
        oL = od.Lupdate(oL, A[i], mpo.H[i])
    gR, oR = pkg.network.makeBoundary(ctx, False), np.ones((1, 1, 1))
    for i in range(N - 1, k + 1, -1):
        gR = pkg.Rupdate(gR, pkg.site_from_dense(ctx, A[i]), mpo, i + 1)
        oR = od.Rupdate(oR, A[i], mpo.H[i])
    return gL, oL, gR, oR


@pytest.mark.parametrize("dl,dr,cplx,r,pf", [
    (1, 2, False, 3, -0.25), (2, 2, False, 1, -0.25), (8, 8, False, 64, -0.25), (5, 9, False, 17, -0.3j),
    (31, 33, False, 12, -0.25), (32, 32, False, 12, -0.25), (32, 33, False, 12, -0.25), (29, 71, False, 5, -0.3j),
    (15, 34, True, 12, -0.1j), (16, 33, True, 12, -0.1j), (33, 64, True, 2, -0.1 - 0.2j), (4, 4, True, 33, -0.2j),
    (128, 130, False, 3, -0.25), (367, 366, False, 3, -0.25), (270, 250, True, 4, -0.2j),
])
def test_krylov_sizes(pkg, ctx, dl, dr, cplx, r, pf):
    rng = np.random.default_rng(dl * 1000 + dr)
    left, mid, right = chain(rng, dl, dr, cplx)
    A = left + mid + right
    k = len(left)
    mpo = pkg.makeMPO(pkg.heisenbergMPO(), 2, len(A))
    gL, oL, gR, oR = environments(pkg, ctx, A, k, mpo)
    h = C.c_void_p()
    dev = [pkg.site_from_dense(ctx, m) for m in mid]
    ctx.call("dmrj_theta2", dev[0].h, dev[1].h, C.byref(h))
    th = pkg.DeviceTensor(ctx, h)
    oth = np.tensordot(mid[0], mid[1], axes=(2, 0))
    out, e = pkg.krylovTimeEvol2(gL, gR, th, mpo, k + 1, r, pf)
    want, we = ot.krylov_expm(lambda t: od.heff2(oL, oR, t, mpo.H[k], mpo.H[k + 1]), oth, r, pf)
    got = out.to_dense()[0]
    err = np.max(np.abs(got - want)) / np.max(np.abs(want))
    print("n", oth.size, "r", r, "err %.1e" % err, "energy %.1e" % abs(e - we), flush=True)
    assert err <= 1e-12
    assert abs(e - we) <= 1e-12 * max(1.0, abs(we))


@pytest.mark.parametrize("dl,dr", [(1, 1), (2, 3), (15, 17), (31, 33), (32, 32), (32, 33), (63, 65), (64, 64), (64, 65),
                                   (130, 129), (367, 366)])
def test_lanczos_sizes(pkg, ctx, dl, dr):
    """The two-vector Lanczos step where its vector kernels change: 4096 and
    16384 elements in one work-group, above that several."""
    rng = np.random.default_rng(dl * 1000 + dr)
    left, mid, right = chain(rng, dl, dr, False)
    A = left + mid + right
    k = len(left)
    mpo = pkg.makeMPO(pkg.heisenbergMPO(), 2, len(A))
    gL, oL, gR, oR = environments(pkg, ctx, A, k, mpo)
    dev = [pkg.site_from_dense(ctx, m) for m in mid]
    h, e = C.c_void_p(), C.c_double()
    ctx.call("dmrj_lanczos2", gL.h, gR.h, dev[0].h, dev[1].h, mpo.device(ctx, k + 1), mpo.device(ctx, k + 2), 0,
             C.byref(h), C.byref(e))
    got = pkg.DeviceTensor(ctx, h).to_dense()[0]
    want_e, want = od.simplelanczos(oL, oR, mid[0], mid[1], mpo.H[k], mpo.H[k + 1])
    err = min(np.max(np.abs(got - want)), np.max(np.abs(got + want))) / np.max(np.abs(want))
    print("n", got.size, "energy %.1e" % abs(e.value - want_e), "state %.1e" % err, flush=True)
    assert abs(e.value - want_e) <= 1e-12 * max(1.0, abs(want_e))
    assert err <= 1e-12
