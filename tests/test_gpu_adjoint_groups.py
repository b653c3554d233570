"""The weighted adjoint where its roots do not fit one group: more than 1 GiB of the Hd2 intermediate, and more than 64
roots without an Hd2 part; vectors with a leading dimension beyond their length."""
import ctypes as C

import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu

TOL = 1e-12  # sums of at most ~5000 products


# 64 x 8, 1024 aux functions, X and Y: 67 MB a root, 16 roots a group
@pytest.mark.parametrize("o,v,P,r,pad", [(64, 8, 1024, 16, 0), (64, 8, 1024, 19, 3), (5, 7, 33, 4, 5)])
@pytest.mark.parametrize("a,b", [((1, 2, 1, 0), (0, 2, 0, 1)), ((0, 1, 0, 1), (0, 1, 0, 1))])
def test_hd2_groups(o, v, P, r, pad, a, b):
    check(o, v, P, r, pad, a, b)


@pytest.mark.parametrize("r,pad", [(64, 0), (65, 0), (130, 2)])
def test_exchange_groups(r, pad):
    check(5, 7, 33, r, pad, (1, 2, 1, 0), (0, 2, 0, 0))


def check(o, v, P, r, pad, a, b):
    rng = np.random.default_rng(o + v + P + r)
    n, N = o + v, o * v
    M = rng.normal(scale=0.3, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    e = np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])
    eps = rng.uniform(-0.2, 1.0, P)
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    opt = px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1)
    A, B = (px.BSE_OPERATOR(*c, eps, t, np.diag(e)).configure(opt) for c in (a, b))
    X, Y = (np.asfortranarray(rng.normal(size=(N + pad, r))) for _ in range(2))
    w = rng.normal(size=r)
    w[r // 2] = 0.0
    de, buf = np.zeros(n), px.DeviceBuffer(t.ctx, P * N * 8)
    px._check(px.lib().xtpgpu_bse_adjoint_weighted_device(A.h, B.h, r, px._dptr(X), px._dptr(Y), N + pad, px._dptr(w),
                                                          px._dptr(de), C.c_void_p(buf.ptr.value)))
    got = buf.download((P, o, v), order="C")
    m = np.ascontiguousarray(M[:o, o:, :].transpose(2, 0, 1))
    ref, dref = np.zeros((P, o, v)), np.zeros(n)
    for i in range(r):
        x, y = (q[:N, i].reshape(o, v) for q in (X, Y))
        sx, sy = (np.tensordot(m, q, 2)[:, None, None] for q in (x, y))
        zx, zy = (q @ m.transpose(0, 2, 1) for q in (x, y))  # X m^T, Y m^T
        g = 2 * a[1] * (x * sx + y * sy) + 2 * b[1] * (x * sy + y * sx)
        g -= 2 * eps[:, None, None] * (b[3] * (zy @ x + zx @ y) + a[3] * (zx @ x + zy @ y))
        ref += w[i] * g
        dref[:o] -= w[i] * a[0] * (x * x + y * y).sum(1)
        dref[o:] += w[i] * a[0] * (x * x + y * y).sum(0)
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)
    assert np.linalg.norm(de - dref) <= TOL * np.linalg.norm(dref)
