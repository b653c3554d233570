"""H X on device buffers that share memory, and with more vectors than a grid's second dimension holds."""
import ctypes as C

import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu


def operator(c, o, v, P, seed, diagonal=True):
    rng = np.random.default_rng(seed)
    n = o + v
    M = rng.normal(scale=0.1, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    e = np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])
    H = np.diag(e)
    if not diagonal:
        m = rng.normal(scale=0.05, size=(n, n))
        H += 0.5 * (m + m.T)
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    op = px.BSE_OPERATOR(*c, rng.uniform(0.3, 1.0, P), t, H, precisions=("fp64", "bf16x3")).configure(
        px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1))
    return op, t, M, rng


# the result's first element behind the vectors' first, and the leading dimensions behind the size
@pytest.mark.parametrize("shift,dx,dy", [(0, 0, 0), (0, 3, 3), (0, 0, 5), (0, 5, 0), (1, 0, 0), (37, 2, 2), (-11, 0, 0),
                                         (-500, 0, 1)])
@pytest.mark.parametrize("o,v", [(4, 300), (30, 17)])
@pytest.mark.parametrize("diagonal", [True, False])
@pytest.mark.parametrize("prec", ["fp64", "bf16x3"])
def test_result_over_the_vectors(shift, dx, dy, o, v, diagonal, prec):
    k, P = 7, 21
    op, t, _, rng = operator((1, 2, 1, 0), o, v, P, o + v, diagonal)
    N = op.size
    ldx, ldy = N + dx, N + dy
    X = np.zeros((ldx, k), order="F")
    X[:N] = rng.normal(size=(N, k))
    want = op.matmul(np.asfortranarray(X[:N]), prec)
    x0, y0 = max(0, -shift), max(0, shift)
    size = max(x0 + ldx * k, y0 + ldy * k)
    host = np.zeros(size)
    host[x0:x0 + ldx * k] = X.ravel(order="F")
    buf = px.DeviceBuffer(t.ctx, size * 8)
    buf.upload(host)
    fn = px.lib().xtpgpu_bse_matmul_device
    ptr = lambda i: C.c_void_p(buf.ptr.value + 8 * i)  # noqa: E731
    px._check(fn(op.h, px._PREC[prec], ptr(x0), ldx, k, ptr(y0), ldy))
    got = buf.download((size,))[y0:y0 + ldy * k].reshape((ldy, k), order="F")[:N]
    assert np.array_equal(got, want)


def test_more_vectors_than_a_grid_dimension():
    """The exchange product of 70000 vectors, whose second half is summed from K splits."""
    P, k = 4096, 70000
    op, _, M, rng = operator((0, 2, 0, 0), 1, 2, P, 5)
    x = rng.normal(size=(2, k))
    A = M[0, 1:, :]
    want = 2.0 * A @ (A.T @ x)
    # two sums of 2 and 4096 products of either sign
    assert np.linalg.norm(op.matmul(x) - want) <= 1e-12 * np.linalg.norm(want)


def test_more_auxiliary_functions_than_a_grid_dimension():
    """The exchange part of the adjoint over 70000 auxiliary functions."""
    P = 70000
    op, _, M, rng = operator((1, 2, 0, 0), 1, 2, P, 6)
    x = rng.normal(size=(2, 1))
    m = M[0, 1:, :]  # (c, P)
    want = 4.0 * (m.T @ x)[:, :, None] * x[:, 0]  # (P, 1, c)
    got = px.bse_adjoint(op, x)[1][0]
    assert np.linalg.norm(got - want) <= 1e-13 * np.linalg.norm(want)
