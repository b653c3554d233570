"""The full-Hqp product H_c^T X - X H_v on the tiles that its width and the number of vectors choose: 32 and 33, 64 and 65
occupied levels, on few workgroups and on more than 256 of them."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o", [1, 31, 32, 33, 48, 64, 65])
@pytest.mark.parametrize("v,k", [(10, 1), (130, 3), (450, 1), (258, 86)])
def test_full_hqp(o, v, k):
    rng = np.random.default_rng(1000 * o + v + k)
    n = o + v
    m = rng.normal(size=(n, n))
    H = 0.5 * (m + m.T)
    t = px.TCMatrix_gwbse().Initialize(1, 0, n - 1, 0, n - 1).set_tensor(np.zeros((n, n, 1)))
    op = px.BSE_OPERATOR(1, 0, 0, 0, np.ones(1), t, H).configure(px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1))
    x = rng.normal(size=(o * v, k))
    X = x.reshape(o, v, k)
    ref = np.einsum("cd,vdk->vck", H[o:, o:], X) - np.einsum("uv,uck->vck", H[:o, :o], X)
    # sums of n products, relative to the sum of their magnitudes
    mag = np.einsum("cd,vdk->vck", np.abs(H[o:, o:]), np.abs(X)) + np.einsum("uv,uck->vck", np.abs(H[:o, :o]), np.abs(X))
    assert (np.abs(op.matmul(x).reshape(o, v, k) - ref) <= 2 * (n + 4) * 2.0**-53 * mag).all()
