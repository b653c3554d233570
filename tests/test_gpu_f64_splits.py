"""FP64 second-stage products of 128 to 257 output tiles, whose K splits the rounds of workgroups choose (3 at 128, 7 at
130, 3 at 150, 4 at 180, 8 at 220, 2 at 240, up to four from 257 on), and with a K too short for more."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [64, 65, 75, 90, 110, 120, 128, 129])  # two tiles of rows each
@pytest.mark.parametrize("o,v,P", [(33, 131, 206), (16, 129, 64)])  # K = 8240 and 1024
def test_hd_splits(o, v, P, k):
    rng = np.random.default_rng(1000 * o + k)
    n = o + v
    M = rng.normal(scale=0.1, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    eps = rng.uniform(0.3, 1.0, P)
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    op = px.BSE_OPERATOR(0, 0, 1, 0, eps, t, np.zeros((n, n))).configure(px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1))
    x = rng.normal(size=(o * v, k))
    X = x.reshape(o, v * k)
    turn = lambda z: z.reshape(o, v, k).transpose(1, 0, 2).reshape(v, o * k)  # noqa: E731
    ref, mag = np.zeros((v, o * k)), np.zeros((v, o * k))
    for p in range(P):
        a, b = M[:o, :o, p], np.ascontiguousarray(M[o:, o:, p])
        ref -= eps[p] * (b @ turn(a @ X))
        mag += eps[p] * (np.abs(b) @ turn(np.abs(a) @ np.abs(X)))
    # sums of v, and of P o, products, relative to the sum of their magnitudes
    assert (np.abs(turn(op.matmul(x)) - ref) <= 2 * (v + P * o + 8) * 2.0**-53 * mag).all()
