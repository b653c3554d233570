"""The operator's packed layouts and its diagonal at the edges of their kernels' rows, tiles and aux shares."""
import numpy as np
import pytest

from oracle import xtp_oracle as X
from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu

# sums of at most a few thousand products: |error| <= K 2^-53 relative to the sum of magnitudes
TOL = 1e-12


@pytest.mark.parametrize("o,v,P", [(1, 1, 1), (2, 8, 15), (3, 15, 16), (8, 17, 17), (9, 31, 33), (16, 32, 31),
                                   (17, 63, 64), (7, 64, 65), (33, 65, 9), (5, 129, 40), (65, 40, 12), (4, 12, 513)])
@pytest.mark.parametrize("c", [(1, 2, 1, 0), (1, 2, 0, 1), (1, 0, 1, 0), (0, 0, 0, 1), (1, 0, 0, 0)])
def test_layouts_and_diagonal(o, v, P, c):
    rng = np.random.default_rng(100 * o + v + P)
    lo, hi = 2, 3  # levels of the tensor below and above the operator's
    n = lo + o + v + hi
    M = rng.normal(scale=0.2, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    H = np.diag(rng.uniform(-1.0, 2.0, o + v))
    eps = rng.uniform(0.2, 1.0, P)
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    op = px.BSE_OPERATOR(*c, eps, t, H, precisions=("fp64", "bf16x3")).configure(
        px.BSEOperator_Options(lo + o - 1, 0, 0, lo, lo + o + v - 1))
    ref = X.bse_dense(*c, eps, M, H, lo + o - 1, 0, lo, lo + o + v - 1)
    assert np.abs(op.diagonal() - np.diag(ref)).max() <= TOL * np.abs(ref).max()
    x = rng.normal(size=(o * v, 2))
    y = ref @ x
    assert np.linalg.norm(op.matmul(x) - y) <= TOL * np.linalg.norm(y)
    # both operands of two products in 16 bits: 4 2^-17, times 2 for sums of either sign
    assert np.linalg.norm(op.matmul(x, "bf16x3") - y) <= 2 * 4 * 2.0**-17 * np.linalg.norm(y)
