"""The first stage of BF16 products where the rule on its three forms changes sides: 192 and 193, 256 and 257 virtual
levels, 12288 tiles and more, and padded 256 x 256 tiles from 448 on. All forms give the same bits."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu

# rounding of both operands of two products to 8 (16) bits: 4 2^-9 (4 2^-17) relative to the norm when
# errors do not cancel, times 2 for the sums of products of either sign
TOL = {"bf16": 2 * 4 * 2.0**-9, "bf16x3": 2 * 4 * 2.0**-17}


@pytest.mark.parametrize("o,v,P,k", [(20, 192, 40, 13), (20, 193, 40, 13), (34, 256, 30, 9), (34, 257, 30, 9),
                                     (44, 440, 30, 31), (44, 448, 30, 31), (64, 250, 400, 30), (64, 250, 400, 32)])
@pytest.mark.parametrize("c", [(0, 0, 1, 0), (0, 0, 0, 1)])
def test_forms(o, v, P, k, c, monkeypatch):
    rng = np.random.default_rng(o * 1000 + v + P + k)
    n = o + v
    M = rng.normal(scale=0.05, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    e = np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    op = px.BSE_OPERATOR(*c, rng.uniform(0.3, 1.0, P), t, np.diag(e), precisions=("fp64", "bf16", "bf16x3")).configure(
        px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1))
    x = rng.normal(size=(o * v, k))
    ref = op.matmul(x, "fp64")
    for prec in ("bf16", "bf16x3"):
        monkeypatch.delenv("XTPGPU_BF16_KERNEL", raising=False)
        got = op.matmul(x, prec)
        assert np.linalg.norm(got - ref) <= TOL[prec] * np.linalg.norm(ref)
        monkeypatch.setenv("XTPGPU_BF16_KERNEL", "staged64")
        assert np.array_equal(op.matmul(x, prec), got)
