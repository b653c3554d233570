"""The second stage of BF16 products where the rule on its three forms changes sides: one round of 256 workgroups and
the next, 64 and 65 columns, rows that just do and do not fill a tile. All forms give the same bits."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu

# rounding of both operands of two products to 8 (16) bits: 4 2^-9 (4 2^-17) relative to the norm when
# errors do not cancel, times 2 for the sums of products of either sign
TOL = {"bf16": 2 * 4 * 2.0**-9, "bf16x3": 2 * 4 * 2.0**-17}


def check(o, v, P, k, c, monkeypatch):
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


@pytest.mark.parametrize("o,v,P", [(20, 260, 90), (32, 129, 70), (33, 128, 64), (64, 257, 66), (65, 256, 64), (102, 303, 41),
                                   (128, 130, 33)])
@pytest.mark.parametrize("k", [3, 16, 32, 43, 65])
@pytest.mark.parametrize("c", [(0, 0, 1, 0), (0, 0, 0, 1)])
def test_forms(o, v, P, k, c, monkeypatch):
    check(o, v, P, k, c, monkeypatch)


@pytest.mark.parametrize("o,v,P,k", [(77, 54, 110, 45), (77, 54, 110, 90), (66, 33, 130, 45), (128, 90, 70, 33), (128, 91, 70, 64),
                                     (128, 94, 70, 45), (128, 211, 70, 32), (128, 213, 70, 33), (16, 7, 600, 64), (64, 65, 140, 90), (96, 130, 33, 70),
                                     (97, 130, 33, 70)])
@pytest.mark.parametrize("c", [(0, 0, 1, 0), (0, 0, 0, 1)])
def test_few_rows(o, v, P, k, c, monkeypatch):
    check(o, v, P, k, c, monkeypatch)
