"""The direct-to-LDS BF16 kernels at the edges of their tiles and of the rules that choose them. They
accumulate every output in the order of the register-staged 128 x 128 tiles (XTPGPU_BF16_KERNEL=staged64),
so the two agree bit for bit."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu

# rounding of both operands of two products to 8 (16) bits: 4 2^-9 (4 2^-17) relative to the norm when
# errors do not cancel, times 2 for the sums of products of either sign
TOL = {"bf16": 2 * 4 * 2.0**-9, "bf16x3": 2 * 4 * 2.0**-17}


def operator(c, o, v, P, seed):
    rng = np.random.default_rng(seed)
    n = o + v
    M = rng.normal(scale=0.05, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    e = np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    return px.BSE_OPERATOR(*c, rng.uniform(0.3, 1.0, P), t, np.diag(e), precisions=("fp64", "bf16", "bf16x3")).configure(
        px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1)), rng


# (o, v, P, k): second-stage tiles of 32 and 256 rows at every width, first-stage products of up to three
# 256-column tiles with rows that do and do not end on a tile, and vectors that end inside a group of four
@pytest.mark.parametrize("o,v,P,k", [(1, 33, 9, 3), (16, 31, 40, 1), (17, 32, 33, 16), (32, 65, 20, 2), (33, 256, 24, 9),
                                     (64, 257, 24, 9), (65, 129, 40, 3), (112, 96, 12, 5), (113, 64, 16, 5),
                                     (128, 520, 70, 9), (129, 260, 33, 4), (30, 300, 600, 19), (31, 301, 600, 19),
                                     (100, 255, 257, 12), (8, 1030, 130, 31), (33, 390, 60, 31),
                                     (64, 388, 60, 12), (30, 400, 100, 17), (97, 360, 90, 17), (64, 380, 130, 17),
                                     (65, 380, 130, 15)])
@pytest.mark.parametrize("c", [(0, 0, 1, 0), (0, 0, 0, 1)])
@pytest.mark.parametrize("prec", ["bf16", "bf16x3"])
def test_first_and_second_stage(o, v, P, k, c, prec, monkeypatch):
    op, rng = operator(c, o, v, P, o * 1000 + v + P + k)
    x = rng.normal(size=(o * v, k))
    got = op.matmul(x, prec)
    ref = op.matmul(x, "fp64")
    assert np.linalg.norm(got - ref) <= TOL[prec] * np.linalg.norm(ref)
    monkeypatch.setenv("XTPGPU_BF16_KERNEL", "staged64")
    assert np.array_equal(op.matmul(x, prec), got)


@pytest.mark.parametrize("o,v,P,nw", [(3, 40, 256, 3), (7, 60, 300, 12), (5, 130, 513, 1), (9, 70, 1100, 4), (3, 11, 1535, 2), (3, 11, 1536, 2), (4, 16, 1601, 3), (2, 67, 1793, 1)])
def test_eps_lower_triangle(o, v, P, nw, monkeypatch):
    rng = np.random.default_rng(P + nw)
    M = rng.normal(scale=0.1, size=(o, o + v, P))
    e = np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])
    rpa = px.RPA(px.TCMatrix_gwbse().Initialize(P, 0, o - 1, 0, o + v - 1).set_tensor(M))
    rpa.configure(o - 1, 0, o + v - 1)
    rpa.setRPAInputEnergies(e)
    w = np.linspace(0.0, 3.0, nw)
    got = rpa.calculate_epsilon(px.EPS_IMAG, w, "bf16x3")
    ref = rpa.calculate_epsilon(px.EPS_IMAG, w)
    assert np.linalg.norm(got - ref) <= TOL["bf16x3"] * np.linalg.norm(ref)
    monkeypatch.setenv("XTPGPU_BF16_KERNEL", "staged64")
    assert np.array_equal(rpa.calculate_epsilon(px.EPS_IMAG, w, "bf16x3"), got)
