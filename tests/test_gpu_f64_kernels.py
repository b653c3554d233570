"""The direct-to-LDS FP64 kernels at the edges of their tiles and of the rules that choose them: the
even deal of the dielectric builds (64 x 64 and 128 x 128 tiles, flocks of frequencies, shared and
whole units) and the split second-stage and exchange products (every width of the narrow tile)."""
import numpy as np
import pytest

from oracle import xtp_oracle as X
from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu

# sums of at most ~4000 products: |error| <= K 2^-53 relative to the sum of magnitudes
TOL = 1e-12


def tensor(rng, o, v, P, scale=0.05):
    n = o + v
    M = rng.normal(scale=scale, size=(n, n, P))
    return 0.5 * (M + M.transpose(1, 0, 2))


def energies(rng, o, v):
    return np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])


@pytest.mark.parametrize("o,v,P,nw", [(1, 1, 1, 1), (2, 3, 16, 4), (3, 21, 63, 1), (3, 22, 64, 5), (5, 13, 65, 12),
                                      (7, 31, 130, 3), (11, 47, 200, 8), (2, 5, 1535, 2), (2, 5, 1536, 4),
                                      (3, 7, 1601, 1)])
def test_eps_even_deal(o, v, P, nw):
    rng = np.random.default_rng(o * 1000 + P + nw)
    M = rng.normal(scale=0.1, size=(o, o + v, P))
    e = energies(rng, o, v)
    t = px.TCMatrix_gwbse().Initialize(P, 0, o - 1, 0, o + v - 1).set_tensor(M)
    rpa = px.RPA(t)
    rpa.configure(o - 1, 0, o + v - 1)
    rpa.setRPAInputEnergies(e)
    w = np.linspace(0.0, 3.0, nw)
    out = rpa.calculate_epsilon(px.EPS_IMAG, w)
    A = M[:, o:, :].reshape(o * v, P)
    D = (e[None, o:] - e[:o, None]).reshape(-1)
    for i in range(nw):
        ref = np.eye(P) + A.T @ ((4.0 * D / (D * D + w[i] * w[i]))[:, None] * A)
        assert np.linalg.norm(out[:, :, i] - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("o,v,P,k", [(1, 1, 1, 1), (1, 9, 40, 3), (3, 17, 33, 16), (15, 5, 50, 2), (16, 20, 24, 17),
                                     (17, 40, 31, 1), (33, 12, 20, 4), (49, 7, 12, 2), (65, 9, 11, 2), (81, 6, 9, 1),
                                     (97, 5, 8, 1), (113, 4, 7, 2), (129, 3, 6, 1), (9, 129, 64, 5)])
@pytest.mark.parametrize("c", [(1, 2, 1, 0), (0, 2, 0, 1)])
def test_products_narrow_tiles(o, v, P, k, c):
    rng = np.random.default_rng(o * 100 + v + P + k)
    M, e = tensor(rng, o, v, P), energies(rng, o, v)
    eps, H = rng.uniform(0.3, 1.0, P), np.diag(e)
    n = o + v
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    op = px.BSE_OPERATOR(*c, eps, t, H).configure(px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1))
    x = rng.normal(size=(o * v, k))
    ref = X.bse_dense(*c, eps, M, H, o - 1, 0, 0, n - 1) @ x
    assert np.linalg.norm(op.matmul(x) - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("o,v,P,r", [(1, 2, 3, 1), (3, 7, 9, 2), (5, 16, 20, 3), (9, 33, 140, 1), (17, 20, 15, 4)])
@pytest.mark.parametrize("a,b,with_y", [((1, 2, 1, 0), (0, 2, 0, 1), True), ((1, 2, 1, 0), None, False),
                                        ((1, 0, 1, 0), (0, 0, 0, 1), True), ((0, 1, 0, 1), (0, 1, 0, 1), True),
                                        ((0, 0, 0, 1), None, False), ((1, 2, 1, 0), (0, 2, 0, 1), False)])
def test_weighted_adjoint_forms(o, v, P, r, a, b, with_y):
    """Every combination of exchange and Hd2 parts, with and without Y, against the formula written out."""
    import ctypes as C
    rng = np.random.default_rng(o + 10 * v + P + r)
    M, e, n = tensor(rng, o, v, P, 0.3), energies(rng, o, v), o + v
    eps = rng.uniform(-0.2, 1.0, P)
    eps[0] = 0.0
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    opt = px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1)
    A = px.BSE_OPERATOR(*a, eps, t, np.diag(e)).configure(opt)
    B = px.BSE_OPERATOR(*b, eps, t, np.diag(e)).configure(opt) if b else None
    Xv = np.asfortranarray(rng.normal(size=(o * v, r)))
    Yv = np.asfortranarray(rng.normal(size=(o * v, r))) if with_y else None
    w = rng.normal(size=r)
    w[0] = 0.0 if r > 2 else w[0]
    de, buf = np.zeros(n), px.DeviceBuffer(t.ctx, P * o * v * 8)
    px._check(px.lib().xtpgpu_bse_adjoint_weighted_device(
        A.h, B.h if B else None, r, px._dptr(Xv), px._dptr(Yv) if with_y else None, o * v, px._dptr(w), px._dptr(de),
        C.c_void_p(buf.ptr.value)))
    got = buf.download((P, o, v), order="C")
    m = M[:o, o:, :].transpose(2, 0, 1)
    ref, dref = np.zeros((P, o, v)), np.zeros(n)
    cxb, c2b = (b[1], b[3]) if b else (0, 0)
    for i in range(r):
        x = Xv[:, i].reshape(o, v)
        y = Yv[:, i].reshape(o, v) if with_y else np.zeros((o, v))
        sx, sy = (np.einsum("pvc,vc->p", m, q)[:, None, None] for q in (x, y))
        g = 2 * a[1] * (x * sx + y * sy) + 2 * cxb * (x * sy + y * sx)
        lmr = lambda p, q: np.einsum("vc,puc,ud->pvd", p, m, q)  # noqa: E731
        g = g - 2 * eps[:, None, None] * (c2b * (lmr(y, x) + lmr(x, y)) + a[3] * (lmr(x, x) + lmr(y, y)))
        ref += w[i] * g
        dref[:o] -= w[i] * a[0] * (x * x + y * y).sum(1)
        dref[o:] += w[i] * a[0] * (x * x + y * y).sum(0)
    assert np.linalg.norm(got - ref) <= TOL * max(np.linalg.norm(ref), 1e-300)
    assert np.linalg.norm(de - dref) <= TOL * max(np.linalg.norm(dref), 1e-300)


@pytest.mark.parametrize("o,v,P,levels,per", [(1, 1, 1, 1, 1), (2, 61, 31, 3, 2), (2, 62, 32, 2, 7), (3, 62, 33, 4, 8),
                                              (5, 123, 64, 2, 9), (5, 130, 40, 1, 17), (7, 240, 65, 6, 3),
                                              (9, 300, 20, 5, 5)])
def test_sigma_ppm_row_widths(o, v, P, levels, per):
    """Row lengths around the 64, 128 and 256-element steps, group sizes 1..8 and beyond, skipped weights."""
    rng = np.random.default_rng(o + v + P)
    M, e, n = tensor(rng, o, v, P), energies(rng, o, v), o + v
    t = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    rpa = px.RPA(t)
    rpa.configure(o - 1, 0, n - 1)
    q0 = max(0, o - levels // 2)
    s = px.Sigma_PPM(t, rpa).configure(o - 1, q0, q0 + levels - 1, 0, n - 1)
    s.ppm_weight, s.ppm_freq = rng.uniform(0, 0.5, P), rng.uniform(0.5, 2.0, P)
    s.ppm_weight[rng.random(P) < 0.2] = 0.0
    s.set_rpa_energies(e)
    lv = rng.permutation(np.repeat(np.arange(levels), per))
    om = rng.uniform(-2, 2, lv.size)
    sig, dsig = s.diag_batch(lv, om)
    f = s.ppm_freq[:, None]
    sh = np.where(np.arange(n)[None, :] < o, f, -f) - e[None, :]
    for i in range(lv.size):
        m2 = (0.5 * s.ppm_weight * s.ppm_freq)[:, None] * M[q0 + lv[i]].T ** 2
        tt = om[i] + sh
        den = tt * tt + 1e-6
        # each sum relative to the sum of its terms' magnitudes
        for got, terms in ((sig[i], m2 * tt / den), (dsig[i], m2 * (1e-6 - tt * tt) / (den * den))):
            assert abs(got - terms.sum()) <= TOL * max(np.abs(terms).sum(), 1e-300)
