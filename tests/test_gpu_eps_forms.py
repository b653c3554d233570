"""Dielectric builds with a long K: the sums' rounding."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu


def rpa_of(M, e, o):
    n = e.size
    rpa = px.RPA(px.TCMatrix_gwbse().Initialize(M.shape[2], 0, o - 1, 0, n - 1).set_tensor(M))
    rpa.configure(o - 1, 0, n - 1)
    rpa.setRPAInputEnergies(e)
    return rpa


def test_fp64_sums_in_pieces():
    """98304 equal products: the roundings of a sum are equal too, over each binade, and add up. Sums of at most
    4096 products each and their 24 results: |error| <= (4096 + 24 + 8) 2^-53 relative (8: energies, weights, the unit
    matrix). One chain over all of K comes to 6.6e-13 at the worst of these frequencies."""
    o, v, P, nw, m = 96, 1024, 256, 100, 0.1
    e = np.concatenate([np.full(o, -0.5), np.full(v, 0.5)])
    w = np.linspace(0.0, 3.0, nw)
    got = rpa_of(np.full((o, o + v, P), m), e, o).calculate_epsilon(px.EPS_IMAG, w)
    x = np.longdouble(m) ** 2 * (o * v) * 4 / (1 + w.astype(np.longdouble) ** 2)
    for i in range(nw):
        assert np.abs(got[:, :, i] / (x[i] + np.eye(P)) - 1).max() <= (4096 + 24 + 8) * 2.0**-53
