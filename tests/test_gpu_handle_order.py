"""Handles that outlive their context, as an interpreter's exit leaves them: destroying them touches nothing of it."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("o,v,P", [(3, 7, 9), (24, 160, 200)])  # small buffers, and blocks that are kept
def test_context_ends_first(o, v, P, order):
    rng = np.random.default_rng(o)
    n = o + v
    M = rng.normal(scale=0.1, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    e = np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])
    ctx = px.Context()
    t = px.TCMatrix_gwbse(ctx).Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    op = px.BSE_OPERATOR(1, 2, 1, 0, rng.uniform(0.3, 1.0, P), t, np.diag(e)).configure(
        px.BSEOperator_Options(o - 1, 0, 0, 0, n - 1))
    rpa = px.RPA(t)
    rpa.configure(o - 1, 0, n - 1)
    s = px.Sigma_PPM(t, rpa).configure(o - 1, 0, o, 0, n - 1)
    s.ppm_weight, s.ppm_freq = rng.uniform(0, 0.5, P), rng.uniform(0.5, 2.0, P)
    s.set_rpa_energies(e)
    rpa.setRPAInputEnergies(e)
    b = px.EpsBatch([rpa], [0.0, 0.5])
    b.run()
    op.matmul(rng.normal(size=(op.size, 2)))
    s.diag_batch(np.array([0]), np.array([0.1]))
    ctx.close()
    for h in ((op, t, s, b), (b, s, t, op))[order]:
        h.close()
    # another context takes over memory that they left
    t2 = px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M)
    assert np.array_equal(t2.get_tensor(), M)
