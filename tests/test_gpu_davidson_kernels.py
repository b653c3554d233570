"""The Davidson's device kernels at the edges of their column groups: correction blocks of 2 to 40 columns (the
device Gram-Schmidt takes 32, the combinations groups of 8, 16 and 32), short and ragged vectors, and
a block of corrections that is linearly dependent."""
import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu

RES = 1e-9  # residual norm at convergence: an eigenvalue is off by no more


class Dense(px.MatrixFreeOperator):
    def __init__(self, mat):
        self.mat = mat
        self.set_size(mat.shape[0])

    def matmul(self, X):
        return self.mat @ X

    def diagonal(self):
        return np.diag(self.mat).copy()


def solver(update):
    ds = px.DavidsonSolver()
    ds.set_tolerance(RES)
    ds.set_size_update(update)
    ds.set_iter_max(200)
    return ds


@pytest.mark.parametrize("n,roots,update", [(65, 1, "max"), (127, 2, "min"), (128, 4, "max"), (129, 9, "min"), (191, 8, "max"),
                                            (257, 11, "safe"), (300, 16, "max"), (321, 17, "min"), (383, 33, "min"),
                                            (500, 20, "max"), (1000, 12, "safe")])
@pytest.mark.parametrize("gs", ["block", "column"])
def test_lowest_roots(n, roots, update, gs, monkeypatch):
    monkeypatch.setenv("XTPGPU_GS", gs)
    rng = np.random.default_rng(n + roots)
    m = rng.uniform(-1.0, 1.0, size=(n, n)) * 0.02
    A = 0.5 * (m + m.T)
    A[np.diag_indices(n)] = 1.0 + 0.5 * np.arange(n)
    w, x = solver(update).solve(Dense(A), roots)[:2]
    ref = np.linalg.eigvalsh(A)[:roots]
    assert np.abs(np.asarray(w) - ref).max() <= RES
    x = np.asarray(x)
    assert np.abs(x.T @ x - np.eye(roots)).max() <= 1e-10  # normalised Ritz vectors of an orthonormal basis


def test_dependent_corrections():
    """Every residual of diag + rank one lies along one vector, and equal diagonal entries make the corrections of
    different roots parallel: the block form finds a failing pivot and goes on as the column form does."""
    n = 200
    d = np.repeat(np.arange(1.0, 21.0), 10)
    u = np.random.default_rng(0).normal(size=n) * 0.05
    A = np.diag(d) + np.outer(u, u)
    out = []
    for gs in ("block", "column"):
        with pytest.MonkeyPatch.context() as mp:
            mp.setenv("XTPGPU_GS", gs)
            try:
                out.append(np.asarray(solver("max").solve(Dense(A), 6)[0]))
            except px.XtpGpuError as e:
                out.append(str(e))
    if isinstance(out[1], str):
        assert out[0] == out[1]
    else:
        assert np.abs(out[0] - out[1]).max() <= 1e-6
