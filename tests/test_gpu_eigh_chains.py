"""Inverse iteration in chunks of rows, and the scaling of the one-workgroup
tridiagonalisation, at orders around the chunks (16 rows, 64 threads) and on
matrices that try their ranges: extreme scales, graded entries, couplings that
vanish and the close pairs of Wilkinson's matrix.  By residual (20 n eps of the
norm, as for the eigensolver elsewhere) and orthogonality: vectors of eigenvalues
further apart than 1e-3 of the norm are not orthogonalised against each other, so
eps / 1e-3 is added to that bound."""
import numpy as np
import pytest

from qxmd_amd import pw
from qxmd_amd.system import diamond_si

pytestmark = pytest.mark.gpu

EPS = 2.220446049250313e-16


@pytest.fixture(scope="module")
def ctx():
    c = pw.PlaneWave(pw.GSphere(diamond_si(1).hcell), 330)
    yield c
    c.close()


def _matrix(kind, n, rng):
    a = rng.standard_normal((n, n))
    a = a + a.T
    if kind == "tiny":
        return a * 1e-120
    if kind == "huge":
        return a * 1e120
    if kind == "graded":
        g = 10.0 ** -np.linspace(0, 14, n)
        return a * np.sqrt(np.outer(g, g))
    if kind == "blocks":  # no coupling between blocks of five
        return a * (np.arange(n)[:, None] // 5 == np.arange(n)[None, :] // 5)
    if kind == "wilkinson":
        return np.diag(np.abs(np.arange(n) - (n - 1) / 2)) + np.diag(np.ones(n - 1), 1) + \
            np.diag(np.ones(n - 1), -1)
    return a


@pytest.mark.parametrize("kind", ["plain", "tiny", "huge", "graded", "blocks", "wilkinson"])
@pytest.mark.parametrize("n", [2, 7, 8, 9, 16, 17, 18, 33, 63, 64, 65, 129, 193, 330])
def test_eigensolver_chains(ctx, n, kind):
    print("order", n, kind, flush=True)
    a = _matrix(kind, n, np.random.default_rng(7 * n))
    w, v = ctx.rseigqr(a)
    scale = np.abs(a).sum(1).max()
    assert np.abs(w - np.linalg.eigvalsh(a)).max() < 20 * n * EPS * scale
    assert np.abs(a @ v - v * w).max() < 20 * n * EPS * scale
    assert np.abs(v.T @ v - np.eye(n)).max() < 20 * n * EPS + EPS / 1e-3
