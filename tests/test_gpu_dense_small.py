"""The one-workgroup Cholesky + inverse and tridiagonalisation at the orders
where their register blocks (64 rows, 16 columns) end, against numpy, and the
pivot rule (above 1e-30, the same at every order) on nearly dependent and on
equal bands.  Bounds: L^-1 L = I to n cond eps; eigenvalues and residuals to
20 n eps of the norm, as for the cooperative kernels."""
import numpy as np
import pytest

from qxmd_amd import pw
from qxmd_amd.system import diamond_si

pytestmark = pytest.mark.gpu

ORDERS = [1, 2, 3, 15, 16, 17, 63, 64, 65, 100, 128, 129, 176, 191, 192, 193]
EPS = 2.220446049250313e-16


@pytest.fixture(scope="module")
def ctx():
    c = pw.PlaneWave(pw.GSphere(diamond_si(1).hcell), 200)
    yield c
    c.close()


@pytest.mark.parametrize("n", ORDERS)
def test_cholesky_inverse(ctx, n):
    print("order", n, flush=True)
    rng = np.random.default_rng(n)
    b = rng.standard_normal((n, 2 * n + 3))
    s = b @ b.T / b.shape[1]
    x, ok = ctx.icholesky(s)
    assert ok
    low = np.linalg.cholesky(s)
    assert np.abs(x @ low - np.eye(n)).max() < 20 * n * EPS * np.linalg.cond(low)
    assert not np.triu(x, 1).any()
    if 2 < n <= 192:  # two equal rows: the second pivot is zero in one workgroup
        q = n // 2
        s[n - 1], s[:, n - 1], s[n - 1, n - 1] = s[q], s[:, q], s[q, q]
        assert not ctx.icholesky(s)[1]
    s[0, 0] = -1.0
    assert not ctx.icholesky(s)[1]


@pytest.mark.parametrize("n", [2, 3, 16, 17, 64, 65, 128, 129, 192, 193, 200])
def test_pivot_rule(ctx, n):
    """Two rows that differ by one pivot p: accepted down to 1e-30 at every order,
    whatever the diagonal.  Every value is a power of two or a sum that FP64
    holds, so L^-1 is exact."""
    print("order", n, flush=True)
    q, r = (n - 1) // 2, n - 1
    for e in (-40, -50, -52):
        s, ref = np.eye(n), np.eye(n)
        s[q, r] = s[r, q] = 1.0
        s[r, r] = 1.0 + 2.0 ** e
        ref[r, r], ref[r, q] = 2.0 ** (-e / 2), -(2.0 ** (-e / 2))
        x, ok = ctx.icholesky(s)
        assert ok, e
        assert np.abs(x - ref).max() <= 4 * EPS * ref.max()
    for d in (1.0, 1.0 - EPS):  # pivots 0 and -eps
        s[r, r] = d
        assert not ctx.icholesky(s)[1]


@pytest.mark.parametrize("n", ORDERS[2:])
@pytest.mark.parametrize("kind", ["random", "clustered", "diagonal"])
def test_eigensolver(ctx, n, kind):
    print("order", n, kind, flush=True)
    rng = np.random.default_rng(100 + n)
    a = rng.standard_normal((n, n))
    a = a + a.T
    if kind == "clustered":
        q, _ = np.linalg.qr(a)
        a = (q * np.repeat(np.arange(1, n + 1), 3)[:n]) @ q.T
        a = 0.5 * (a + a.T)
    if kind == "diagonal":
        a = np.diag(np.diag(a))
    w, v = ctx.rseigqr(a)
    scale = max(np.abs(a).sum(1).max(), 1.0)
    assert np.abs(w - np.linalg.eigvalsh(a)).max() < 20 * n * EPS * scale
    assert np.abs(a @ v - v * w).max() < 20 * n * EPS * scale
    assert np.abs(v.T @ v - np.eye(n)).max() < 20 * n * EPS + 1e-14
