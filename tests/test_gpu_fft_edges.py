"""The two-step pencil FFTs on every edge they cover, as x, y and z edge:
(T + V)|psi> and the density of three bands against numpy's FFT.  FP64 bounds
as for the other local-part tests (1e-12 of the largest value); FP32 lines
accumulate about sqrt(6 log2 n) roundings of 6e-8 per transform pair, 3e-6 is
the bound of the mixed form."""
import numpy as np
import pytest

from qxmd_amd import pw

pytestmark = pytest.mark.gpu

EDGES = [16, 18, 20, 21, 24, 25, 27, 28, 30, 32, 35, 36, 40, 42, 45, 48, 49, 50, 54, 56, 60, 63, 64,
         70, 72, 75, 80, 81, 84, 90, 96, 98, 100, 105, 108, 112, 120, 126, 128]
GRIDS = [(e, EDGES[(i + 13) % 39], EDGES[(i + 26) % 39]) for i, e in enumerate(EDGES)]
GRIDS += [(e, e, e) for e in (16, 20, 27, 28, 42, 56, 63, 84, 100, 112, 126)]
GRIDS += [(60, 60, 90), (27, 56, 56), (30, 128, 30), (14, 30, 30), (30, 30, 125)]


def _to_grid(c, idx, m_idx, nd):
    f = np.zeros((c.shape[0], int(np.prod(nd))), np.complex128)
    f[:, idx] = c
    f[:, m_idx[1:]] = c[:, 1:].conj()
    f[:, 0] = c[:, 0].real
    return np.fft.ifftn(f.reshape(-1, nd[2], nd[1], nd[0]), axes=(1, 2, 3), norm="forward")


@pytest.mark.parametrize("nd", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_local_and_density_on_edges(nd):
    # a sphere whose extent is about a quarter of every edge, as the cutoffs
    # 20 / 80 Ry give
    print("edges", nd, flush=True)
    hcell = np.diag([2 * np.pi * (n / 4.0 - 0.3) / np.sqrt(20.0) for n in nd])
    gs = pw.GSphere(hcell)
    gs.nd, gs.N = nd, int(np.prod(nd))
    n = gs.nplw + 1
    h, k, l = (np.asarray(a[:n], np.int64) for a in (gs.nga, gs.ngb, gs.ngc))
    idx = h % nd[0] + nd[0] * (k % nd[1] + nd[1] * (l % nd[2]))
    m_idx = (-h) % nd[0] + nd[0] * ((-k) % nd[1] + nd[1] * ((-l) % nd[2]))
    rng = np.random.default_rng(sum(nd))
    nb = 3
    psi = rng.standard_normal((nb, 2 * n))
    psi[:, 1] = 0.0
    v = rng.standard_normal(gs.N)
    occ = np.array([2.0, 1.3, 0.4])
    ctx = pw.PlaneWave(gs, nb)
    try:
        ctx.put(0, psi)
        rho0 = {p: ctx.density(0, nb, occ, 1.0, p) for p in (pw.FP64, pw.MIXED)}
        ctx.set_glocal(v)
        got = {}
        for p in (pw.FP64, pw.MIXED):
            ctx.local(0, 1, nb, p)
            got[p] = ctx.get(1, nb)
        rho = {p: ctx.density(0, nb, occ, 1.0, p) for p in (pw.FP64, pw.MIXED)}
    finally:
        ctx.close()
    f = _to_grid(psi[:, 0::2] + 1j * psi[:, 1::2], idx, m_idx, nd)
    g = np.fft.fftn(f * v.reshape(nd[2], nd[1], nd[0]), axes=(1, 2, 3), norm="forward")
    g = g.reshape(nb, -1)[:, idx]
    ref = psi * np.repeat(gs.recnrm[:n], 2)
    ref[:, 0::2] += g.real
    ref[:, 1::2] += g.imag
    rref = np.einsum("b,bzyx->zyx", occ, f.real ** 2).reshape(-1)
    for p, tol in ((pw.FP64, 1e-12), (pw.MIXED, 3e-6)):
        assert np.abs(got[p] - ref).max() < tol * np.abs(ref).max()
        assert np.abs(rho[p] - rref).max() < tol * np.abs(rref).max()
        assert np.array_equal(rho0[p], rho[p])  # the density does not need a potential


@pytest.mark.parametrize("e", [100, 112])
def test_two_step_density_after_a_cube(e, monkeypatch):
    """e x e planes of a cube and of a slab have rows of their own strides (a slab
    keeps a second twiddle table in LDS): after the cube, the slab's FP64 density
    still runs on the two-step kernels, whose rounding is not that of the Stockham
    lines."""
    occ = np.array([2.0])
    rho = {}
    for nd in ((e, e, e), (e, e, 16)):
        print("edges", nd, flush=True)
        gs = pw.GSphere(np.diag([2 * np.pi * (n / 4.0 - 0.3) / np.sqrt(20.0) for n in nd]))
        gs.nd, gs.N = nd, int(np.prod(nd))
        psi = np.random.default_rng(e).standard_normal((1, 2 * (gs.nplw + 1)))
        psi[:, 1] = 0.0
        ctx = pw.PlaneWave(gs, 1)
        try:
            ctx.put(0, psi)
            rho["two-step"] = ctx.density(0, 1, occ, 1.0)
            monkeypatch.setenv("QX_GENERIC_FFT", "1")
            rho["Stockham"] = ctx.density(0, 1, occ, 1.0)
            monkeypatch.delenv("QX_GENERIC_FFT")
        finally:
            ctx.close()
        assert np.abs(rho["two-step"] - rho["Stockham"]).max() < 1e-12 * rho["Stockham"].max()
        assert not np.array_equal(rho["two-step"], rho["Stockham"])
