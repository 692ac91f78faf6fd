"""The contractions with a dimension of the output below 256, through the KB
term of H|psi> on random tables: row and column counts around the tile edges
(16, 48, 64), one band, odd projector counts (rows that are not 16-byte
aligned), against numpy.  FP64: sums of 1648 products in another order, 1e-13
of the largest value.  Mixed: two FP32 products of operands rounded to FP32,
sqrt(1648) 6e-8 = 2.4e-6 of the largest value."""
import numpy as np
import pytest

from qxmd_amd import pw
from qxmd_amd.system import diamond_si

pytestmark = pytest.mark.gpu

SHAPES = [(1, 5), (4, 1), (5, 6), (16, 16), (17, 15), (32, 20), (47, 64), (48, 48), (49, 47),
          (64, 65), (65, 64), (97, 33), (130, 81), (255, 255), (384, 31), (31, 300)]


@pytest.mark.parametrize("npj,nb", SHAPES)
def test_kb_shapes(npj, nb):
    print("KB term", npj, "projectors", nb, "bands", flush=True)
    gs = pw.GSphere(diamond_si(1).hcell)
    n = gs.nplwex
    rng = np.random.default_rng(1000 * npj + nb)
    psi = rng.standard_normal((nb, n))
    psi[:, 1] = 0.0
    eq = rng.standard_normal((npj, 1, n))
    d = rng.standard_normal((npj, 1))
    b = eq[:, 0, :]
    p = 2.0 * psi @ b.T - np.outer(psi[:, 0], b[:, 0]) - 2.0 * np.outer(psi[:, 1], b[:, 1])
    ref = (p * d[:, 0]) @ b
    ctx = pw.PlaneWave(gs, nb)
    try:
        ctx.set_glocal(rng.standard_normal(gs.N))
        ctx.put(0, psi)
        for prec, tol in ((pw.FP64, 1e-13), (pw.MIXED, 2.4e-6)):
            ctx.set_kb(np.zeros((1, 1, n)), np.zeros(1, np.int32), np.zeros((1, 1)))
            ctx.hpsi(0, 1, nb, prec)  # no projectors: the local part alone
            local = ctx.get(1, nb)
            ctx.set_kb(eq, np.ones(npj, np.int32), d)
            ctx.hpsi(0, 1, nb, prec)
            got = ctx.get(1, nb) - local
            again = ctx.hpsi(0, 2, nb, prec) or ctx.get(2, nb) - local
            assert np.abs(got - ref).max() < tol * np.abs(ref).max()
            if nb > 4:  # matrix-vector products below that add K slices atomically
                assert np.array_equal(got, again)  # no sum depends on timing
        _, sl = ctx.hckbpp_g(psi, np.zeros_like(psi), want_slmir=True, lmmax=1, natom=npj)
        assert np.abs(sl[:, :, 0] - p).max() < 1e-13 * np.abs(p).max()
    finally:
        ctx.close()


@pytest.mark.parametrize("npj,nb", [(2043, 40), (2046, 40), (1241, 66), (651, 127)])
def test_kb_long(si64, npj, nb):
    """The mixed KB term on both sides of 2^30 products, where 64 x 64 tiles take
    over from 32 x 32 ones.  Two FP32 products of operands rounded to FP32:
    sqrt(13134) 6e-8 = 6.9e-6 of the largest value."""
    print("KB term", npj, "projectors", nb, "bands", flush=True)
    n = si64.nplwex
    rng = np.random.default_rng(npj)
    psi = rng.standard_normal((nb, n))
    psi[:, 1] = 0.0
    b = rng.standard_normal((npj, n))
    d = rng.standard_normal((npj, 1))
    p = 2.0 * psi @ b.T - np.outer(psi[:, 0], b[:, 0])
    ref = (p * d[:, 0]) @ b
    ctx = pw.PlaneWave(pw.GSphere(si64.cell.hcell), nb)
    try:
        ctx.set_glocal(np.zeros(ctx.gs.N))
        ctx.put(0, psi)
        ctx.set_kb(b[:, None, :], np.ones(npj, np.int32), d)
        ctx.hpsi(0, 1, nb, pw.MIXED)
        got = ctx.get(1, nb) - psi * np.repeat(ctx.gs.recnrm[: n // 2], 2)
        assert np.abs(got - ref).max() < 6.9e-6 * np.abs(ref).max()
    finally:
        ctx.close()


@pytest.mark.parametrize("npj,nb", [(5500, 32), (3648, 192)])
def test_fp32_chains(si64, npj, nb):
    """FP32 products are added in FP32 over about 1024 k and from there in FP64.
    The products are 1.5 + 2^-13 x bit: sums of up to 1365 of them stay below 2048,
    where FP32 holds every multiple of 2^-13, so the projection is exact and the
    back-projection gets it rounded to FP32 once; longer chains round on the way.
    Outputs with tiles enough (of 32 x 32 and of 64 x 64) to leave K in one or
    two slices by their number alone."""
    print("FP32 chains", npj, nb, flush=True)
    n = si64.nplwex
    rng = np.random.default_rng(7)
    psi = 1.5 + 2.0 ** -13 * rng.integers(0, 2, (nb, n))
    psi[:, 1] = 0.0
    ctx = pw.PlaneWave(pw.GSphere(si64.cell.hcell), nb)
    try:
        ctx.set_glocal(np.zeros(ctx.gs.N))
        ctx.put(0, psi)
        p = 2.0 * psi.sum(1) - psi[:, 0]
        ref = psi * np.repeat(ctx.gs.recnrm[: n // 2], 2) + p.astype(np.float32)[:, None]
        d = np.zeros((npj, 1))
        d[npj - 1] = 1.0  # the one projector that counts
        ctx.set_kb(np.ones((npj, 1, n)), np.ones(npj, np.int32), d)
        ctx.hpsi(0, 1, nb, pw.MIXED)
        # FP64 roundings of sums below 65536
        assert np.abs(ctx.get(1, nb) - ref).max() < 1e-10
    finally:
        ctx.close()
