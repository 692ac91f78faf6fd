"""The two-step transforms of Bloch bands on every edge they cover: (T + V) c
against the numpy oracle at k-points inside and outside the first zone (the h
range of a sphere is then not symmetric, or on one side of zero), and on two
grids with an edge that is not covered, which the Stockham kernels take."""
import numpy as np
import pytest

from oracle import kpoint as OK
from qxmd_amd import pw

pytestmark = pytest.mark.gpu

EDGES = [16, 18, 20, 21, 24, 25, 27, 28, 30, 32, 35, 36, 40, 42, 45, 48, 49, 50, 54, 56, 60, 63, 64,
         70, 72, 75, 80, 81, 84, 90, 96, 98, 100, 105, 108, 112, 120, 126, 128]
GRIDS = [(e, EDGES[(i + 13) % 39], EDGES[(i + 26) % 39]) for i, e in enumerate(EDGES)]
GRIDS = [g for g in GRIDS if g[0] * g[1] <= 8192]
GRIDS += [(128, 16, 20), (126, 20, 16), (120, 27, 24), (112, 16, 30), (105, 21, 18)]
GRIDS += [(e, e, e) for e in (16, 20, 28, 30, 42, 64, 90)] + [(14, 30, 30), (30, 14, 30)]


@pytest.mark.parametrize("nd", GRIDS, ids=lambda n: "x".join(map(str, n)))
def test_khpsi_local_on_edges(nd):
    print("edges", nd, flush=True)
    hcell = np.diag([2 * np.pi * (n / 4.0 - 0.3) / np.sqrt(20.0) for n in nd])
    gs = pw.GSphere(hcell)
    gs.nd, gs.N = nd, int(np.prod(nd))
    rng = np.random.default_rng(sum(nd))
    v = rng.standard_normal(gs.N)
    nb = 2
    ctx = pw.PlaneWave(gs, 2)
    try:
        ctx.set_glocal(v)
        far = [[0.4 * n for n in nd], [-0.4 * n for n in nd]]
        near = [[0, 0, 0], [0.5, 0.25, -0.4], [0.2 * nd[0], -0.2 * nd[1], 0.2 * nd[2]]]
        for kf, ecut in ((near, 20.0), (far, 1.2)):
            ctx.kpoints_set(kf, 2 * np.pi * np.linalg.inv(hcell).T, ecut, nb)
            data = []
            for ik in range(len(kf)):
                hkl, kin = ctx.kpoints_sphere(ik)
                c = rng.standard_normal((nb, len(kin))) + 1j * rng.standard_normal((nb, len(kin)))
                ctx.kput(0, ik, c)
                data.append((c, hkl, kin))
            ctx.khpsi(0, 1)
            for ik, (c, hkl, kin) in enumerate(data):
                ref = OK.hk_apply(c, hkl, kin, v.reshape(nd[2], nd[1], nd[0]))
                assert np.abs(ctx.kget(1, ik) - ref).max() < 1e-12 * np.abs(ref).max(), ik
    finally:
        ctx.close()


@pytest.mark.parametrize("e", [16, 20, 30, 36, 40])
@pytest.mark.parametrize("over", [0, 1])
def test_khpsi_local_many_blocks(e, over):
    """(k, band) blocks just below and at 4096 planes, where the plane pass takes two
    wavefronts a block on two to four row groups (20, 30, 36; 16 has one, 40 five)."""
    nk = (4096 + e - 1) // e - 1 + over
    print("edge", e, "blocks", nk, flush=True)
    hcell = np.eye(3) * 2 * np.pi * (e / 4.0 - 0.3) / np.sqrt(20.0)
    gs = pw.GSphere(hcell)
    gs.nd, gs.N = (e, e, e), e ** 3
    rng = np.random.default_rng(e)
    v = rng.standard_normal(gs.N)
    kf = rng.uniform(-0.5, 0.5, (nk, 3))
    ctx = pw.PlaneWave(gs, 1)
    try:
        ctx.set_glocal(v)
        ctx.kpoints_set(kf, 2 * np.pi * np.linalg.inv(hcell).T, 20.0, 1)
        data = []
        for ik in range(nk):
            hkl, kin = ctx.kpoints_sphere(ik)
            c = rng.standard_normal((1, len(kin))) + 1j * rng.standard_normal((1, len(kin)))
            ctx.kput(0, ik, c)
            data.append((c, hkl, kin))
        ctx.khpsi(0, 1)
        for ik in list(range(0, nk, 7)) + [nk - 1]:
            c, hkl, kin = data[ik]
            ref = OK.hk_apply(c, hkl, kin, v.reshape(e, e, e))
            assert np.abs(ctx.kget(1, ik) - ref).max() < 1e-12 * np.abs(ref).max(), ik
    finally:
        ctx.close()
