"""Nonlocal forces where the projectors do not fit one set of weighted bands:
contexts of few bands (rows of the force workspace, in two chunks), of fewer
bands than projectors (a slot, in chunks) and of more, for one to twenty bands and
for an odd number above 256, against the oracle."""
import numpy as np
import pytest

import oracle as O
import test_gpu_parity as parity
from qxmd_amd.system import initial_wavefunctions, model_kb_projectors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbmax,nb", [(1, 1), (5, 5), (20, 20), (67, 20), (150, 20), (300, 20),
                                      (257, 257)])
def test_kb_forces_rows(si64, nbmax, nb):
    print("forces", nbmax, nb, flush=True)
    gs, ctx, H, v = parity._setup(si64, nbmax)
    eq, lmx, vcl, cl = model_kb_projectors(si64, si64.cell)
    psi, _ = O.schmidt(initial_wavefunctions(si64, nb))
    occ = np.linspace(2.0, 0.0, nb)
    ctx.put(0, psi)
    f = ctx.kb_forces(0, nb, occ, np.zeros((len(lmx), 3)))
    nw = si64.nplw + 1
    _, sl = O.hckbpp_g(eq, lmx, vcl, psi, np.zeros_like(psi))
    fo = O.kbnlpp_frc2(eq, lmx, vcl, psi, occ, sl, si64.gx[:nw], si64.gy[:nw], si64.gz[:nw])
    # as for the device forces elsewhere: sums over bands and waves that cancel
    assert np.abs(f - fo).max() < 1e-10 * np.abs(fo).max()
