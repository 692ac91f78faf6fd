"""The FP64 products that leave half of the work out, by Gram-Schmidt against the
oracle: the overlap on and below the diagonal tiles, psi L^-T up to each tile's
last column, at band counts on, below and above the edges of the 96 and 128
tiles, with each work schedule, and the orthonormality of the result.  Odd
counts have the same overlap and take gemm_small.hip for psi L^-T."""
import numpy as np
import pytest

import oracle as O
from qxmd_amd import pw
from qxmd_amd.system import initial_wavefunctions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [256, 257, 258, 286, 288, 289, 290, 384, 385, 386])
def test_schmidt_tile_edges(si64, nb):
    print("schmidt", nb, flush=True)
    raw = initial_wavefunctions(si64, nb)
    ref, okr = O.schmidt(raw)
    ctx = pw.PlaneWave(pw.GSphere(si64.cell.hcell), nb)
    try:
        for sched in (pw.SCHED_TIMED, pw.SCHED_STREAMK, pw.SCHED_SLICED):
            pw.set_gemm_schedule(sched)
            got, ok = ctx.schmidt_host(raw)
            assert ok and okr
            # as for 300 bands: the Cholesky factor's condition times round-off
            assert np.abs(got - ref).max() < 1e-10 * np.abs(ref).max()
            s = 2 * got @ got.T - np.outer(got[:, 0], got[:, 0])
            assert np.abs(s - np.eye(nb)).max() < 1e-11
    finally:
        pw.set_gemm_schedule(pw.SCHED_TIMED)
        ctx.close()
