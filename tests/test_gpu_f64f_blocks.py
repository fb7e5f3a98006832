"""GPU: the fast FP64 form in cooperative blocks, whose wavefronts swap edge fluxes: one cell far
out of the range of the others, or not a number, in one wavefront of a block.  The other
wavefronts' cells are those of one-cell-per-lane, one-step launches (independent wavefronts)."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import banner, gpu_run

pytestmark = pytest.mark.gpu


# cells at a wavefront's edge (2 cells per lane: the first item's wavefronts hold cells -1 - h ...
# of 128 each), inside the first, second and third wavefront
@pytest.mark.parametrize("lim", [S.LIM_MINMOD, S.LIM_MC])
@pytest.mark.parametrize("cell", [100, 121, 127, 128, 133, 200, 300])
@pytest.mark.parametrize("launch", [(2, 3, 4, 0), (4, 3, 4, 0), (8, 3, 4, 0)])
def test_one_odd_cell_in_a_block(launch, cell, lim):
    n = 2500
    pb = S.problem(1, 2, n, precision=S.F64F, limiter=lim)
    ic = np.array(icgen.random_1d(n, 10, block=9)).reshape(3, n)
    banner("f64f odd cell", launch, cell, lim)
    thin = ic.copy()
    thin[0, cell] = 2.0**-210
    want = gpu_run(pb, thin.reshape(-1), 3, (1, 1, 1, 0))[1]
    assert np.isfinite(want).all()
    np.testing.assert_array_equal(gpu_run(pb, thin.reshape(-1), 3, launch)[1], want)
    nan = ic.copy()
    nan[2, cell] = np.nan
    far = np.abs(np.arange(n) - cell) > 6  # two cells a step
    want = gpu_run(pb, nan.reshape(-1), 3, (1, 1, 1, 0))[1][:, far]
    assert np.isfinite(want).all()
    np.testing.assert_array_equal(gpu_run(pb, nan.reshape(-1), 3, launch)[1][:, far], want)
