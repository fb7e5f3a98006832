"""GPU: the FP64 first-order row pipeline (1 or 2 steps per launch on states above 448 MB, here 7.5e6
cells), at the edges of its items: domains of a few rows or columns and of one strip and a remainder,
both walls, rectangular cells, 1 and 4 wavefronts per block, heights with a remainder, a last launch
of fewer steps; and a batch whose tiny domains take it too.  Bitwise against the oracle."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import banner, gpu_run, opb

pytestmark = pytest.mark.gpu

CELLS = 7500000


@pytest.mark.parametrize("bc", [S.BC_REFLECT, S.BC_OUTFLOW])
@pytest.mark.parametrize("nx,ny", [(CELLS // 3 + 1, 3), (3, CELLS // 3 + 1), (CELLS // 63 + 1, 63), (2501, 3001), (CELLS // 66, 67)])
def test_pipeline(orc, nx, ny, bc):
    steps = 3
    pb = S.problem(2, 1, nx, ny, precision=S.F64, bc=bc, lx=1.0, ly=(0.9 if bc == S.BC_OUTFLOW else 1.0) * ny / nx)
    ic = icgen.random_2d(nx, ny, 41, block=3)
    want = orc.run(opb(orc, pb), orc.F64, ic, steps, nthreads=8)[1]
    for launch in ((1, 1, 1, 0), (1, 2, 4, 0), (23, 2, 1, 0), (50, 1, 4, 0)):
        banner("pipeline", nx, ny, bc, launch)
        np.testing.assert_array_equal(gpu_run(pb, ic, steps, launch)[1], want, err_msg=str(launch))


@pytest.mark.parametrize("launch", [(1, 2, 1, 0), (1, 1, 4, 4), (30, 2, 4, 8)])
def test_batch_with_tiny_domains(orc, launch):
    shapes = [(2, 2), (2600, 2900), (3, 70), (70, 3), (2, 5), (65, 64), (33, 127)]
    steps = [7, 3, 5, 4, 2, 6, 1]
    pbs = [S.problem(2, 1, nx, ny, precision=S.F64, lx=1.0, ly=ny / nx) for nx, ny in shapes]
    ics = [icgen.random_2d(nx, ny, 50 + i, block=3) for i, (nx, ny) in enumerate(shapes)]
    banner("pipeline batch", launch)
    b = S.Batch(pbs, ics, steps)
    b.set_launch(*launch)
    b.run()
    for i, pb in enumerate(pbs):
        want = orc.run(opb(orc, pb), orc.F64, ics[i], steps[i], nthreads=8)[1]
        np.testing.assert_array_equal(b.conserved(i), want, err_msg="%s" % (shapes[i],))
    b.close()
