"""GPU: the 2D second-order row kernel (one step per launch) at the edges of its tiling: domains
of 2-5 rows and columns, strips that end at, one before and one past a wall (62, 63, 64, 122,
124, 125 columns), items of every remainder against the four-row loop, rectangular cells
(DT/DY not 1/8) and both walls; bitwise against the oracle."""
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import assert_same, banner, gpu_run, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [S.F64, S.REF32, S.C32, S.C32K])
@pytest.mark.parametrize("shape,rows", [((2, 2), 1), ((3, 5), 1), ((5, 62), 2), ((4, 63), 3), ((9, 64), 4), ((7, 122), 5),
                                        ((13, 124), 6), ((11, 125), 7), ((23, 187), 8), ((40, 70), 9), ((31, 66), 1)])
def test_edges(orc, prec, shape, rows):
    for bc, lim, dy in ((S.BC_REFLECT, S.LIM_MC, 1.0), (S.BC_OUTFLOW, S.LIM_MINMOD, 0.9)):  # cell heights in DX
        pb = S.problem(2, 2, *shape, precision=prec, bc=bc, limiter=lim, lx=1.0, ly=dy * shape[1] / shape[0])
        ic = icgen.random_2d(*shape, 5 + rows, block=3)
        banner("row2d", prec, shape, rows, bc, lim)
        assert_same(pb, gpu_run(pb, ic, 3, (rows, 1, 4, 0)), oracle_run(orc, pb, ic, 3), "row2d edges")
