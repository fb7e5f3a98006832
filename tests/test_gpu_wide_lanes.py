"""GPU: eight cells per lane in the FP64 forms, whose states pass through LDS between memory order
and lane order: tubes of one to a few segments, a cell more or less than they hold, so that the
first, the last and inner segments are whole or cut.  FP64 bitwise against the oracle; F64F bitwise
against one cell per lane."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import assert_same, banner, gpu_run, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", [1, 4])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("bc", [S.BC_OUTFLOW, S.BC_REFLECT])
def test_segment_edges(orc, order, bc, waves):
    for n in (2, 9, 64, 509, 510, 511, 512, 513, 959, 960, 961, 1472, 1999, 2046, 2049, 4100):
        for k in (1, 8):
            pb = S.problem(1, order, n, precision=S.F64, bc=bc)
            ic = icgen.random_1d(n, 30 + n, block=5)
            banner("wide lanes", order, bc, waves, n, k)
            assert_same(pb, gpu_run(pb, ic, 2 * k + 1, (8, k, waves, 0)), oracle_run(orc, pb, ic, 2 * k + 1), "n=%d" % n)
            pb = S.problem(1, order, n, precision=S.F64F, bc=bc)
            np.testing.assert_array_equal(gpu_run(pb, ic, 2 * k + 1, (8, k, waves, 0))[1],
                                          gpu_run(pb, ic, 2 * k + 1, (1, 1, 1, 0))[1], err_msg="F64F n=%d" % n)
