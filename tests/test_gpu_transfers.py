"""GPU: states and results across the sizes at which a transfer goes through one pinned buffer,
several, or several threads (4 MiB), singly and gathered from the instances of a batch."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import banner

pytestmark = pytest.mark.gpu


# 3 variables: one double below, at and above 4 MiB of values; many buffers with an odd rest
@pytest.mark.parametrize("prec", [S.F64, S.C32K])
@pytest.mark.parametrize("n", [174762, 174763, 349526, 1500007])
def test_round_trip(prec, n):
    pb = S.problem(1, 1, n, precision=prec)
    banner("transfers", prec, n)
    with S.Solver(pb, icgen.random_1d(n, 1, block=1000)) as a, S.Solver(pb, S.ic_tube(n)) as b:
        want, prim = a.conserved(), a.primitives()
        b.set_state_raw(a.state_raw())
        np.testing.assert_array_equal(b.conserved(), want)
        np.testing.assert_array_equal(b.primitives(), prim)
        np.testing.assert_array_equal(b.conserved(), want)


def test_batch_of_uneven_sizes():
    """Each instance of a batch holds what a solver of its own holds."""
    sizes = [3, 100003, 64, 174763, 5, 400001, 1000, 174762]
    pbs = [S.problem(1, 1, n, precision=S.F64) for n in sizes]
    ics = [icgen.random_1d(n, 20 + i, block=500) for i, n in enumerate(sizes)]
    banner("transfers batch")
    b = S.Batch(pbs, ics, [1] * len(sizes))
    for i, n in enumerate(sizes):
        with S.Solver(pbs[i], ics[i]) as s:
            np.testing.assert_array_equal(b.conserved(i), s.conserved(), err_msg="n=%d" % n)
            np.testing.assert_array_equal(b.primitives(i), s.primitives(), err_msg="n=%d" % n)
    b.close()
