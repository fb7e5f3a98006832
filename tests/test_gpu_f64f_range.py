"""GPU: the fast FP64 form's scaled arithmetic (densities and energies within [2^-200, 2^400], at
most 64 steps per launch) against its general one.  Density times a power of two scales every
quantity exactly, so a run outside the range gives the same bits, scaled; and launches of more
than 64 steps give those of shorter ones."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import banner, gpu_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lim", [S.LIM_MINMOD, S.LIM_MC])
@pytest.mark.parametrize("launch", [(1, 8, 1, 0), (2, 16, 1, 0), (8, 16, 1, 0), (4, 16, 4, 0)])
@pytest.mark.parametrize("power", [399, 450, -199, -300])
def test_outside_the_scaled_range(lim, launch, power):
    n = 1003
    pb = S.problem(1, 2, n, precision=S.F64F, limiter=lim)
    ic = np.array(icgen.random_1d(n, 9, block=11)).reshape(3, n)
    far = ic.copy()
    far[0] = np.ldexp(far[0], power)
    banner("f64f range", lim, launch, power)
    got = gpu_run(pb, far.reshape(-1), 40, launch)[1]
    np.testing.assert_array_equal(np.ldexp(got, -power), gpu_run(pb, ic.reshape(-1), 40, launch)[1])


def test_a_mixed_state_takes_one_form_per_wavefront():
    """One cell of a wavefront out of range: its neighbours' values stay those of the oracle-checked
    one-cell-per-lane, one-step launches."""
    n = 700
    pb = S.problem(1, 2, n, precision=S.F64F)
    ic = np.array(icgen.random_1d(n, 10, block=9)).reshape(3, n)
    ic[0, 300] = 2.0**-210
    banner("f64f mixed")
    want = gpu_run(pb, ic.reshape(-1), 3, (1, 1, 1, 0))[1]
    assert np.isfinite(want).all()
    np.testing.assert_array_equal(gpu_run(pb, ic.reshape(-1), 3, (8, 3, 1, 0))[1], want)


def test_more_than_64_steps_per_launch():
    n = 2001
    pb = S.problem(1, 2, n, precision=S.F64F)
    ic = icgen.random_1d(n, 11, block=30)
    banner("f64f long launches")
    np.testing.assert_array_equal(gpu_run(pb, ic, 203, (8, 100, 1, 0))[1], gpu_run(pb, ic, 203, (8, 50, 1, 0))[1])
