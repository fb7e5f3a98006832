"""GPU: the fast FP64 form's scaled arithmetic at energies and densities of any scale, where fluxes
(of order E sqrt(E/rho)) are far larger or smaller than the state: one step against the oracle,
and states that leave the scaled form's range in the middle of a launch."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import assert_oracle_match, banner, gpu_run, oracle_run

pytestmark = pytest.mark.gpu


def scaled(n, seed, rho, energy, block):
    """Random blocks with density times 2^rho and energy times 2^energy, Mach numbers kept."""
    ic = np.array(icgen.random_1d(n, seed, block=block)).reshape(3, n)
    ic[0] = np.ldexp(ic[0], rho)
    ic[1] = np.ldexp(ic[1], (energy - rho) // 2)
    ic[2] = np.ldexp(ic[2], energy - rho)
    return ic.reshape(-1)


# one step of round-off: the tolerance of short runs
@pytest.mark.parametrize("lim", [S.LIM_MINMOD, S.LIM_MC])
@pytest.mark.parametrize("launch", [(1, 1, 1, 0), (8, 4, 1, 0)])
@pytest.mark.parametrize("rho,energy", [(0, 140), (0, 152), (0, 350), (0, 380), (-200, 400), (400, -200), (-148, 148),
                                        (148, -148), (148, 148), (-148, -148), (-152, 152), (152, -152)])
def test_one_step_at_any_scale(orc, rho, energy, launch, lim):
    n = 1003
    pb = S.problem(1, 2, n, precision=S.F64F, limiter=lim)
    ic = scaled(n, 9, rho, energy, 1)  # every cell its own, so that a first step has slopes
    banner("f64f scale", rho, energy, launch, lim)
    want = oracle_run(orc, pb, ic, 1)[1]
    assert np.isfinite(want).all()
    assert_oracle_match(S.F64F, gpu_run(pb, ic, 1, launch)[1], want, "one step")


# sound speeds of 2^10 .. 2^120 cells per step: the state grows by powers of the speed each step
# (energies from 2^26 to 2^600 in four) and loses positivity in some cells
@pytest.mark.parametrize("lim", [S.LIM_MINMOD, S.LIM_MC])
@pytest.mark.parametrize("power", [20, 80, 120, 160, 200, 240])
def test_growth_within_a_launch(power, lim):
    n = 1003
    pb = S.problem(1, 2, n, precision=S.F64F, limiter=lim)
    ic = scaled(n, 9, 0, power, 11)
    banner("f64f growth", power, lim)
    want = gpu_run(pb, ic, 4, (1, 1, 1, 0))[1]
    assert np.isfinite(want).all(axis=0).sum() > 100
    for launch in ((2, 4, 1, 0), (8, 4, 1, 0), (4, 2, 1, 0), (2, 4, 4, 0)):
        np.testing.assert_array_equal(gpu_run(pb, ic, 4, launch)[1], want, err_msg=str(launch))
