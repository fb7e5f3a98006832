"""GPU: the fast FP64 form's constants are the nearest doubles.  Its sound speed is sqrt(gamma R/CV)
sqrt(q/rho); over many states the roundings of the operations average out, and what is left is the
rounding of that constant, at most half a unit in the last place (2/3 x 2^-53 of 0.748)."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import banner

pytestmark = pytest.mark.gpu


def test_sound_speed_is_not_biased():
    n = 40000
    pb = S.problem(1, 2, n, precision=S.F64F)
    banner("f64f bias")
    with S.Solver(pb, icgen.random_1d(n, 77, block=1)) as s:
        s.step(2)  # every bit of the state in use
        rho, m, E = s.conserved().astype(np.longdouble)
        a = s.stage_fluxes()["a"]
    cv = np.longdouble(1.0 / (1.4 - 1.0))
    exact = np.sqrt(np.longdouble(1.4) / cv * (E - m * m / rho / 2) / rho)
    bias = float(((a - exact) / exact).mean()) * 2.0**53
    print("mean error of the sound speed: %.3f x 2^-53" % bias)
    assert abs(bias) <= 2 / 3 + 0.02
