"""GPU: steps of the reference forms on states as thin as the type holds, whose products with
DT/DX reach the denormal range and round there, and mixed with ordinary ones.  Bitwise against
the oracle."""
import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import MODES, banner, gpu_run, opb

pytestmark = pytest.mark.gpu

LOW = {S.F64: [-960, -1000, -1015, -1021], S.REF32: [-60, -100, -115, -124, -127]}


def check(orc, pb, ic, steps, launches):
    with np.errstate(all="ignore"):
        want = orc.run(opb(orc, pb), MODES[pb.precision], ic, steps, nthreads=4)[1]
        for launch in launches:
            got = gpu_run(pb, ic, steps, launch)[1]
            np.testing.assert_array_equal(got, want, err_msg="%s" % (launch,))


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("prec", [S.F64, S.REF32])
@pytest.mark.parametrize("mixed", [False, True])
def test_thin_tubes(orc, prec, order, mixed):
    n = 1503
    for power in LOW[prec]:
        ic = np.array(icgen.random_1d(n, 31, block=4)).reshape(3, n)
        ic[0] = np.ldexp(ic[0], power)
        if mixed:
            ic[0, 400:420] = 1.0
            ic[0, 1000:] = 1.0
        banner("thin 1d", prec, order, power, mixed)
        pb = S.problem(1, order, n, precision=prec, limiter=S.LIM_MC if order == 2 else S.LIM_MINMOD)
        check(orc, pb, ic, 5, ((1, 1, 1, 0), (2, 5, 1, 0), (8, 5, 1, 0), (2, 5, 4, 0), (4, 2, 4, 0)))


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("prec", [S.F64, S.REF32])
@pytest.mark.parametrize("mixed", [False, True])
def test_thin_planes(orc, prec, order, mixed):
    nx, ny = 67, 131
    for power in LOW[prec]:
        ic = np.array(icgen.random_2d(nx, ny, 32, block=4)).reshape(4, nx, ny)
        ic[0] = np.ldexp(ic[0], power)
        if mixed:
            ic[0, 20:23, 30:60] = 1.0
            ic[0, 40:] = 1.0
        banner("thin 2d", prec, order, power, mixed)
        for lx, ly in ((67 / 131, 1.0), (1.0, 1.0)):  # square cells, and others
            pb = S.problem(2, order, nx, ny, precision=prec, lx=lx, ly=ly, limiter=S.LIM_MC if order == 2 else S.LIM_MINMOD)
            check(orc, pb, ic.reshape(4, -1), 5, ((1, 1, 4, 0), (1, 2, 4, 0), (1, 4, 4, 0)) if order == 1 else ((1, 1, 4, 0),))
