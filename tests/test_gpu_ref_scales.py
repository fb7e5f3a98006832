"""GPU: the reference forms' primitive recovery and split fluxes at densities and momenta of any
scale, down to the denormal range: the quotients' remainders are exact only in part of it, so the
shared reciprocals are for cells inside (RefRange in shll_device.h).  Bitwise against the oracle."""
import numpy as np
import pytest

import shll_amd as S
from test_gpu_parity import MODES, banner, opb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("decades", ["low", "high", "all"])
@pytest.mark.parametrize("shape", [(20011,), (131, 150)])
@pytest.mark.parametrize("prec", [S.F64, S.REF32])
def test_stage_fluxes_at_any_density(orc, prec, shape, decades):
    rng = np.random.default_rng(23)
    n, nvel = int(np.prod(shape)), len(shape)
    lim = 1000 if prec == S.F64 else 120
    lo, hi = {"low": (-1.06 * lim, -0.3 * lim), "high": (0.3 * lim, lim), "all": (-lim, lim)}[decades]
    rho = 2.0 ** rng.uniform(lo, hi, n)
    T = 2.0 ** rng.uniform(-4, 4, n)
    v = [2.0 ** rng.uniform(-lim / 2, 1, n) * rng.choice([-1.0, 1.0], n) for _ in range(nvel)]
    for q in v:
        q[rng.random(n) < 0.5] *= 0.5 ** rng.integers(0, 40)
        q[rng.random(n) < 0.1] = 0.0
    ic = np.stack([rho, *v, T])
    banner("stage scales", prec, shape, decades)
    for order in (1, 2):
        pb = S.problem(len(shape), order, *shape, precision=prec)
        with np.errstate(all="ignore"), S.Solver(pb, ic) as s:
            got = s.stage_fluxes()
            want = orc.stage(opb(orc, pb), MODES[prec], ic)
        for key in got:
            np.testing.assert_array_equal(got[key], want[key].reshape(got[key].shape), err_msg="%s o%d" % (key, order))
