"""GPU: the reference forms' primitive recovery takes shared reciprocals and fused operations
for cells in range and the operators themselves for the others (RefArith in shll_device.h), per
cell.  One step from states on both sides of every edge of that range -- temperatures over 40
(FP64: 400) decades, Mach numbers down to zero, a few non-finite and vacuum cells -- equals the
oracle's bits."""
import numpy as np
import pytest

import shll_amd as S
from test_gpu_parity import banner, opb

pytestmark = pytest.mark.gpu


def wild(rng, n, nvel, decades, mach):
    """Primitives with T = 10^U(-decades, decades), velocities of Mach 10^U(-mach, 0.3) or 0."""
    T = 10.0 ** rng.uniform(-decades, decades, n)
    T[rng.random(n) < 0.3] = 1.0
    v = []
    for _ in range(nvel):
        m = 10.0 ** rng.uniform(-mach, 0.3, n) * rng.choice([-1.0, 1.0], n)
        m[rng.random(n) < 0.3] = 0.0
        v.append(m * np.sqrt(1.4 * T))
    rho = 10.0 ** rng.uniform(-3, 3, n)
    bad = rng.integers(0, n, 6)
    rho[bad[0]], T[bad[1]], rho[bad[2]], v[0][bad[3]], T[bad[4]] = 0.0, np.nan, np.inf, np.nan, -1.0
    return np.stack([rho, *v, T])


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("shape", [(777,), (33, 70)])
@pytest.mark.parametrize("prec", [S.F64, S.REF32])
def test_one_step_from_wild_states(orc, prec, shape, order):
    rng = np.random.default_rng(17 + order)
    n = int(np.prod(shape))
    dec, mach = (200, 220) if prec == S.F64 else (17, 20)
    pb = S.problem(len(shape), order, *shape, precision=prec)
    banner("wild states", prec, shape, order)
    with np.errstate(all="ignore"):
        ic = wild(rng, n, len(shape), dec, mach)
        with S.Solver(pb, ic) as s:
            s.step(1)
            got = s.conserved()
        _, ref = orc.run(opb(orc, pb), orc.F64 if prec == S.F64 else orc.REF32, ic, 1)
    np.testing.assert_array_equal(got, ref)
