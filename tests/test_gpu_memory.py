"""GPU: device memory held by a solver or batch that has been made and stepped and not yet read: its
two state buffers (and a batch's initial state), not the doubles its initial data came in."""
import ctypes
import time

import numpy as np
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import banner

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert S.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("prec,words", [(S.F64, 8), (S.REF32, 4), (S.C32K, 8)])
@pytest.mark.parametrize("batch", [False, True])
def test_initial_data_are_not_kept(prec, words, batch):
    n = 1500
    ic = icgen.random_2d(n, n, 3, block=100)
    pb = S.problem(2, 1, n, n, precision=prec)
    banner("memory", prec, batch)
    with S.Solver(S.problem(2, 1, 64, 64, precision=prec), icgen.random_2d(64, 64, 1)) as warm:  # runtime's own
        warm.step(5)
        warm.primitives()
    state = 4 * words * n * n
    before = free_bytes()
    if batch:
        s = S.Batch([pb], [ic], [3])
        s.run()
        held = 3 * state
    else:
        s = S.Solver(pb, ic)
        s.step(3)
        held = 2 * state
    most = held + (24 << 20)  # the initial data: 72 MB
    for _ in range(100):  # the runtime returns freed memory a moment later
        used = before - free_bytes()
        if used < most:
            break
        time.sleep(0.02)
    assert used < most, "used %d, state buffers %d" % (used, held)
    got = s.primitives(0) if batch else s.primitives()
    assert np.isfinite(got).all()
    s.close()
