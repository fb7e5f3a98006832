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
    # reads pass through that buffer too, between any steps
    first = s.primitives(0) if batch else s.primitives()
    if not batch:
        cons = s.conserved()
        s.step(2)
        s.primitives()
        s.step(3)
        with S.Solver(pb, ic) as t:
            t.step(3)
            np.testing.assert_array_equal(t.conserved(), cons)
            t.step(5)
            np.testing.assert_array_equal(t.state_raw(), s.state_raw())
    assert np.isfinite(first).all()
    s.close()


@pytest.mark.parametrize("prec", [S.F64F, S.REF32, S.C32, S.C32K])
def test_initial_data_of_uneven_batches(prec):
    """Large initial data pass through the second state buffer, in REF32 half of the cells at a time:
    halves and transfers end inside instances, in their padding and between them.  Each
    instance is that of a solver of its own, whose data fit one transfer."""
    for sizes in ([3, 100003, 64, 170000, 5, 160001, 1000, 130001], [100000] * 4, [64, 128, 174700, 174700, 64, 128], [350000, 2]):
        ics = [icgen.random_1d(n, 20 + i, block=500) for i, n in enumerate(sizes)]
        pbs = [S.problem(1, 1, n, precision=prec) for n in sizes]
        banner("initial data", prec, sizes)
        b = S.Batch(pbs, ics, [1] * len(sizes))
        for i, n in enumerate(sizes):
            part = min(n, 170000)  # 4 MB
            with S.Solver(S.problem(1, 1, part, precision=prec), np.array(ics[i]).reshape(3, n)[:, :part].reshape(-1)) as s:
                np.testing.assert_array_equal(b.conserved(i)[:, :part], s.conserved(), err_msg="n=%d" % n)
            if part < n:
                with S.Solver(S.problem(1, 1, n - part, precision=prec), np.array(ics[i]).reshape(3, n)[:, part:].reshape(-1)) as s:
                    np.testing.assert_array_equal(b.conserved(i)[:, part:], s.conserved(), err_msg="n=%d" % n)
        b.close()
