"""GPU: the FP64 step kernels' short division and square-root sequences (quot, rcp_nr2, sqrt_rcp,
rsq_sqrt in shll_device.h) against the IEEE operators, on 2^28 random arguments of the range that they
are used in: the reference form's equal bit for bit, the fast form's square root, whose two roundings
(of x y and of the result) are half a unit each, at most 2 ulp away."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu

PROBE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "probes", "libquotient_probe.so")


def test_quotients_and_roots():
    if not os.path.exists(PROBE):
        pytest.fail("tests/probes/libquotient_probe.so is not built (run __graft_entry__.build())")
    lib = ctypes.CDLL(PROBE)
    out = (ctypes.c_ulonglong * 4)()
    print("[gpu-case] quotients", flush=True)
    assert lib.probe_quotients(ctypes.c_int(256), ctypes.c_ulonglong(20261206), out) == 0
    print("mismatches: quotient %d, root %d, quotient by the root %d; rsq_sqrt's root at most %d ulp" % tuple(out))
    assert tuple(out[:3]) == (0, 0, 0)
    assert out[3] <= 2
