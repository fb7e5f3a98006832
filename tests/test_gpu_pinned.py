"""GPU: transfers where the process can pin no memory.  A shim in front of the runtime's
hipHostMalloc, in a process of its own, refuses; construction, reads, restarts and sums go on through
ordinary memory, with the same values.  And what stays pinned once no solver is left (the shim counts)."""
import os
import subprocess
import sys

import pytest

import shll_amd as S
from test_gpu_parity import banner

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))

SHIM = r"""
#include <stddef.h>
static int (*real_malloc)(void**, size_t, unsigned), (*real_free)(void*);
int refuse, made, freed;
void shim(void* m, void* f) { *(void**)&real_malloc = m; *(void**)&real_free = f; }
int hipHostMalloc(void** p, size_t n, unsigned flags) {
    if (refuse) return 2; /* hipErrorOutOfMemory */
    ++made;
    return real_malloc(p, n, flags);
}
int hipHostFree(void* p) { ++freed; return real_free(p); }
"""

# the shim comes ahead of the runtime in the library's symbol search; through the library's own handle
# the runtime's functions are found
HEAD = """
import ctypes, sys
sys.path[:0] = [%r, %r]
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import icgen
import shll_amd as S
addr = lambda f: ctypes.cast(f, ctypes.c_void_p)
shim.shim(addr(S.lib().hipHostMalloc), addr(S.lib().hipHostFree))
refuse, made, freed = (ctypes.c_int.in_dll(shim, n) for n in ("refuse", "made", "freed"))
""" % (HERE + "/golden", os.path.join(os.path.dirname(HERE), "shll-sve-cfd_amd"))


def run(tmp_path, body):
    src, lib = tmp_path / "shim.c", tmp_path / "libshim.so"
    src.write_text(SHIM)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)])
    r = subprocess.run([sys.executable, "-c", HEAD + body, str(lib)], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, SHLL_AMD_LIB=S.LIB_PATH))
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout + r.stderr


def test_without_pinned_memory(tmp_path):
    banner("no pinned memory")
    run(tmp_path, """
def values(n):
    pb = S.problem(2, 1, n, n, precision=S.C32K)
    ic = icgen.random_2d(n, n, 5, block=8)
    with S.Solver(pb, ic) as s, S.Solver(pb, S.ic_circle(n, n)) as t:
        s.step(6)
        t.set_state_raw(s.state_raw())
        out = [s.primitives(), s.conserved(), s.conserved_sums(), np.stack(s.state_raw()), t.conserved()]
    b = S.Batch([pb, pb], [ic, ic], [3, 6])
    b.run()
    out += [b.primitives(0), b.conserved(1), b.conserved_sums()]
    b.close()
    return out

refuse.value = 1
without = [values(n) for n in (64, 700)]
assert made.value == 0
refuse.value = 0
for a, b in zip(without, [values(n) for n in (64, 700)]):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)
assert made.value > 0
print("done")
""")


def test_pinned_memory_is_given_back(tmp_path):
    """Large transfers pin a buffer or two per thread; of those, four stay when the last solver goes."""
    banner("pinned memory given back")
    run(tmp_path, """
n = 1500
ic = icgen.random_2d(n, n, 5, block=8)
pb = S.problem(2, 1, n, n, precision=S.F64)
small = S.Solver(S.problem(1, 1, 100, precision=S.F64), S.ic_tube(100))
with S.Solver(pb, ic) as s:
    s.primitives()
assert made.value > 4 and freed.value == 0, (made.value, freed.value)
small.conserved()
small.close()
assert made.value - freed.value == 4, (made.value, freed.value)
pinned = made.value
for _ in range(3):
    with S.Solver(S.problem(2, 1, 100, 100, precision=S.F64), S.ic_circle(100, 100)) as s:
        s.step(3)
        s.primitives()
assert made.value == pinned
print("done")
""")
