"""GPU: the 2D first-order register tiles at the edges of their tiling: domains of a few rows and
columns, one row or column more or less than tiles and strips hold, every number of steps per
launch, rectangular cells (DT/DY not 1/8), both walls, a last launch of fewer steps; and each
tile height on a domain large enough to take it.  Bitwise against the oracle."""
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import assert_same, banner, gpu_run, oracle_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [S.F64, S.REF32, S.C32, S.C32K])
@pytest.mark.parametrize("shape,k", [((2, 2), 1), ((3, 5), 8), ((14, 62), 1), ((15, 63), 1), ((13, 124), 2), ((25, 125), 2),
                                     ((10, 64), 3), ((23, 117), 3), ((8, 57), 4), ((13, 121), 4), ((33, 65), 4),
                                     ((17, 49), 8), ((41, 97), 8)])
def test_edges(orc, prec, shape, k):
    for bc, dy in ((S.BC_REFLECT, 1.0), (S.BC_OUTFLOW, 0.9)):
        pb = S.problem(2, 1, *shape, precision=prec, bc=bc, lx=1.0, ly=dy * shape[1] / shape[0])
        ic = icgen.random_2d(*shape, 3 + k, block=3)
        banner("tile2d", prec, shape, k, bc)
        assert_same(pb, gpu_run(pb, ic, 2 * k + 1, (1, k, 4, 0)), oracle_run(orc, pb, ic, 2 * k + 1), "tile edges")


@pytest.mark.parametrize("prec,shape,k", [(S.F64, (410, 600), 2), (S.REF32, (60, 100), 8), (S.C32, (310, 700), 4),
                                          (S.C32K, (310, 700), 4), (S.C32K, (1610, 1100), 4)])
def test_taller_tiles(orc, prec, shape, k):
    pb = S.problem(2, 1, *shape, precision=prec, lx=1.0, ly=shape[1] / shape[0])
    ic = icgen.random_2d(*shape, 11, block=7)
    banner("tall tiles", prec, shape, k)
    assert_same(pb, gpu_run(pb, ic, k + 2, (1, k, 4, 0)), oracle_run(orc, pb, ic, k + 2), "tall tiles")


@pytest.mark.parametrize("k", [2, 3, 4])
def test_f64_heights_on_many_tiles(orc, k):
    """More tiles of 24 rows than twice the compute units: 16 rows below 4 steps per launch."""
    pb = S.problem(2, 1, 1003, 701, precision=S.F64, lx=1.0, ly=701 / 1003)
    ic = icgen.random_2d(1003, 701, 12, block=7)
    banner("F64 heights", k)
    assert_same(pb, gpu_run(pb, ic, 2 * k + 1, (1, k, 4, 0)), oracle_run(orc, pb, ic, 2 * k + 1), "F64 heights")


@pytest.mark.parametrize("prec", [S.F64, S.REF32, S.C32, S.C32K])
@pytest.mark.parametrize("shape,k", [((10, 62), 1), ((11, 63), 1), ((8, 61), 2), ((17, 66), 2), ((6, 64), 3), ((13, 59), 3),
                                     ((4, 60), 4), ((5, 57), 4), ((9, 121), 4)])
def test_one_row_per_wavefront(orc, prec, shape, k):
    """Few tiles: 12 rows, of which 12 - 2k are owned, at one row or column more or less."""
    pb = S.problem(2, 1, *shape, precision=prec, lx=1.0, ly=shape[1] / shape[0])
    ic = icgen.random_2d(*shape, 5 + k, block=3)
    banner("12 rows", prec, shape, k)
    assert_same(pb, gpu_run(pb, ic, 2 * k + 1, (1, k, 4, 0)), oracle_run(orc, pb, ic, 2 * k + 1), "12 rows")


@pytest.mark.parametrize("prec", [S.F64, S.REF32, S.C32, S.C32K])
@pytest.mark.parametrize("shape,k", [((2049, 3), 4), ((4321, 4), 1), ((4001, 5), 2), ((6017, 3), 4), ((9000, 3), 3),
                                     ((9300, 3), 3), ((32001, 2), 4)])
def test_heights_of_long_domains(orc, prec, shape, k):
    """Many tiles of a few columns: the taller tiles, with a last one of few rows."""
    pb = S.problem(2, 1, *shape, precision=prec, lx=1.0, ly=shape[1] / shape[0])
    ic = icgen.random_2d(*shape, 6 + k, block=5)
    banner("long", prec, shape, k)
    assert_same(pb, gpu_run(pb, ic, k + 1, (1, k, 4, 0)), oracle_run(orc, pb, ic, k + 1), "long domains")
