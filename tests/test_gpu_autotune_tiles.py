"""GPU: where the 2D first-order steps run on register tiles, whose height and block do not depend
on the launch shape, the autotuner tries each number of steps per launch once per graph length: the
recorded shape has the library's rows (1) and 4 waves per block."""
import pytest

import icgen
import shll_amd as S
from test_gpu_parity import banner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [S.F64, S.REF32, S.C32, S.C32K])
def test_equal_kernels_are_one_candidate(prec, tmp_path, monkeypatch):
    for i, shape in enumerate(((100, 130), (200, 70), (260, 260), (64, 300))):
        monkeypatch.setenv("SHLL_TUNE_CACHE", str(tmp_path / ("tune%d.txt" % i)))
        pb = S.problem(2, 1, *shape, precision=prec, lx=1.0, ly=shape[1] / shape[0])
        banner("autotune tiles", prec, shape)
        with S.Solver(pb, icgen.random_2d(*shape, 8, block=5)) as s:
            s.autotune(48)
            rows, k, waves, graph = s.get_launch()
        assert (rows, waves) == (1, 4) and k in (1, 2, 3, 4, 8), (rows, k, waves, graph)
