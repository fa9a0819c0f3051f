"""GPU: the reference multigrid's sweep kernels -- sweep counts other than four, which
the tile kernels do not take, and a finest grid beyond them -- with periodic images and
variable coefficients: FP64 solves equal to the oracle bit for bit. The coarse levels that
fit one workgroup run there with any count.
"""
import pytest

import test_gpu_rg_tile as tile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,levels,sweeps", [("periodic", (48, 20, 28), 4, 3), ("two_phase", (48, 20, 28), 4, 2),
                                                  ("two_phase", (64, 32, 32), 2, 1), ("periodic", (40, 48, 32), 3, 5),
                                                  ("outlet", (40, 48, 32), 3, 3), ("periodic", (64, 64, 48), 4, 4),
                                                  ("two_phase", (96, 48, 32), 3, 4)])
def test_rg_sweeps(hip, oracle_mod, kind, n, levels, sweeps):
    tile.test_rg_tile(hip, oracle_mod, kind, n, levels, sweeps)
