"""GPU: the dense coarsest inverse at the limits where the back substitution's LDS size
changes (128, 256, 512 and 1024 cells), at each limit and next past it, with a partial last
block of columns: equal to the oracle bit for bit.
"""
import pytest

import test_gpu_coarsest as base

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(8, 8, 2), (13, 5, 2), (16, 8, 2), (19, 7, 2), (16, 16, 2), (19, 3, 9), (32, 16, 2)])
def test_coarsest_limits(hip, oracle_mod, n):
    base.test_coarsest_inverse(hip, oracle_mod, "two_phase", n)
