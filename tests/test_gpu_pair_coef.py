"""GPU: the SpMV of variable coefficients on 256- and 512-cell rows, whose lanes read
the faces of four cells as vectors: x walls, and periodic x, where the last lane's last
face is the row's first; one chunk of cells a half row (256) and two (512); four rows of
a block sharing their y neighbours (ny a multiple of 4) and not. The first SpMV of a
solve and the ones with the direction update, in several PCG iterations: FP64 equal to
the oracle bit for bit. FP32 and BF16 z in the same passes: their solves reach the FP64
solution's residual (|D u| = dt |r|, tests of the row kernels) in as many iterations.
"""
import numpy as np
import pytest

import test_gpu_row_kernels as rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["two_phase", "two_phase_x"])
@pytest.mark.parametrize("n,kw", [((256, 8, 8), dict(precond="mg")), ((512, 8, 8), dict(precond="mg", flexible=1)),
                                  ((256, 6, 5), dict(precond="jacobi")), ((512, 7, 4), dict(precond="jacobi")),
                                  ((512, 4, 4), dict(precond="jacobi", flexible=1))])
def test_pair_spmv_variable(hip, oracle_mod, kind, n, kw):
    print(f"case: variable pair-form SpMV {kind} {n} {kw}", flush=True)
    kw = dict(kw, max_iter=6, tol=1e-12)
    g = hip.SMACContext(**rows._desc(kind, n))
    g.set_profiling(True)
    out, sg = rows._solve(g, kind, **kw)
    assert {"first_spmv", "dir_spmv"} <= set(g.kernel_names())
    ref, so = rows._solve(oracle_mod.OracleContext(**rows._desc(kind, n)), kind, **kw)
    assert sg == so and sg[0] == 6
    assert np.max(np.abs(ref)) > 0.0 and np.array_equal(out, ref), float(np.max(np.abs(out - ref)))


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("n", [(256, 8, 8), (512, 8, 8)])
def test_pair_spmv_variable_mixed(hip, n, precision):
    rows.test_mixed_step(hip, "two_phase_x", n, precision, {}, ("first_spmv", "dir_spmv"))
