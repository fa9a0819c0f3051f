"""GPU: variable face coefficients read as vectors (level_coefs): the two- and
four-rows-per-wave half sweeps and the vector residual of the mixed V-cycles, with
one sweep before and after (levels of two sweeps of this size take the tile
kernels), walls and periodic x (the last face is the first).

One V-cycle (the stationary iteration stopped after one iteration: dp = M b)
against the FP64 form's, which the oracle fixes: FP32 and BF16 storage change M b
by ~1e-6 and ~1e-2 of its maximum, a wrong face by O(1) at its cells.
"""
import numpy as np
import pytest

from conftest import rel_err_mod_mean
from mydemcfd_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("perx", [0, 1])
@pytest.mark.parametrize("n,precision,tol", [((128, 16, 8), "fp32", 5e-6), ((256, 8, 8), "fp32", 5e-6),
                                             ((512, 8, 8), "fp32", 5e-6), ((256, 16, 8), "bf16", 5e-2),
                                             ((512, 8, 8), "bf16", 5e-2)])
def test_variable_vcycle(hip, n, precision, tol, perx):
    print(f"case: one {precision} V-cycle, variable coefficients, {n}, periodic x {perx}", flush=True)
    desc = cases.dam_break_desc(n, length=tuple(v / 32.0 for v in n), rho=(1.0, 20.0), mu=(1e-3, 5e-3))
    desc["periodic"] = (perx, 0, 0)
    out = []
    for p in ("fp64", precision):
        ctx = hip.SMACContext(**desc)
        rng = np.random.default_rng(8)
        ctx.upload("alpha", rng.uniform(0.0, 1.0, ctx.shape("alpha")))
        ctx.update_properties(True)
        for f in ("ustar", "vstar", "wstar"):
            ctx.upload(f, rng.standard_normal(ctx.shape(f)))
        st = ctx.pressure_solve(1e-3, precond="mg", precision=p, stationary=1, tol=0.0, max_iter=1, nu1=1, nu2=1,
                                flexible=int(p != "fp64"))
        assert st.iters == 1
        out.append(ctx.download("dp"))
    err = rel_err_mod_mean(out[1], out[0], n)
    print(f"  max|M_{precision} b - M_fp64 b| / max|M_fp64 b| = {err:.3e}", flush=True)
    assert err <= tol
