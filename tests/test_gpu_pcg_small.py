"""GPU: the PCG passes of small grids (k_pcg_dir, k_pcg_res).

Rows on both sides of what changes with the size: one partial row of lanes and
several, fewer row partials than the 1024 lanes of the canonical tree and more
(where a block takes 16 rows instead of 4), the largest row count, odd rows;
all three preconditioners, plain and flexible, stopped by convergence and by
max_iter (where the last direction update is skipped). FP64 equal to the oracle
bit for bit, since every sum keeps the canonical order.
"""
import numpy as np
import pytest

from mydemcfd_amd import cases

pytestmark = pytest.mark.gpu

CASES = [("jacobi", (5, 3, 2), 0, 9), ("jacobi", (21, 17, 13), 0, 400), ("jacobi", (21, 17, 13), 1, 7),
         ("jacobi", (131, 31, 33), 0, 12), ("jacobi", (130, 32, 32), 1, 12), ("jacobi", (33, 128, 64), 0, 12),
         ("jacobi", (64, 129, 64), 0, 12), ("mg", (20, 12, 28), 0, 400), ("mg", (20, 36, 32), 1, 3),
         ("ref_gmg", (24, 24, 48), 0, 400)]


@pytest.mark.parametrize("two_phase", [False, True])
@pytest.mark.parametrize("precond,n,flexible,max_iter", CASES)
def test_small_pcg(hip, oracle_mod, precond, n, flexible, max_iter, two_phase):
    print(f"case: small PCG {precond} {n} flexible={flexible} two_phase={two_phase}", flush=True)
    size = tuple(v / 16.0 for v in n)
    desc = cases.dam_break_desc(n, length=size, rho=(1.0, 20.0)) if two_phase else dict(cases.cavity_desc(n), size=size)
    rng = np.random.default_rng(3)
    g, o = hip.SMACContext(**desc), oracle_mod.OracleContext(**desc)
    fields = {f: 0.1 * rng.standard_normal(o.shape(f)) for f in ("ustar", "vstar", "wstar")}
    if two_phase:
        fields["alpha"] = rng.uniform(0.0, 1.0, o.shape("alpha"))
    kw = dict(precond=precond, flexible=flexible, max_iter=max_iter, tol=1e-9, check_every=4)
    for c in (g, o):
        for f, a in fields.items():
            c.upload(f, a)
        c.update_properties(True)
    for _ in range(2):
        sg, so = g.pressure_solve(1e-3, **kw), o.pressure_solve(1e-3, **kw)
        assert (sg.iters, sg.converged, sg.rel_res, sg.linf_res_dt) == (so.iters, so.converged, so.rel_res,
                                                                       so.linf_res_dt)
        assert np.array_equal(g.download("dp"), o.download("dp"))
