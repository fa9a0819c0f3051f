"""GPU: the direction update inside the SpMV for rows of any length (k_pcg_dir
without the sums), on grids beyond the two-pass iteration's row count: rows of less
than a wave, of one and of more; walls, periodic images, two phases; Jacobi and
multigrid, the stationary iteration (alpha = 1, beta = 0), stopped by convergence
and by max_iter (where the last direction update is k_xpay's). FP64 equal to the
oracle bit for bit.
"""
import numpy as np
import pytest

from mydemcfd_amd import cases

pytestmark = pytest.mark.gpu

CASES = [("jacobi", "cavity", (9, 95, 87), dict(max_iter=9)), ("jacobi", "two_phase", (70, 91, 91), dict(max_iter=6)),
         ("mg", "periodic", (24, 96, 96), dict(max_iter=400)), ("mg", "two_phase", (24, 96, 96), dict(max_iter=5)),
         ("mg", "periodic", (16, 96, 96), dict(max_iter=4, tol=0.0, stationary=1)),
         ("jacobi", "periodic", (130, 92, 90), dict(max_iter=5, flexible=1))]


@pytest.mark.parametrize("precond,kind,n,kw", CASES)
def test_dir_rows(hip, oracle_mod, precond, kind, n, kw):
    print(f"case: direction in the SpMV {precond} {kind} {n} {kw}", flush=True)
    size = tuple(v / 16.0 for v in n)
    if kind == "two_phase":
        desc = cases.dam_break_desc(n, length=size, rho=(1.0, 20.0))
    else:
        desc = dict(cases.periodic_desc(n) if kind == "periodic" else cases.cavity_desc(n), size=size)
    rng = np.random.default_rng(3)
    g, o = hip.SMACContext(**desc), oracle_mod.OracleContext(**desc)
    fields = {f: 0.1 * rng.standard_normal(o.shape(f)) for f in ("ustar", "vstar", "wstar")}
    if kind == "two_phase":
        fields["alpha"] = rng.uniform(0.0, 1.0, o.shape("alpha"))
    kw = dict(dict(precond=precond, tol=1e-9, check_every=2), **kw)
    for c in (g, o):
        for f, a in fields.items():
            c.upload(f, a)
        c.update_properties(True)
    sg, so = g.pressure_solve(1e-3, **kw), o.pressure_solve(1e-3, **kw)
    assert (sg.iters, sg.converged, sg.rel_res) == (so.iters, so.converged, so.rel_res)
    assert np.array_equal(g.download("dp"), o.download("dp"))
