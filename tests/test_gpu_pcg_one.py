"""GPU: the Jacobi PCG in one workgroup (k_pcg_one).

Rows of 16, 32 and 64 lanes with odd and full lengths, one row slot and several,
grids on both sides of the largest it takes (the two passes beyond); walls, periodic
images, two phases; both stop rules, plain and flexible, stopped by convergence, by
max_iter between two checks, and after more iterations than one launch makes. FP64
equal to the oracle bit for bit, since every sum keeps the canonical order.
"""
import numpy as np
import pytest

from mydemcfd_amd import cases

pytestmark = pytest.mark.gpu

CASES = [("cavity", (2, 3, 2), 0, 50), ("cavity", (9, 8, 8), 1, 400), ("cavity", (32, 16, 4), 0, 400),
         ("periodic", (6, 10, 12), 0, 400), ("cavity", (21, 17, 13), 0, 2000), ("two_phase", (21, 17, 3), 1, 6),
         ("two_phase", (32, 8, 8), 0, 700), ("cavity", (32, 16, 16), 0, 11), ("cavity", (32, 32, 16), 0, 11), ("periodic", (33, 9, 3), 1, 9),
         ("two_phase", (64, 8, 4), 0, 11), ("two_phase", (64, 16, 16), 0, 11), ("cavity", (63, 5, 6), 0, 400), ("cavity", (65, 4, 4), 0, 13),
         ("two_phase", (127, 4, 4), 1, 8), ("cavity", (127, 8, 8), 1, 8), ("periodic", (128, 16, 8), 0, 9), ("cavity", (128, 11, 11), 0, 9)]


def _desc(kind, n):
    size = tuple(v / 16.0 for v in n)
    if kind == "two_phase":
        return cases.dam_break_desc(n, length=size, rho=(1.0, 20.0))
    return dict(cases.periodic_desc(n) if kind == "periodic" else cases.cavity_desc(n), size=size)


@pytest.mark.parametrize("rule", ["rel_l2", "ref_linf_dt"])
@pytest.mark.parametrize("kind,n,flexible,max_iter", CASES)
def test_pcg_one(hip, oracle_mod, kind, n, flexible, max_iter, rule):
    print(f"case: one-workgroup PCG {kind} {n} flexible={flexible} {rule}", flush=True)
    if kind == "periodic":
        n = tuple(max(v, 4) for v in n)
    rng = np.random.default_rng(3)
    g, o = hip.SMACContext(**_desc(kind, n)), oracle_mod.OracleContext(**_desc(kind, n))
    fields = {f: 0.1 * rng.standard_normal(o.shape(f)) for f in ("ustar", "vstar", "wstar")}
    if kind == "two_phase":
        fields["alpha"] = rng.uniform(0.0, 1.0, o.shape("alpha"))
    kw = dict(precond="jacobi", flexible=flexible, max_iter=max_iter, tol=1e-9, check_every=4, stop_rule=rule)
    for c in (g, o):
        for f, a in fields.items():
            c.upload(f, a)
        c.update_properties(True)
    for _ in range(2):
        sg, so = g.pressure_solve(1e-3, **kw), o.pressure_solve(1e-3, **kw)
        assert (sg.iters, sg.converged, sg.rel_res, sg.linf_res_dt) == (so.iters, so.converged, so.rel_res,
                                                                       so.linf_res_dt)
        assert np.array_equal(g.download("dp"), o.download("dp"))
