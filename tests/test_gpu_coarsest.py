"""GPU: the dense inverse of the coarsest multigrid level (k_pinv_assemble,
k_pinv_panel, k_pinv_back) against the oracle's sequential loops.

mg_levels = 1 makes the whole box the coarsest level, so one V-cycle is the
product with the inverse alone. Sizes: below, at and just past one 32-column
panel, a partial last panel, and both sides of the limits where the back
substitution changes its columns per wave (256, 512 cells) up to the largest
(1024). Every sum has the sequential order, so the solution is the oracle's bit
for bit.
"""
import numpy as np
import pytest

from mydemcfd_amd import _abi, cases

pytestmark = pytest.mark.gpu

BOXES = [(2, 2, 2), (4, 4, 2), (3, 11, 2), (4, 4, 4), (13, 5, 2), (9, 9, 3), (16, 4, 4), (43, 3, 2), (8, 8, 8),
         (43, 6, 2), (10, 10, 10), (16, 8, 8)]


def _desc(kind, n):
    size = tuple(v / 8.0 for v in n)
    if kind == "periodic":
        return cases.periodic_desc(n, length=1.0)
    if kind == "outlet":
        table = ((_abi.BC_NOSLIP, 0.0, 0.0, 0.0), (_abi.BC_INFLOW, 0.5, 0.0, 0.0), (_abi.BC_OUTLET, 0.0, 0.0, 0.0))
        return dict(n=n, size=size, side_bcid=(1, 2, 0, 0, 0, 0), bc_table=table, mu=(0.01, 0.01))
    return cases.dam_break_desc(n, length=size, rho=(1.0, 1000.0))


@pytest.mark.parametrize("kind,n", [("two_phase", n) for n in BOXES] +
                         [("outlet", (9, 9, 3)), ("outlet", (10, 10, 10)), ("periodic", (4, 4, 4)),
                          ("periodic", (8, 8, 6))])
def test_coarsest_inverse(hip, oracle_mod, kind, n):
    print(f"case: coarsest inverse {kind} {n}", flush=True)
    rng = np.random.default_rng(7)
    g, o = hip.SMACContext(**_desc(kind, n)), oracle_mod.OracleContext(**_desc(kind, n))
    fields = {f: 0.1 * rng.standard_normal(o.shape(f)) for f in ("ustar", "vstar", "wstar")}
    if kind == "two_phase":
        fields["alpha"] = rng.uniform(0.0, 1.0, o.shape("alpha"))
    kw = dict(precond="mg", mg_levels=1, stationary=1, tol=0.0, max_iter=1)
    for c in (g, o):
        for f, a in fields.items():
            c.upload(f, a)
        c.update_properties(True)
    for _ in range(2):  # the second solve reuses the inverse
        g.pressure_solve(1e-3, **kw)
        o.pressure_solve(1e-3, **kw)
        a, b = g.download("dp"), o.download("dp")
        assert np.all(np.isfinite(b)) and np.max(np.abs(b)) > 0.0
        assert np.array_equal(a, b), float(np.max(np.abs(a - b)))
