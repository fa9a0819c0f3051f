"""GPU: the reference multigrid's small levels (k_rg_down, k_rg_up, k_rg_tail).

Levels in one workgroup with one and with four cells a thread, tiles with
partial ends and several blocks, axes that stop coarsening before others, walls,
outlets and periodic images, four sweeps (the tile form) and others (the sweep
kernels): FP64 solves equal to the oracle bit for bit.
"""
import numpy as np
import pytest

from mydemcfd_amd import _abi, cases

pytestmark = pytest.mark.gpu

CASES = [("cavity", (24, 24, 24), 4, 4), ("periodic", (24, 24, 24), 4, 4), ("periodic", (48, 20, 28), 4, 4),
         ("two_phase", (48, 20, 28), 4, 4), ("two_phase", (64, 32, 32), 4, 4), ("outlet", (40, 48, 32), 3, 4),
         ("two_phase", (32, 40, 24), 2, 4), ("cavity", (24, 24, 48), 4, 2)]


def _desc(kind, n):
    size = tuple(v / 16.0 for v in n)
    if kind == "periodic":
        return dict(cases.periodic_desc(n, length=1.0), size=size)
    if kind == "cavity":
        return dict(cases.cavity_desc(n, re=100.0), size=size)
    if kind == "outlet":
        table = ((_abi.BC_NOSLIP, 0.0, 0.0, 0.0), (_abi.BC_INFLOW, 0.5, 0.0, 0.0), (_abi.BC_OUTLET, 0.0, 0.0, 0.0))
        return dict(n=n, size=size, side_bcid=(1, 2, 0, 0, 0, 0), bc_table=table, mu=(0.01, 0.01))
    return cases.dam_break_desc(n, length=size, rho=(1.0, 50.0))


@pytest.mark.parametrize("kind,n,levels,sweeps", CASES)
def test_rg_tile(hip, oracle_mod, kind, n, levels, sweeps):
    print(f"case: reference multigrid {kind} {n} x{levels}, {sweeps} sweeps", flush=True)
    rng = np.random.default_rng(5)
    g, o = hip.SMACContext(**_desc(kind, n)), oracle_mod.OracleContext(**_desc(kind, n))
    kw = dict(precond="ref_gmg", mg_levels=levels, ref_sweeps=sweeps, tol=0.0, max_iter=3)
    for _ in range(2):  # the second solve: new coefficients on the same levels
        fields = {f: 0.1 * rng.standard_normal(o.shape(f)) for f in ("ustar", "vstar", "wstar")}
        if kind == "two_phase":
            fields["alpha"] = rng.uniform(0.0, 1.0, o.shape("alpha"))
        for c in (g, o):
            for f, a in fields.items():
                c.upload(f, a)
            c.update_properties(True)
            c.pressure_solve(1e-3, **kw)
        a, b = g.download("dp"), o.download("dp")
        assert np.max(np.abs(b)) > 0.0 and np.array_equal(a, b), float(np.max(np.abs(a - b)))
