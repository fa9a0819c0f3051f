"""GPU: the tile kernels of the small multigrid levels (k_mg_down, k_mg_up).

One V-cycle (the stationary iteration stopped after one: dp = M b) on boxes
whose levels are smaller than a tile and its halo (periodic images of images),
end in partial tiles, or have several of them: FP64 equal to the oracle, FP32
and BF16 against the GPU FP64 one. The mixed forms are only close (rounding of
some twenty stages of 2^-24 and 2^-9 each, amplified little by a smoother), but
a wrong neighbour, colour or weight changes M b by O(1).
"""
import numpy as np
import pytest

from mydemcfd_amd import _abi, cases

pytestmark = pytest.mark.gpu

CASES = [("periodic", (4, 4, 4), 2), ("periodic", (8, 4, 12), 2), ("periodic", (20, 12, 28), 2),
         ("periodic", (40, 24, 56), 3), ("cavity", (4, 6, 8), 2), ("cavity", (20, 12, 28), 2),
         ("cavity", (64, 32, 16), 3), ("two_phase", (4, 6, 8), 2), ("two_phase", (18, 16, 14), 2),
         ("two_phase", (40, 24, 56), 3), ("outlet", (20, 12, 28), 2), ("outlet", (32, 40, 16), 3)]


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


def _solve(ctx, kind, levels, precision, seed):
    rng = np.random.default_rng(seed)
    for f in ("ustar", "vstar", "wstar"):
        ctx.upload(f, 0.1 * rng.standard_normal(ctx.shape(f)))
    if kind == "two_phase":
        ctx.upload("alpha", rng.uniform(0.0, 1.0, ctx.shape("alpha")))
    ctx.update_properties(True)
    ctx.pressure_solve(1e-3, precond="mg", mg_levels=levels, precision=precision, stationary=1, tol=0.0, max_iter=1)
    return ctx.download("dp")


@pytest.mark.parametrize("kind,n,levels", CASES)
def test_tile_vcycle(hip, oracle_mod, kind, n, levels):
    print(f"case: tile V-cycle {kind} {n} x{levels}", flush=True)
    ref = _solve(oracle_mod.OracleContext(**_desc(kind, n)), kind, levels, "fp64", 11)
    out = _solve(hip.SMACContext(**_desc(kind, n)), kind, levels, "fp64", 11)
    scale = np.max(np.abs(ref))
    assert scale > 0.0 and np.array_equal(out, ref), float(np.max(np.abs(out - ref)) / scale)
    for precision, tol in (("fp32", 1e-5), ("bf16", 0.1)):
        out = _solve(hip.SMACContext(**_desc(kind, n)), kind, levels, precision, 11)
        assert np.max(np.abs(out - ref)) <= tol * scale, (precision, float(np.max(np.abs(out - ref)) / scale))
