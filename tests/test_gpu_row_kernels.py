"""GPU: the row kernels of the PCG and of the V-cycle, on grids that reach them.

Levels of up to 2^18 cells with two sweeps before and after take the tile kernels,
and grids of up to 8192 rows the two-pass PCG, so these run one sweep on either side
(which the tiles do not take) or a grid beyond the limits; the names of the profile
say which kernels ran.

* FP64: the vector smoother, the two- and four-rows-per-wave ones, the half sweep that
  also forms the PCG's dots, the vector residual, restriction and prolongation, the
  one- and three-chunk passes of the PCG and the general ones: equal to the oracle bit
  for bit, uniform and variable coefficients, walls and periodic images.
* FP32 and BF16: one step to 1e-9. With b = -(1/dt) D u* and the solver's residual r the
  corrected velocity has D u = -dt r whatever the preconditioner, so |D u| / |D u*| is
  the reported residual (up to the drift of the recursive one, 5 % of it or rounding).
  A V-cycle that is wrong costs iterations: at most 6 more than FP64, half as many again
  in BF16 (8-bit mantissa).
"""
import numpy as np
import pytest

from mydemcfd_amd import cases

pytestmark = pytest.mark.gpu


def _desc(kind, n):
    size = tuple(v / 32.0 for v in n)
    if kind == "two_phase":
        return cases.dam_break_desc(n, length=size, rho=(1.0, 20.0), mu=(1e-3, 5e-3))
    if kind == "two_phase_x":  # x periodic
        return dict(_desc("two_phase", n), periodic=(1, 0, 0))
    return dict(cases.periodic_desc(n) if kind == "periodic" else cases.cavity_desc(n), size=size)


def _solve(ctx, kind, **kw):
    rng = np.random.default_rng(17)
    for f in ("ustar", "vstar", "wstar"):
        ctx.upload(f, 0.1 * rng.standard_normal(ctx.shape(f)))
    if kind.startswith("two_phase"):
        ctx.upload("alpha", rng.uniform(0.0, 1.0, ctx.shape("alpha")))
    ctx.update_properties(True)
    st = ctx.pressure_solve(1e-3, **kw)
    return ctx.download("dp"), (st.iters, st.converged, st.rel_res)


ONE = dict(precond="mg", nu1=1, nu2=1, max_iter=5, tol=1e-12)
TWO = dict(precond="mg", max_iter=3, tol=1e-12)
JAC = dict(precond="jacobi", max_iter=4, tol=1e-12)
SMOOTH = ("mg_rbgs_l0", "mg_restrict_l0", "mg_prolong_l0")
# kind, box, options, names of kernels that ran (None: of those of SMOOTH)
FP64 = [
    # one sweep: the vector form with dots (512), two rows a wave with dots (128), the
    # vector form (256), the general one (384), plain and flexible
    ("periodic", (512, 8, 8), ONE, SMOOTH + ("mg_rbgs_dot",)),
    ("periodic", (512, 8, 8), dict(ONE, flexible=1), SMOOTH + ("mg_rbgs_dot",)),
    ("periodic", (128, 8, 8), ONE, SMOOTH + ("mg_rbgs_dot",)),
    ("periodic", (128, 8, 8), dict(ONE, flexible=1), SMOOTH + ("mg_rbgs_dot",)),
    ("periodic", (256, 16, 8), ONE, SMOOTH),
    ("periodic", (384, 8, 8), ONE, SMOOTH),
    ("cavity", (512, 8, 8), ONE, SMOOTH + ("mg_rbgs_dot",)),
    ("cavity", (128, 16, 12), ONE, SMOOTH),
    ("cavity", (256, 8, 8), dict(ONE, nu1=1, nu2=2), SMOOTH),
    ("cavity", (64, 32, 24), dict(ONE, nu1=2, nu2=1), SMOOTH),
    ("two_phase", (128, 8, 12), ONE, SMOOTH),
    ("two_phase", (256, 8, 8), ONE, SMOOTH),
    # four rows a wave
    ("periodic", (64, 32, 16), ONE, SMOOTH),
    ("two_phase", (64, 16, 8), ONE, SMOOTH),
    # two sweeps on levels beyond the tiles, tiles below them
    ("periodic", (512, 32, 32), TWO, SMOOTH + ("mg_rbgs_dot",)),
    ("cavity", (64, 128, 64), TWO, SMOOTH),
    ("two_phase", (64, 64, 64), TWO, SMOOTH),
    ("two_phase_x", (128, 64, 32), TWO, SMOOTH),
    # the PCG's passes beyond the two-pass form: one and three chunks a row, rows of
    # any length; beyond 2^22 cells with the direction update in a pass of its own
    ("periodic", (384, 64, 32), TWO, SMOOTH + ("update_zs",)),
    ("cavity", (128, 96, 96), dict(JAC, flexible=1), ("update", "dot2", "jacobi", "dir_spmv")),
    ("two_phase", (90, 94, 90), JAC, ("update", "dot2", "jacobi", "dir_spmv")),
    ("periodic", (384, 112, 100), JAC, ("update", "dot2", "jacobi", "xpay")),
    ("cavity", (200, 150, 145), dict(JAC, flexible=1), ("update", "dot2", "jacobi", "xpay")),
]


@pytest.mark.parametrize("kind,n,kw,names", FP64)
def test_fp64_equals_oracle(hip, oracle_mod, kind, n, kw, names):
    print(f"case: row kernels {kind} {n} {kw}", flush=True)
    g = hip.SMACContext(**_desc(kind, n))
    g.set_profiling(True)
    out, sg = _solve(g, kind, **kw)
    ran = g.kernel_names()
    assert set(names) <= set(ran) and "mg_down_l0" not in ran and "pcg_one" not in ran, ran
    ref, so = _solve(oracle_mod.OracleContext(**_desc(kind, n)), kind, **kw)
    scale = np.max(np.abs(ref))
    assert sg == so
    assert scale > 0.0 and np.array_equal(out, ref), float(np.max(np.abs(out - ref)) / scale)


def _div(ctx, names):
    nx, ny, nz = ctx.n
    u, v, w = (ctx.download(f) for f in names)
    h = [s / m for s, m in zip(ctx.size, ctx.n)]
    z, y, x = slice(1, nz + 1), slice(1, ny + 1), slice(1, nx + 1)
    d = (u[z, y, 2:nx + 2] - u[z, y, x]) / h[0]
    d += (v[z, 2:ny + 2, x] - v[z, y, x]) / h[1]
    d += (w[2:nz + 2, y, x] - w[z, y, x]) / h[2]
    return float(np.linalg.norm(d))


def _step(ctx, kind, **kw):
    rng = np.random.default_rng(23)
    for a, f in enumerate("uvw"):
        x = 0.1 * rng.standard_normal(ctx.shape(f))
        if not ctx.periodic[a]:  # no flow through the walls
            np.moveaxis(x, 2 - a, 0)[[1, ctx.n[a] + 1]] = 0.0
        ctx.upload(f, x)
    if kind.startswith("two_phase"):
        ctx.upload("alpha", rng.uniform(0.0, 1.0, ctx.shape("alpha")))
        ctx.update_properties(True)
    return ctx.step(1e-3, precond="mg", tol=1e-9, max_iter=400, **kw)


V1 = dict(nu1=1, nu2=1)
MIXED = [
    # four rows a wave, two rows a wave (with dots on uniform grids), the vector form
    ("periodic", (128, 16, 8), "fp32", V1, ("mg_rbgs_l0",)),
    ("two_phase", (128, 16, 8), "fp32", V1, ("mg_rbgs_l0",)),
    ("periodic", (256, 16, 8), "fp32", V1, ("mg_rbgs_l0", "mg_rbgs_dot", "update_zs")),
    ("cavity", (256, 8, 8), "fp32", V1, ("mg_rbgs_l0", "mg_rbgs_dot")),
    ("periodic", (512, 8, 8), "fp32", V1, ("mg_rbgs_l0", "mg_rbgs_dot")),
    ("periodic", (256, 32, 8), "bf16", V1, ("mg_rbgs_l0", "update_zs")),
    ("two_phase", (256, 16, 8), "bf16", V1, ("mg_rbgs_l0",)),
    ("cavity", (512, 8, 8), "bf16", V1, ("mg_rbgs_l0", "mg_rbgs_dot")),
    # two sweeps, the residual update with the next half sweep on it, and the direction
    # pass for rows of any length, beyond the tiles and the two-pass form
    ("periodic", (128, 96, 96), "fp32", {}, ("mg_rbgs_l0", "update_zs", "dir_spmv")),
    ("periodic", (128, 96, 96), "bf16", {}, ("mg_rbgs_l0", "update_zs", "dir_spmv")),
    ("cavity", (24, 96, 96), "fp32", {}, ("dir_spmv",)),
    ("two_phase", (24, 96, 96), "bf16", {}, ("dir_spmv",)),
]


@pytest.mark.parametrize("kind,n,precision,kw,names", MIXED)
def test_mixed_step(hip, kind, n, precision, kw, names):
    print(f"case: row kernels {precision} {kind} {n} {kw}", flush=True)
    ref = _step(hip.SMACContext(**_desc(kind, n)), kind, **kw)
    ctx = hip.SMACContext(**_desc(kind, n))
    ctx.set_profiling(True)
    st = _step(ctx, kind, precision=precision, flexible=1, **kw)
    ran = ctx.kernel_names()
    assert set(names) <= set(ran), ran
    ratio = _div(ctx, ("u", "v", "w")) / _div(ctx, ("ustar", "vstar", "wstar"))
    print(f"  iters {st.iters} ({ref.iters}), rel_res {st.rel_res:.3e}, |D u|/|D u*| {ratio:.3e}", flush=True)
    assert st.converged and ref.converged and st.rel_res < 1e-9
    assert ratio <= 1.05 * st.rel_res + 1e-12
    assert st.iters <= ref.iters + (max(6, ref.iters // 2) if precision == "bf16" else 6)
