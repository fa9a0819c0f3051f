"""GPU: what has ended when a call returns.

* An adjoint step that fails (here: a level count that the grid does not have) leaves
  no copy from the caller's arrays on the stream.
* A pressure solve has ended, also the V-cycle that was queued ahead of the check that
  stopped it.
* Steps whose solver options change the hierarchy or its graph, taken while the last
  step's work is still queued, give the fields of steps that each waited for the one before.
"""
import numpy as np
import pytest

from mydemcfd_amd import _abi, cases

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

F64 = torch.float64


def _idle(ctx):
    return torch.cuda.ExternalStream(ctx.lib.smac_stream(ctx.h)).query()


@pytest.mark.parametrize("vof", [False, True])
def test_failed_adjoint_leaves_nothing_queued(hip, vof):
    n = (160, 160, 160)
    print(f"case: failing adjoint step {n} vof={vof}", flush=True)
    ctx = hip.SMACContext(**(cases.dam_break_desc(n) if vof else cases.cavity_desc(n)))
    # the copies of the whole arrays take longer than the refusal behind them
    vel = [torch.zeros(ctx.shape(f), dtype=F64, device="cuda") for f in "uvw"]
    bar = [torch.zeros_like(t) for t in vel]
    p = torch.zeros(ctx.shape("p"), dtype=F64, device="cuda")
    q = [torch.zeros_like(p) for _ in range(3)]
    torch.cuda.synchronize()
    kw = dict(precond="mg", mg_levels=12)
    for _ in range(2):  # the first call also allocates, which waits for the GPU
        with pytest.raises(_abi.SmacError) as e:
            if vof:
                ctx.adjoint_vof_step(1e-3, 1, 0, q[0].data_ptr(), [t.data_ptr() for t in vel], p.data_ptr(),
                                     q[1].data_ptr(), [t.data_ptr() for t in bar], q[2].data_ptr(), **kw)
            else:
                ctx.adjoint_step(1e-3, [t.data_ptr() for t in vel], [t.data_ptr() for t in bar], p.data_ptr(), **kw)
        assert _idle(ctx)
        assert e.value.status == _abi.SMAC_ERR_INVALID_GRID


@pytest.mark.parametrize("precond,kw", [("mg", dict(tol=0.9)), ("mg", dict(tol=0.0, max_iter=1)),
                                        ("mg", dict(tol=0.9, precision="fp32", flexible=1)),
                                        ("ref_gmg", dict(tol=0.9)), ("jacobi", dict(tol=0.0, max_iter=3))])
def test_pressure_solve_has_ended(hip, precond, kw):
    n = (192, 192, 192)
    print(f"case: end of a solve {precond} {kw}", flush=True)
    ctx = hip.SMACContext(**cases.periodic_desc(n))
    rng = np.random.default_rng(4)
    for f in ("ustar", "vstar", "wstar"):
        ctx.upload(f, rng.standard_normal(ctx.shape(f)))
    for _ in range(2):
        ctx.pressure_solve(1e-3, precond=precond, **kw)
        assert _idle(ctx)
    ctx.upload("ustar", np.full(ctx.shape("ustar"), np.nan))
    with pytest.raises(_abi.SmacError) as e:
        ctx.pressure_solve(1e-3, precond=precond, **kw)
    assert _idle(ctx)
    assert e.value.status == _abi.SMAC_ERR_NAN


def test_options_change_behind_a_queued_vcycle(hip):
    n = (96, 96, 96)
    print(f"case: changing V-cycle options behind queued work {n}", flush=True)
    rng = np.random.default_rng(6)
    fields = {}
    ctxs = [hip.SMACContext(**cases.periodic_desc(n)) for _ in range(2)]
    for f in "uvw":
        fields[f] = rng.standard_normal(ctxs[0].shape(f))
    for c in ctxs:
        for f, a in fields.items():
            c.upload(f, a)
    # a tolerance that the first update meets: the V-cycle behind its check is queued
    forms = [dict(), dict(nu1=1), dict(nu1=1, nu2=1), dict(precision="fp32", flexible=1), dict(mg_levels=6)] * 3
    for kw in forms:
        for wait, c in enumerate(ctxs):
            c.step(1e-4, precond="mg", tol=0.9, **kw)
            if wait:
                c.sync()
    for f in "uvwp":
        assert np.array_equal(ctxs[0].download(f), ctxs[1].download(f)), f
