"""GPU: the transposed predictor (k_predict_vjp) over its tiles: boxes smaller
than a tile, partial tiles along x and y, several blocks of planes along z; walls
of every type that the adjoint takes, periodic axes beside walls; one-phase,
two-phase, after a VoF transport.

The transpose identity <w, J d> = <J^T w, d> of one step against the closest of
the central and the two one-sided second-order differences at 1e-6 (the step is
piecewise smooth), to 1e-6 of the product, forwards solved by 40 stationary
multigrid cycles: the bound and the solves of the other adjoint checks.
"""
import numpy as np
import pytest

from mydemcfd_amd import _abi, cases
from test_gpu_adjoint import TIGHT, TWO_PHASE_RHO, _dot, smooth_field
from test_gpu_adjoint_vof import _one_sided, smooth_alpha

pytestmark = pytest.mark.gpu

DT = 1e-3
TABLE = ((_abi.BC_NOSLIP, 0.0, 0.0, 0.0), (_abi.BC_NOSLIP, 0.2, -0.1, 0.1), (_abi.BC_SLIP, 0.0, 0.0, 0.0),
         (_abi.BC_INFLOW, 0.0, 0.1, 0.05))
KINDS = {"walls": ((0, 0, 0), (0, 3, 1, 2, 2, 0)), "slip_x": ((0, 0, 1), (2, 2, 0, 1, 0, 0)),
         "periodic": ((1, 1, 1), (0, 0, 0, 0, 0, 0))}


@pytest.mark.parametrize("n", [(4, 4, 4), (70, 6, 8), (8, 18, 22)])
@pytest.mark.parametrize("mode,kind", [("one", "walls"), ("one", "slip_x"), ("one", "periodic"), ("two", "walls"),
                                       ("two", "slip_x"), ("vof", "walls"), ("vof", "slip_x")])
def test_predictor_transpose(hip, mode, kind, n):
    import torch

    print(f"case: transposed predictor {mode} {kind} {n}", flush=True)
    per, sides = KINDS[kind]
    length = tuple(v / 8.0 for v in n)
    desc = dict(n=n, size=length, periodic=per, side_bcid=sides, bc_table=TABLE,
                rho=TWO_PHASE_RHO if mode != "one" else (1.0, 1.0), mu=(1e-3, 5e-3))
    ctx = hip.SMACContext(**desc)
    names = ["u", "v", "w", "p"] + (["alpha"] if mode == "vof" else [])
    masks = {f: torch.tensor(cases.state_mask(n, per, "p" if f == "alpha" else f), device="cuda") for f in names}
    rng = np.random.default_rng(31)
    st0 = {f: 0.05 * smooth_field(ctx.shape(f), rng) for f in ("u", "v", "w")}
    st0["p"] = np.zeros(ctx.shape("p"))
    alpha = smooth_alpha(n, length, w=2.0)
    if mode == "vof":
        st0["alpha"] = alpha
    elif mode == "two":
        ctx.upload("alpha", alpha)
    st0 = {f: torch.tensor(st0[f], dtype=torch.float64, device="cuda").contiguous() for f in names}
    opts = ctx.opts(**TIGHT)
    d = {f: torch.tensor(smooth_field(st0[f].shape, rng), device="cuda") * masks[f] for f in names}
    gen = torch.Generator(device="cuda")
    gen.manual_seed(31)
    w = {f: torch.randn(st0[f].shape, generator=gen, device="cuda", dtype=torch.float64) * masks[f] for f in names}
    d["p"] = torch.zeros_like(d["p"])
    w["p"] = torch.zeros_like(w["p"])

    def forward(st):
        torch.cuda.synchronize()
        for f, t in st.items():
            ctx.upload_device(f, t.data_ptr(), t.numel())
        if mode == "vof":
            ctx.update_properties(True)
            ctx.transport_alpha(DT, 2, 0)
        r = ctx.step(DT, opts)
        assert r.rel_res < 1e-12, r.as_dict()
        out = {f: torch.empty_like(t) for f, t in st.items()}
        for f, t in out.items():
            ctx.download_device(f, t.data_ptr(), t.numel())
        torch.cuda.synchronize()
        return out

    base = forward(st0)

    def f(e):
        out = forward({k: st0[k] + e * d[k] for k in st0})
        return _dot(w, {k: out[k] - base[k] for k in out}, masks)

    g = {k: t.clone() for k, t in w.items()}
    torch.cuda.synchronize()
    un, gu = [st0[k].data_ptr() for k in ("u", "v", "w")], [g[k].data_ptr() for k in ("u", "v", "w")]
    if mode == "vof":
        s = ctx.adjoint_vof_step(DT, 2, 0, st0["alpha"].data_ptr(), un, st0["p"].data_ptr(), g["alpha"].data_ptr(),
                                 gu, g["p"].data_ptr(), opts)
    else:
        s = ctx.adjoint_step(DT, un, gu, g["p"].data_ptr(), opts)
    assert s.rel_res < 1e-12, s.as_dict()
    torch.cuda.synchronize()
    for k in g:  # entries that are not state are zero on return
        assert float(g[k][~masks[k]].abs().max()) == 0.0, k
    rel = _one_sided(f, _dot(g, d, masks))
    print(f"  relative distances: one-sided {rel[0]:.2e} (+) {rel[1]:.2e} (-), central {rel[2]:.2e}", flush=True)
    assert min(rel) <= 1e-6, rel
