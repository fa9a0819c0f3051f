"""Timed cases of the SMAC step: what programs on this library call every time step.

A case names a loop (kind), a box (nx, ny, nz interior cells), a pressure
solver (precond) and the storage of its V-cycle (precision):

  step         smac_step of a one-phase flow: a periodic box (Taylor-Green plus
               a random solenoidal field), a lid-driven cavity, or a channel
               from an inflow to an outlet side
  vof_loop     the two-phase loop step: VoF transport of alpha, then smac_step
  config_loop  the reference's driver loop: CFL numbers, VoF transport, step,
               ghost update (reference multigrid, max-norm stop rule)
  two_way      the coupled CFD-DEM loop step: volume fractions and impulses in,
               Poisson coefficients, two-way predictor, solve, correction
  rollout      nsteps steps through torch.autograd, forward and backward
  vof_rollout  the same for the VoF loop

The stepping kinds advance the state in place in tensors bound to the context;
the rollouts map input tensors to output tensors and gradients.
"""
import math

import torch

import mydemcfd_amd
from mydemcfd_amd import _abi, autograd

F64 = torch.float64
TWO_PI = 2.0 * math.pi


def _case(name, kind, n, precond="mg", precision="fp64", flow="", iters=8, **kw):
    c = dict(name=name, kind=kind, flow=flow, nx=n[0], ny=n[1], nz=n[2], precond=precond, precision=precision,
             iters=iters)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: a ragged box of a few thousand cells, which only
        # Jacobi-PCG takes: launches and host latency
        _case("cavity_21x17x13_jacobi", "step", (21, 17, 13), "jacobi", flow="cavity", iters=60),
        # the 64^3 cavity with Jacobi-PCG: hundreds of small iterations per step
        _case("cavity_64_jacobi", "step", (64, 64, 64), "jacobi", flow="cavity", iters=200),
        # the reference's driver loop as its JSON configuration sets it up
        # (dam break, reference multigrid), at twice the sample's resolution
        _case("config_loop_64x32x32", "config_loop", (64, 32, 32), "ref_gmg", flow="dam", iters=24),
        # a mid-size periodic box in the narrowest storage
        _case("tg_128_bf16", "step", (128, 128, 128), precision="bf16", flow="tg", iters=8),
        # the 256^3 Taylor-Green run in full double precision
        _case("tg_256_fp64", "step", (256, 256, 256), flow="tg", iters=7),
        # the 512^3 headline step, mixed FP32
        _case("tg_512_fp32", "step", (512, 512, 512), precision="fp32", flow="tg", iters=8),
        # the 256x128x128 dam break, 1000:1, mixed FP32, two VoF substeps
        _case("dam_256x128x128_fp32", "vof_loop", (256, 128, 128), precision="fp32", flow="dam", iters=13),
        # a small dam break on a box that is no power of two, FP64
        _case("dam_96x48x80_fp64", "vof_loop", (96, 48, 80), flow="dam", iters=13),
        # inflow to outlet: Dirichlet outlet faces, coefficients in arrays
        _case("channel_128x64x64_fp32", "step", (128, 64, 64), precision="fp32", flow="channel", iters=10),
        # the coupled loop's step on a walled box
        _case("two_way_80x48x64_fp64", "two_way", (80, 48, 64), flow="cavity", iters=11),
        # gradient of a periodic rollout (the 128^3 gradient configuration)
        _case("rollout_128_fp32", "rollout", (128, 128, 128), precision="fp32", flow="tg", iters=9, nsteps=2),
        # gradient through the VoF loop (alpha-dependent operator, transport)
        _case("vof_rollout_128x64x64_fp32", "vof_rollout", (128, 64, 64), precision="fp32", flow="dam", iters=13,
              nsteps=1),
    ]


def _round(x, m):
    return max(m, int(round(x / m)) * m)


def _pick(rng, lo, hi, sizes):
    """One of `sizes`, the nearest to a point spread over the logarithm of [lo, hi]."""
    t = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(sizes, key=lambda s: abs(math.log(s / t)))


# sizes m 2^k the multigrid halves down to at most 10 cells per axis
MG_SIZES = [24, 28, 32, 36, 40, 48, 56, 64, 72, 80, 96, 112, 128, 144, 160, 192, 224, 256, 288, 320, 384]


def draw(rng):
    kind = rng.choice(["jacobi", "tg", "tg", "cavity", "dam", "dam", "config", "channel", "two_way", "rollout",
                       "vof_rollout"])
    prec = rng.choice(["fp64", "fp32", "fp32", "bf16"])
    mg2 = [s for s in MG_SIZES if s % 8 == 0]
    if kind == "jacobi":  # any size, odd ones included
        n = tuple(int(round(math.exp(rng.uniform(math.log(9), math.log(70))))) for _ in range(3))
        return _drop(_case("", "step", n, "jacobi", flow="cavity", iters=3 * max(n)))
    if kind == "tg":
        m = _pick(rng, 32, 384, MG_SIZES)
        return _drop(_case("", "step", (m, m, m), precision=prec, flow="tg", iters=8))
    if kind == "cavity":
        n = tuple(_pick(rng, 32, 192, [s for s in mg2 if s % 16 == 0]) for _ in range(3))
        n = _levels(n)
        return _drop(_case("", "step", n, precision=prec, flow="cavity", iters=11))
    if kind in ("dam", "vof_rollout"):
        top = 112 if kind == "dam" else 64
        m = math.exp(rng.uniform(math.log(16), math.log(top)))
        n = _levels(tuple(_round(f * m * rng.uniform(0.85, 1.15), 8) for f in (2, 1, 1)))
        if kind == "dam":
            return _drop(_case("", "vof_loop", n, precision=prec, flow="dam", iters=13))
        return _drop(_case("", "vof_rollout", n, precision="fp32" if prec == "bf16" else prec, flow="dam", iters=13,
                           nsteps=1))
    if kind == "config":
        m = math.exp(rng.uniform(math.log(16), math.log(64)))
        n = tuple(_round(f * m * rng.uniform(0.85, 1.15), 16) for f in (2, 1, 1))
        return _drop(_case("", "config_loop", n, "ref_gmg", flow="dam", iters=24))
    if kind == "channel":
        n = _levels(tuple(_pick(rng, 32, 128, [s for s in mg2 if s % 16 == 0]) for _ in range(3)))
        return _drop(_case("", "step", n, precision=prec, flow="channel", iters=10))
    if kind == "two_way":
        n = _levels(tuple(_pick(rng, 32, 128, [s for s in mg2 if s % 16 == 0]) for _ in range(3)))
        return _drop(_case("", "two_way", n, precision=prec, flow="cavity", iters=11))
    m = _pick(rng, 24, 128, MG_SIZES)
    return _drop(_case("", "rollout", (m, m, m), precision="fp32" if prec == "bf16" else prec, flow="tg", iters=9,
                       nsteps=1 + rng.randrange(3)))


def _drop(c):
    c.pop("name")
    return c


def _levels(n):
    """The box itself if the multigrid can coarsen it to 1024 cells, else the
    nearest cube-like one that it can."""
    q = list(n)
    while q[0] * q[1] * q[2] > 512 and all(v % 2 == 0 and v >= 4 for v in q):
        q = [v // 2 for v in q]
    if q[0] * q[1] * q[2] <= 1024:
        return n
    return tuple(_round(v, 32) for v in n)


# ------------------------------------------------------------------ inputs
def _n(case):
    return case["nx"], case["ny"], case["nz"]


def _opts(ctx, case):
    kw = dict(precond=case["precond"], precision=case["precision"], flexible=0 if case["precision"] == "fp64" else 1,
              tol=1e-8, max_iter=2000)
    if case["kind"] == "config_loop":  # the reference's rule: max|r| dt < tol, checked every 5 iterations
        kw.update(stop_rule="ref_linf_dt", check_every=5)
    else:
        kw.update(stop_rule="rel_l2")
        if case["precond"] == "jacobi":
            kw.update(check_every=10)
    if case["kind"] in ("rollout", "vof_rollout"):
        kw.update(tol=1e-10)
    return ctx.opts(**kw)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _smooth(shape, seed, modes=6, kmax=3):
    """A sum of random cosine waves on the index box `shape`, unit RMS."""
    g = torch.Generator()
    g.manual_seed(int(seed))
    ax = [torch.arange(s, device="cuda", dtype=F64) / s for s in shape]
    out = torch.zeros(shape, device="cuda", dtype=F64)
    for _ in range(modes):
        k = torch.randint(-kmax, kmax + 1, (3,), generator=g).tolist()
        ph = float(torch.rand(1, generator=g)) * TWO_PI
        a = float(torch.randn(1, generator=g))
        arg = (TWO_PI * k[0] * ax[0])[:, None, None] + (TWO_PI * k[1] * ax[1])[None, :, None] + \
            (TWO_PI * k[2] * ax[2])[None, None, :] + ph
        out += a * torch.cos(arg)
    return out / out.square().mean().sqrt().clamp_min(1e-30)


def _tg_interior(n, seed):
    """(u, v, w) on the faces 1..N of a periodic [0, 2 pi)^3 box, (z, y, x):
    Taylor-Green plus 5 % of the kinetic energy in a random-phase field with a
    k^-5/3 spectrum up to k = 32, the curl of a random potential."""
    nx, ny, nz = n
    h = [TWO_PI / m for m in n]
    kmax = min(32, min(n) // 3)
    kx = torch.fft.rfftfreq(nx, d=1.0 / nx, device="cuda", dtype=F64)[None, None, :]
    ky = torch.fft.fftfreq(ny, d=1.0 / ny, device="cuda", dtype=F64)[None, :, None]
    kz = torch.fft.fftfreq(nz, d=1.0 / nz, device="cuda", dtype=F64)[:, None, None]
    k = torch.sqrt(kx * kx + ky * ky + kz * kz)
    amp = torch.where((k >= 1.0) & (k <= kmax), k.clamp_min(1.0) ** ((-5.0 / 3.0 - 4.0) / 2.0), torch.zeros_like(k))
    del k
    g = _gen(seed)
    pot = []
    for _ in range(3):
        ph = torch.rand(amp.shape, generator=g, device="cuda", dtype=F64) * TWO_PI
        mag = torch.randn(amp.shape, generator=g, device="cuda", dtype=F64) * amp
        pot.append(torch.fft.irfftn(torch.polar(mag.abs(), ph), s=(nz, ny, nx), dim=(0, 1, 2)))
    del amp, ph, mag

    def d(a, axis):  # forward difference along x, y or z (0, 1, 2)
        return (torch.roll(a, -1, 2 - axis) - a) / h[axis]

    pu = d(pot[2], 1) - d(pot[1], 2)
    pv = d(pot[0], 2) - d(pot[2], 0)
    pw = d(pot[1], 0) - d(pot[0], 1)
    del pot
    xf = [torch.arange(m, device="cuda", dtype=F64) * s for m, s in zip(n, h)]
    xc = [x + 0.5 * s for x, s in zip(xf, h)]
    u = torch.sin(xf[0])[None, None, :] * torch.cos(xc[1])[None, :, None] * torch.cos(xc[2])[:, None, None]
    v = -torch.cos(xc[0])[None, None, :] * torch.sin(xf[1])[None, :, None] * torch.cos(xc[2])[:, None, None]
    e0 = u.square().mean() + v.square().mean()
    e1 = pu.square().mean() + pv.square().mean() + pw.square().mean()
    s = torch.sqrt(0.05 / 0.95 * e0 / e1)
    return u + s * pu, v + s * pv, s * pw


def _periodic_box(a, shape):
    """Interior values (faces or cells 1..N) with their periodic images, in the reference layout."""
    ix = [(torch.arange(s, device="cuda") - 1) % m for s, m in zip(shape, a.shape)]
    return a.index_select(0, ix[0]).index_select(1, ix[1]).index_select(2, ix[2]).contiguous()


def _walled_velocity(ctx, seed, scale, base=(0.0, 0.0, 0.0)):
    """Smooth velocities that vanish (or hold `base`) on the boundary faces of their own axis."""
    out = {}
    for a, f in enumerate("uvw"):
        shape = ctx.shape(f)
        x = scale * _smooth(shape, 7 * seed + a)
        m = shape[2 - a]
        w = torch.sin(math.pi * (torch.arange(m, device="cuda", dtype=F64) - 1).clamp(0, m - 3) / (m - 3))
        view = [1, 1, 1]
        view[2 - a] = m
        out[f] = (x * w.view(view) + base[a]).contiguous()
    return out


def _desc(case):
    n = _n(case)
    wall = (_abi.BC_NOSLIP, 0.0, 0.0, 0.0)
    if case["flow"] == "tg":
        re = 500.0 if case["kind"] == "rollout" else 1600.0
        return dict(n=n, size=(TWO_PI,) * 3, periodic=(1, 1, 1), bc_table=(wall,), mu=(1 / re, 1 / re))
    if case["flow"] == "cavity":  # unit cell size relative to the longest side; the lid on y-max
        s = max(n)
        return dict(n=n, size=tuple(v / s for v in n), side_bcid=(1, 1, 1, 2, 1, 1),
                    bc_table=(wall, wall, (_abi.BC_NOSLIP, 1.0, 0.0, 0.0)), mu=(0.01, 0.01))
    if case["flow"] == "channel":  # inflow on x-min, outlet on x-max, no-slip y, slip z
        s = max(n)
        return dict(n=n, size=tuple(v / s for v in n), side_bcid=(1, 2, 3, 3, 4, 4),
                    bc_table=(wall, (_abi.BC_INFLOW, 0.5, 0.0, 0.0), (_abi.BC_OUTLET, 0.0, 0.0, 0.0), wall,
                              (_abi.BC_SLIP, 0.0, 0.0, 0.0)), mu=(0.01, 0.01))
    s = max(n) / 2.0  # dam break: the longest side is 2
    return dict(n=n, size=tuple(v / s for v in n), side_bcid=(1,) * 6, bc_table=(wall, wall), rho=(1.0, 1000.0),
                mu=(1e-5, 1e-3), g=(0.0, 0.0, -9.81))


def _dt(case):
    """A step well under the convective and viscous CFL limits."""
    d = _desc(case)
    h = min(s / m for s, m in zip(d["size"], _n(case)))
    conv = {"tg": 0.12, "cavity": 0.15, "channel": 0.15, "dam": 0.04}[case["flow"]] * h
    return min(conv, 0.1 * h * h / max(d["mu"]))


def _fields(ctx, case, seed):
    n = _n(case)
    if case["flow"] == "tg":
        out = {f: _periodic_box(a, ctx.shape(f)) for f, a in zip("uvw", _tg_interior(n, seed))}
    elif case["flow"] == "cavity":
        out = _walled_velocity(ctx, seed, 0.2)
    elif case["flow"] == "channel":
        out = _walled_velocity(ctx, seed, 0.1, (0.5, 0.0, 0.0))
    else:  # a heavy column x < x0, z < z0, its surface smeared over a cell or two, nearly at rest
        out = _walled_velocity(ctx, seed, 0.02)
        g = torch.Generator()
        g.manual_seed(int(seed))
        x0, z0 = (0.2 + 0.2 * torch.rand(2, generator=g, dtype=F64)).tolist()
        shape = ctx.shape("alpha")
        z, _, x = (torch.arange(s, device="cuda", dtype=F64).clamp(1, s - 2) - 0.5 for s in shape)
        ax = torch.clamp(x0 * n[0] - x + 0.5, 0.0, 1.0)
        az = torch.clamp(2.0 * z0 * n[2] - z + 0.5, 0.0, 1.0)
        out["alpha"] = (az[:, None, None] * ax[None, None, :]).expand(shape).contiguous()
    out["p"] = torch.zeros(ctx.shape("p"), device="cuda", dtype=F64)
    return out


def prepare(case, seed):
    ctx = mydemcfd_amd.SMACContext(**_desc(case))
    st = dict(ctx=ctx, case=case, dt=_dt(case), opts=_opts(ctx, case), k=0)
    fields = _fields(ctx, case, seed)
    if case["kind"] in ("rollout", "vof_rollout"):
        names = ("alpha", "u", "v", "w", "p") if case["kind"] == "vof_rollout" else ("u", "v", "w", "p")
        st["ins"] = [fields[f].requires_grad_() for f in names]
        # cotangents of a loss on the final state: its interior entries
        st["cot"] = []
        for i, f in enumerate(names):
            c = torch.zeros(ctx.shape(f), device="cuda", dtype=F64)
            nx, ny, nz = _n(case)
            c[1:nz + 1, 1:ny + 1, 1:nx + 1] = torch.randn((nz, ny, nx), generator=_gen(seed + 31 * i + 1),
                                                          device="cuda", dtype=F64)
            st["cot"].append(c)
        torch.cuda.synchronize()
        return st
    planes, py, px = ctx.device_layout()
    st["box"] = {}
    for f, a in fields.items():
        box = torch.zeros((planes, py, px), device="cuda", dtype=F64)
        s = a.shape
        box[:s[0], :s[1], :s[2]] = a
        st["box"][f] = box
    if case["kind"] == "two_way":
        sh = ctx.shape("p")
        eps = 0.7 + 0.08 * _smooth(sh, 5 * seed + 1).clamp(-3, 3)
        old = eps + 0.02 * st["dt"] * _smooth(sh, 5 * seed + 2)
        st["dem"] = {"eps": eps.contiguous(), "eps_old": old.contiguous(), "eps_half": (0.5 * (eps + old)).contiguous()}
        vol = math.prod(s / m for s, m in zip(_desc(case)["size"], _n(case)))
        for a, f in enumerate(("impx", "impy", "impz")):
            st["dem"][f] = (1e-4 * vol * _smooth(ctx.shape(f), 5 * seed + 3 + a)).contiguous()
    torch.cuda.synchronize()  # the context's stream takes the tensors over
    for f, box in st["box"].items():
        ctx.bind_device(f, box.data_ptr(), box.numel())
    if "alpha" in fields:
        ctx.update_properties(True)
    return st


def _interior(st, names):
    nx, ny, nz = _n(st["case"])
    return {f: st["box"][f][1:nz + 1, 1:ny + 1, 1:nx + 1] for f in names}


def _whole(st, names):
    out = {}
    for f in names:
        s = st["ctx"].shape(f)
        out[f] = st["box"][f][:s[0], :s[1], :s[2]]
    return out


def run(st):
    ctx, dt, opts, kind = st["ctx"], st["dt"], st["opts"], st["case"]["kind"]
    st["k"] += 1
    if kind == "step":
        ctx.step(dt, opts)
        if st["case"]["flow"] == "channel":  # the outlet faces take their new values here
            ctx.update_boundary_ghost(dt)
        return _interior(st, "uvwp")
    if kind == "vof_loop":
        ctx.transport_alpha(dt, 2, st["k"])
        ctx.step(dt, opts)
        return _interior(st, ("u", "v", "w", "p", "alpha"))
    if kind == "config_loop":
        cfl = ctx.calc_cfl(dt)
        ctx.transport_alpha(dt, 2, st["k"])
        ctx.step(dt, opts)
        ctx.update_boundary_ghost(dt)
        return dict(_whole(st, ("u", "v", "w", "p", "alpha")), cfl=list(cfl))
    if kind == "two_way":
        for f, a in st["dem"].items():
            ctx.upload_device(f, a.data_ptr(), a.numel())
        ctx.update_poisson_beta_two_way()
        ctx.predictor_two_way(dt)
        ctx.pressure_solve(dt, opts)
        ctx.correct(dt)
        return _interior(st, "uvwp")
    if kind == "rollout":
        outs = autograd.rollout(ctx, *st["ins"], dt, st["case"]["nsteps"], opts)
    else:
        outs = autograd.vof_rollout(ctx, *st["ins"], dt, st["case"]["nsteps"], 2, opts)
    grads = torch.autograd.grad(outs, st["ins"], st["cot"])
    nx, ny, nz = _n(st["case"])
    return {"out": [o.detach()[1:nz + 1, 1:ny + 1, 1:nx + 1] for o in outs],
            "grad": [g[1:nz + 1, 1:ny + 1, 1:nx + 1] for g in grads]}


def work(case):
    """The canonical bytes of the path per cell (each array of a pass read or
    written once): predictor, right-hand side, correction, and `iters` PCG
    iterations with one application of the preconditioner each."""
    nx, ny, nz = _n(case)
    cells = float(nx * ny * nz)
    w = {"fp64": 8.0, "fp32": 4.0, "bf16": 2.0}[case["precision"]]
    var = case["flow"] in ("dam", "channel") or case["kind"] == "two_way"
    flex = 16.0 if case["precision"] != "fp64" else 0.0
    if case["precond"] == "mg":
        pre = 17.43 * w + (17.14 * w if var else 0.0)
    elif case["precond"] == "jacobi":
        pre = 16.0
    else:
        pre = 8.0 * 8.0 * (3.0 + (3.0 if var else 0.0)) * 8.0 / 7.0
    solve = 32.0 + 32.0 + pre + case["iters"] * (104.0 + pre + flex + (24.0 if var else 0.0))
    step = 128.0 + (48.0 if var else 0.0) + solve
    flops = 500.0 + case["iters"] * 200.0
    if case["kind"] in ("vof_loop", "config_loop", "vof_rollout"):
        step += 2 * 3 * 40.0 + 100.0
        flops += 2 * 3 * 150.0
    if case["kind"] == "two_way":
        step += 6 * 24.0
    if case["kind"] == "rollout":  # per step: the step, its transpose with a second solve, checkpoints
        step = case["nsteps"] * (2.0 * step + 100.0)
        flops *= 3.0 * case["nsteps"]
    if case["kind"] == "vof_rollout":  # the step taken twice and transposed
        step = case["nsteps"] * (3.0 * step + 200.0)
        flops *= 4.0 * case["nsteps"]
    return {"bytes": step * cells, "flops": flops * cells}


# ------------------------------------------------------------------ exact
def _minmod(a, b):
    return torch.where(a * b > 0.0, torch.where(a.abs() < b.abs(), a, b), torch.zeros_like(a))


def _predictor_periodic(vel, h, dt, nu):
    """u* of a periodic box with unit density at zero pressure: MUSCL-minmod
    advection and the viscous stress, explicit Euler."""
    def at(a, axis, s):  # a at q + s e_axis
        return torch.roll(a, -s, 2 - axis)

    star = []
    for a in range(3):
        c = vel[a]
        acc = torch.zeros_like(c)
        for e in range(3):
            nxt = at(c, e, 1)
            if e == a:
                m = 0.5 * (c + nxt)
                t = 2.0 * nu * (nxt - c) / h[a]
            else:
                b = at(vel[e], e, 1)
                bm = at(b, a, -1)
                m = 0.5 * (b + bm)
                t = nu * ((b - bm) / h[a] + (nxt - c) / h[e])
            sl = _minmod(nxt - c, c - at(c, e, -1))
            flux = m * torch.where(m > 0.0, c + 0.5 * sl, nxt - 0.5 * at(sl, e, 1)) - t
            acc -= (flux - at(flux, e, -1)) / h[e]
        star.append(c + dt * acc)
    return star


def exact(case, seed):
    """The projected velocity of a periodic step: the predictor in plain
    tensors, the Poisson equation by FFT. The pressure is left out (its mean is
    free), and so are walls, two phases and gradients."""
    if case["kind"] != "step" or case["flow"] != "tg":
        return None
    n, dt = _n(case), _dt(case)
    size, nu = _desc(case)["size"], _desc(case)["mu"][0]
    h = [s / m for s, m in zip(size, n)]
    star = _predictor_periodic(list(_tg_interior(n, seed)), h, dt, nu)

    def fwd(a, axis):
        return (torch.roll(a, -1, 2 - axis) - a) / h[axis]

    div = sum(fwd(star[a], a) for a in range(3))
    b = torch.fft.rfftn(div / dt)
    del div
    freq = [torch.arange(n[0] // 2 + 1, device="cuda", dtype=F64)[None, None, :],
            torch.arange(n[1], device="cuda", dtype=F64)[None, :, None],
            torch.arange(n[2], device="cuda", dtype=F64)[:, None, None]]
    lam = sum((2.0 * torch.cos(TWO_PI * f / m) - 2.0) / (s * s) for f, m, s in zip(freq, n, h))
    lam[0, 0, 0] = 1.0
    b = b / lam
    b[0, 0, 0] = 0.0
    p = torch.fft.irfftn(b, s=(n[2], n[1], n[0]))
    out = {f: (star[a] - dt * (p - torch.roll(p, 1, 2 - a)) / h[a]).cpu() for a, f in enumerate("uvw")}
    out["p"] = None
    return out
