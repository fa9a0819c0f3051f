"""GPU: the predictor of grids with walls or property arrays (k_predict_rim,
k_predict_inner): boxes with no inner faces, with one, and with several blocks
of them; every wall type, periodic axes beside walls; one-phase, two-phase,
after a VoF transport, two-way, two-way after a transport. u*, v*, w* equal to
the oracle's bit for bit.
"""
import numpy as np
import pytest

from mydemcfd_amd import _abi, cases

pytestmark = pytest.mark.gpu

SIZES = [(2, 3, 4), (5, 6, 7), (6, 6, 6), (7, 9, 6), (70, 8, 11)]
MODES = ["one", "two", "vof", "tw", "tw_two", "tw_vof"]
TABLE = ((_abi.BC_NOSLIP, 0.0, 0.0, 0.0), (_abi.BC_NOSLIP, 0.4, -0.2, 0.3), (_abi.BC_INFLOW, 0.5, 0.1, -0.1),
         (_abi.BC_OUTLET, 0.0, 0.0, 0.0), (_abi.BC_SLIP, 0.0, 0.0, 0.0))
KINDS = {"walls": ((0, 0, 0), (0, 1, 1, 4, 4, 0)), "through": ((0, 0, 0), (2, 3, 4, 1, 3, 2)),
         "mixed": ((1, 0, 0), (0, 0, 1, 3, 4, 2)), "mixed_z": ((0, 1, 1), (4, 2, 0, 0, 0, 0)),
         "periodic": ((1, 1, 1), (0, 0, 0, 0, 0, 0))}


@pytest.mark.parametrize("kind,n", [(k, n) for k in KINDS for n in SIZES if min(n) >= 4 or not any(KINDS[k][0])])
@pytest.mark.parametrize("mode", MODES)
def test_predictor(hip, oracle_mod, mode, kind, n):
    print(f"case: predictor {mode} {kind} {n}", flush=True)
    per, sides = KINDS[kind]
    two = mode not in ("one", "tw")
    desc = dict(n=n, size=tuple(v / 8.0 for v in n), periodic=per, side_bcid=sides, bc_table=TABLE,
                rho=(1.0, 5.0) if two else (1.0, 1.0), mu=(0.01, 0.03) if two else (0.01, 0.01), g=(0.1, -1.0, 0.2))
    g, o = hip.SMACContext(**desc), oracle_mod.OracleContext(**desc)
    rng = np.random.default_rng(17)
    fields = {f: 0.3 * rng.standard_normal(o.shape(f)) for f in ("u", "v", "w", "p")}
    if two:
        fields["alpha"] = (rng.uniform(size=o.shape("alpha")) > 0.5).astype(np.float64)
    if mode.startswith("tw"):
        for s, f in enumerate(("eps", "eps_old", "eps_half")):
            fields[f] = cases.void_fraction(n, per, 7 + s)
        for f in ("impx", "impy", "impz"):
            fields[f] = 1e-4 * rng.standard_normal(o.shape(f))
    out = []
    for c in (g, o):
        for f, a in fields.items():
            c.upload(f, a)
        c.update_properties(True)
        if mode.endswith("vof"):
            c.transport_alpha(1e-3, 2, 1)
        (c.predictor_two_way if mode.startswith("tw") else c.predictor)(1e-3)
        out.append([c.download(f) for f in ("ustar", "vstar", "wstar")])
    for f, a, b in zip("uvw", *out):
        assert np.max(np.abs(b)) > 0.0 and np.array_equal(a, b), (f, float(np.max(np.abs(a - b))))
