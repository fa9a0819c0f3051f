"""GPU: the norms that the host reads while the GPU works on come through memory that is
coherent whatever HIP_HOST_COHERENT makes of the default: a process with it off steps
with every preconditioner as this one does, bit for bit.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT
from mydemcfd_amd import cases

pytestmark = pytest.mark.gpu

FORMS = [dict(precond="jacobi", check_every=3), dict(precond="mg"), dict(precond="mg", precision="fp32", flexible=1),
         dict(precond="ref_gmg")]


def steps(hip):
    out = []
    for n in ((32, 32, 32), (16, 12, 8)):
        for kw in FORMS:
            if n != (32, 32, 32) and kw["precond"] != "jacobi":
                continue
            ctx = hip.SMACContext(**cases.cavity_desc(n))
            for _ in range(3):
                st = ctx.step(1e-3, tol=1e-8, **kw)
                out.append(np.array([st.iters, st.converged, st.rel_res, st.linf_res_dt]))
            out += [np.array(ctx.calc_cfl(1e-3))] + [ctx.download(f) for f in "uvwp"]
            ctx.close()
    return out


def test_coherence_by_request(hip, tmp_path):
    print("case: HIP_HOST_COHERENT=0", flush=True)
    path = str(tmp_path / "steps.npz")
    code = ("import sys; sys.path[:0] = sys.argv[1:3]; import numpy as np, mydemcfd_amd, test_gpu_host_coherent as t; "
            "np.savez(sys.argv[3], *t.steps(mydemcfd_amd))")
    subprocess.run([sys.executable, "-c", code, ROOT, os.path.join(ROOT, "tests"), path],
                   env=dict(os.environ, HIP_HOST_COHERENT="0"), check=True, timeout=100)
    with np.load(path) as other:
        mine = steps(hip)
        assert len(other.files) == len(mine)
        for k, a in zip(other.files, mine):
            assert np.array_equal(other[k], a), k
