"""GPU: the device copies of a field (upload_device, download_device) take the copy
kernel for memory of the context's GPU alone. Pinned host memory, which the runtime
can copy as well, goes through the runtime (the kernel's name in the profile counts
its launches), as memory of another GPU does; both give the field bit for bit. A
buffer that is not 8-byte aligned is the runtime's too.
"""
import numpy as np
import pytest

from mydemcfd_amd import cases

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _launches(ctx):
    return ctx.kernel_time("field_copy")[0] if "field_copy" in ctx.kernel_names() else 0


@pytest.mark.parametrize("n", [(9, 5, 6), (70, 13, 8)])
@pytest.mark.parametrize("field", ["u", "w", "p"])
def test_field_copy_routes(hip, n, field):
    print(f"case: device copies {field} {n}", flush=True)
    ctx = hip.SMACContext(**cases.cavity_desc(n))
    ctx.set_profiling(True)
    shape = ctx.shape(field)
    count = int(np.prod(shape))
    a = np.random.default_rng(2).standard_normal(shape)
    dev = torch.from_numpy(a).cuda()
    out = torch.zeros_like(dev)
    pinned = torch.empty(shape, dtype=torch.float64, pin_memory=True)
    pinned.copy_(torch.from_numpy(a))
    back = torch.zeros(shape, dtype=torch.float64).pin_memory()
    odd = torch.zeros(8 * count + 4, dtype=torch.uint8, device="cuda")[4:]
    odd.copy_(torch.from_numpy(np.frombuffer(a.tobytes(), dtype=np.uint8).copy()))
    torch.cuda.synchronize()
    # (source, destination, does the kernel copy it?)
    for src, dst, kernel in ((dev, out, True), (pinned, back, False), (odd, out, False)):
        ctx.upload(field, np.zeros(shape))
        dst.zero_()
        torch.cuda.synchronize()
        before = _launches(ctx)
        ctx.upload_device(field, src.data_ptr(), count)
        assert _launches(ctx) - before == (1 if kernel else 0)
        before = _launches(ctx)
        ctx.download_device(field, dst.data_ptr(), count)
        assert _launches(ctx) - before == (0 if dst is back else 1)
        assert np.array_equal(dst.cpu().numpy(), a)
