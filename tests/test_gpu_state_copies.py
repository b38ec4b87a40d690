"""acDeviceLoadMeshFromDevicePtr and acDeviceStoreMeshToDevicePtr on states that are copied whole and on states that are
copied field by field, on both sides of 512 MiB: a state comes back bit for bit, and each field is where the device
exposes it."""
import numpy as np
import pytest

from astaroth_amd import astaroth as ac

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# 8 fields of (n + 6)^3 cells: 484 and 797 MiB in FP32, 11 and 778 MiB in FP64
@pytest.mark.parametrize("prec,n", [("fp32", (240, 250, 246)), ("fp32", (288, 294, 290)), ("fp64", (50, 60, 44)),
                                    ("fp64", (222, 230, 231))])
def test_state_round_trip(prec, n, require_gpu):
    lib = ac.load(prec)
    nbytes = 8 * int(np.prod([v + 6 for v in n])) * lib.np_real(0).nbytes
    print(f"case state copies {prec} n={n} {nbytes >> 20} MiB", flush=True)
    info = lib.config(n, AC_len=(2 * np.pi,) * 3)
    mx, my, mz = info["AC_mlocal"]
    t = torch.empty((ac.NUM_VTXBUF_HANDLES, mz, my, mx), dtype=torch.float32 if prec == "fp32" else torch.float64,
                    device="cuda")
    t.copy_(torch.arange(t.numel(), device="cuda").view(t.shape))  # no two fields alike
    back = torch.zeros_like(t)
    torch.cuda.synchronize()
    with ac.Device(lib, info) as dev:
        ac.check(lib.acDeviceLoadMeshFromDevicePtr(dev.handle, 0, t.data_ptr()), "load")
        ac.check(lib.acDeviceStoreMeshToDevicePtr(dev.handle, 0, back.data_ptr()), "store")
        dev.sync()
        assert torch.equal(t, back)
        for q in (0, 3, 7):
            want = (float(t[q, :, 3:-3, 3:-3][3:-3].min()), float(t[q, :, 3:-3, 3:-3][3:-3].max()))
            assert (dev.reduce_scal("RTYPE_MIN", q), dev.reduce_scal("RTYPE_MAX", q)) == want
