"""The role-split kernel's compensation records (each thread of a column packs its own half of them) against
the oracle: the case, the widths, the bounds and the comparison with plain FP32 of test_gpu_kahan_parity.py, for
each column block on a grid that it divides and one that it does not."""
import ctypes

import numpy as np
import pytest

from astaroth_amd import astaroth as ac
import oracle.oracle as O
from tests.test_gpu_kahan_parity import BOUND, c1_info, run, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shape", [((64, 32, 32), (64, 4, 32)), ((70, 30, 27), (64, 4, 10)),
                                     ((32, 32, 32), (32, 4, 32)), ((45, 30, 33), (32, 4, 11)),
                                     ((32, 32, 32), (16, 8, 32)), ((35, 29, 26), (16, 8, 7))])
def test_split_kahan_vs_oracle(n, shape, require_gpu):
    lib = ac.load("fp32")
    dt, steps = np.float32(1e-3), 10
    info = c1_info(lib, n, shape, 2, 0)
    mesh = ac.HostMesh(lib, info)
    assert lib.acHostMeshInitFourier(ctypes.byref(mesh.struct), 2024, 16, 4, 0.05, 0.0) == 0
    model = mesh.data.astype(np.float64)
    cfg = O.config_from_info(info)
    for _ in range(steps):
        O.integrate_step(model, cfg, float(dt))
    O.periodic_fill(model, cfg)
    errs = {}
    for kb in (0, 8, 16, 32):
        kind = ctypes.c_int()
        with ac.Device(lib, c1_info(lib, n, shape, 2, kb)) as dev:
            lib.acDeviceGetSolveKernel(dev.handle, ctypes.byref(kind))
        assert kind.value == 2
        errs[kb] = O.field_errors(model, run(lib, c1_info(lib, n, shape, 2, kb), mesh.data.copy(), dt, steps))
        say(f"case split kahan vs oracle n={n} shape={shape} kb={kb}: " +
            " ".join(f"{e['maxrel']:.2e}" for e in errs[kb]))
    for kb in (0, 8, 16, 32):
        for q, e in enumerate(errs[kb]):
            assert e["maxrel"] < BOUND[kb] and e["l2"] < BOUND[kb], (kb, q, e)
    for kb in (8, 16, 32):
        for q in (0, 7):  # they start at zero and stay small: their error is the rounding of the update
            assert errs[kb][q]["maxrel"] < errs[0][q]["maxrel"], (kb, q)
