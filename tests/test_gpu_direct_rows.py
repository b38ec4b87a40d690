"""The direct solve kernel on FP32 grids of at most one block per CU, where its workgroups take rows of 64 cells or
blocks of 16 x 4 x 4, whichever makes fewer (rows up to twice as many): ragged rows and blocks on both sides of the
line, plain and with compensation records, against the oracle."""
import ctypes

import numpy as np
import pytest

from astaroth_amd import astaroth as ac
import oracle.oracle as O

pytestmark = pytest.mark.gpu


# rows: 65 and 130 cells wide, fewer rows than blocks, 1.8 times as many; blocks: exactly twice as many, four times
@pytest.mark.parametrize("n", [(65, 9, 6), (130, 20, 8), (100, 5, 7), (24, 20, 18), (32, 12, 16), (16, 13, 17)])
@pytest.mark.parametrize("kb,upwd,entropy", [(0, True, True), (16, False, True), (32, True, False)])
def test_direct_rows_and_blocks(n, kb, upwd, entropy, require_gpu):
    print(f"case direct rows n={n} kahan={kb} upwd={upwd} entropy={entropy}", flush=True)
    lib = ac.load("fp32")
    info = lib.config(n, AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3, AC_eta=5e-3,
                      AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=upwd, AC_lentropy=entropy, AC_kahan_bits=kb,
                      AC_solve_tile_x=-1)
    mesh = ac.HostMesh(lib, info)
    assert lib.acHostMeshInitFourier(ctypes.byref(mesh.struct), 9, 16, 4, 0.05, 0.0) == 0
    dt, steps = 1e-3, 2
    kind = ctypes.c_int()
    with ac.Device(lib, info) as dev:
        lib.acDeviceGetSolveKernel(dev.handle, ctypes.byref(kind))
        dev.load_mesh(mesh)
        for _ in range(steps):
            dev.step(lib.np_real(dt))
        dev.periodic()
        out = ac.HostMesh(lib, info)
        dev.store_mesh(out)
    assert kind.value == -1
    model = mesh.data.astype(np.float64)
    cfg = O.config_from_info(info)
    for _ in range(steps):
        O.integrate_step(model, cfg, dt)
    O.periodic_fill(model, cfg)
    for q, e in enumerate(O.field_errors(model, out.data)):
        assert e["maxrel"] < 2e-5, (q, e)  # the bound of the solve kernels' tests on this kind of state
