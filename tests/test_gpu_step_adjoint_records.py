"""acDeviceIntegrateStepAdjoint on a device with compensation records: the state and the records that belong to
it stay, so that the next step is the one without the call, bit for bit; and the adjoint is the one of an
uncompensated device with the same state."""
import ctypes

import numpy as np
import pytest

from astaroth_amd import astaroth as ac

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def config(lib, n, shape, kind, kb):
    return lib.config(n, AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3,
                      AC_eta=5e-3, AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=True, AC_lentropy=True,
                      AC_kahan_bits=kb, AC_solve_tile_x=shape[0], AC_solve_tile_y=shape[1],
                      AC_solve_zchunk=shape[2], AC_solve_kernel=kind)


def step_adjoint(lib, dev, dt):
    """lambda_f, lambda_w and the parameter sums from seeded adjoint states."""
    shape = dev_shape(dev)
    g = torch.Generator(device="cpu").manual_seed(5)
    lf, lw = (torch.randn(shape, generator=g).cuda() for _ in range(2))
    work = torch.empty(int(lib.acAdjointWorkspaceBytes(dev.handle)), dtype=torch.uint8, device="cuda")
    scratch, params = torch.empty_like(lf), torch.zeros(2, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ac.check(lib.acDeviceIntegrateStepAdjoint(
        dev.handle, 0, dt, *(ctypes.c_void_p(t.data_ptr()) for t in (scratch, lf, lw, work, params))), "adjoint")
    dev.sync()
    return [t[:, 3:-3, 3:-3, 3:-3].cpu().numpy() for t in (lf, lw)] + [params.cpu().numpy()]


def dev_shape(dev):
    mx, my, mz = dev.info["AC_mlocal"]
    return (ac.NUM_VTXBUF_HANDLES, mz, my, mx)


# direct (staged and not), delay-line, role-split
@pytest.mark.parametrize("n,shape,kind", [((45, 30, 41), (-1, 0, 0), 0), ((17, 9, 6), (-1, 0, 0), 0),
                                          ((64, 8, 16), (64, 4, 16), 0), ((33, 21, 18), (32, 4, 9), 2)])
@pytest.mark.parametrize("kb", [8, 16, 32])
def test_records_stay(n, shape, kind, kb, require_gpu):
    print(f"case step adjoint records n={n} shape={shape} kind={kind} kahan={kb}", flush=True)
    lib = ac.load("fp32")
    info = config(lib, n, shape, kind, kb)
    mesh = ac.HostMesh(lib, info)
    assert lib.acHostMeshInitFourier(ctypes.byref(mesh.struct), 2024, 16, 4, 0.05, 0.0) == 0
    dt = lib.np_real(1e-3)
    outs = []
    for call in (True, False):
        with ac.Device(lib, info) as dev:
            dev.load_mesh(mesh)
            for _ in range(3):
                dev.step(dt)
            if call:
                state = torch.empty(dev_shape(dev), device="cuda")
                dev.periodic()
                ac.check(lib.acDeviceStoreMeshToDevicePtr(dev.handle, 0, ctypes.c_void_p(state.data_ptr())), "store")
                dev.sync()
                adjoint = step_adjoint(lib, dev, dt)
            dev.step(dt)
            out = ac.HostMesh(lib, info)
            dev.store_mesh(out)
            outs.append(out.data.copy())
    assert np.isfinite(outs[0]).all()
    assert np.array_equal(outs[0], outs[1])
    with ac.Device(lib, config(lib, n, shape, kind, 0)) as dev:
        ac.check(lib.acDeviceLoadMeshFromDevicePtr(dev.handle, 0, ctypes.c_void_p(state.data_ptr())), "load")
        dev.sync()
        for a, b in zip(adjoint, step_adjoint(lib, dev, dt)):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b)
