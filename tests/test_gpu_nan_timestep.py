"""The device-resident timestep of a state that has blown up: a velocity that is NaN everywhere gives a NaN
timestep and a NaN simulated time (the cheapest sign a run has) where the role-split, the direct or the
forcing kernel reduces the velocity; a finite state gives finite ones."""
import ctypes

import numpy as np
import pytest

from astaroth_amd import astaroth as ac

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["fp32", "fp64"])
def lib(request, require_gpu):
    return ac.load(request.param)


# autotuned (role-split) on a ragged and on a divisible grid, its blocks past the edge, direct
@pytest.mark.parametrize("n,shape,kind", [((100, 20, 12), (0, 0, 0), 0), ((64, 8, 16), (32, 4, 16), 2),
                                          ((65, 9, 7), (16, 8, 3), 2), ((128, 8, 8), (-1, 0, 0), 0)])
@pytest.mark.parametrize("forcing", [False, True])
@pytest.mark.parametrize("blown", [True, False])
def test_timestep_of_a_nan_state(lib, n, shape, kind, forcing, blown):
    print(f"case nan timestep {lib.precision} n={n} shape={shape} kind={kind} forcing={forcing} {blown}", flush=True)
    info = lib.config(n, AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3, AC_eta=5e-3,
                      AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=True, AC_lentropy=True, AC_lforcing=forcing,
                      AC_switch_forcing=-1.0, AC_solve_tile_x=shape[0], AC_solve_tile_y=shape[1],
                      AC_solve_zchunk=shape[2], AC_solve_kernel=kind)
    mesh = ac.HostMesh(lib, info)
    assert lib.acHostMeshInitFourier(ctypes.byref(mesh.struct), 5, 16, 4, 0.05, 0.0) == 0
    data = mesh.data.copy()
    if blown:
        data[1:4] = np.nan
    courant = lib.np_real(0.2)
    dt, time = ctypes.c_double(), ctypes.c_double()
    with ac.Device(lib, info) as dev:
        dev.load_mesh(mesh)
        ac.check(lib.acDeviceUpdateTimestepCFL(dev.handle, 0, courant), "cfl")
        dev.load_mesh(ac.HostMesh(lib, info, data))
        ac.check(lib.acDeviceIntegrateStepsCFL(dev.handle, 0, 2, courant, ctypes.byref(time)), "steps")
        ac.check(lib.acDeviceGetTimestep(dev.handle, 0, ctypes.byref(dt)), "timestep")
    assert np.isnan(dt.value) == blown and np.isnan(time.value) == blown
