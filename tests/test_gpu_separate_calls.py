"""The reference API's loop of separate calls, acDevicePeriodicBoundconds + acDeviceIntegrateSubstep +
acDeviceSwapBuffers per substep: against the oracle for each kind of solve kernel, and at 256^3 against
acDeviceIntegrateStep, halos included, bit for bit."""
import ctypes

import numpy as np
import pytest

from astaroth_amd import astaroth as ac
import oracle.oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["fp32", "fp64"])
def lib(request, require_gpu):
    return ac.load(request.param)


def config(lib, n, shape=(0, 0, 0), kind=0):
    return lib.config(n, AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3, AC_eta=5e-3,
                      AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=True, AC_lentropy=True, AC_solve_tile_x=shape[0],
                      AC_solve_tile_y=shape[1], AC_solve_zchunk=shape[2], AC_solve_kernel=kind)


def initial(lib, info, seed=7):
    mesh = ac.HostMesh(lib, info)
    assert lib.acHostMeshInitFourier(ctypes.byref(mesh.struct), seed, 16, 4, 0.05, 0.0) == 0
    data = mesh.data.copy()
    rng = np.random.default_rng(seed)
    for q in (0, 7):
        data[q] += 0.01 * rng.standard_normal(data[q].shape).astype(data.dtype)
    O.periodic_fill(data, O.config_from_info(info))
    return data


def separate_steps(dev, dt, steps):
    for _ in range(steps):
        for s in range(3):
            dev.periodic()
            dev.substep(s, dt)
            dev.swap()


def stored(lib, info, dev):
    out = ac.HostMesh(lib, info)
    dev.store_mesh(out)
    return out.data


# autotuned (role-split), role-split, delay-line, ring, direct from LDS blocks and from the caches, sweep
@pytest.mark.parametrize("n,shape,kind", [((37, 21, 18), (0, 0, 0), 0), ((33, 21, 18), (32, 4, 9), 2),
                                          ((64, 8, 16), (64, 4, 16), 0), ((32, 8, 32), (32, 8, 32), 0),
                                          ((45, 30, 41), (-1, 0, 0), 0), ((17, 9, 6), (-1, 0, 0), 0),
                                          ((64, 32, 32), (64, 4, 32), 1)])
def test_separate_calls_vs_oracle(lib, n, shape, kind):
    if kind == 1 and lib.precision == "fp64":
        pytest.skip("the sweep kernel is FP32 only")
    print(f"case separate calls vs oracle {lib.precision} n={n} shape={shape} kind={kind}", flush=True)
    info = config(lib, n, shape, kind)
    data = initial(lib, info)
    dt, steps = 2e-3, 2
    with ac.Device(lib, info) as dev:
        dev.load_mesh(ac.HostMesh(lib, info, data))
        separate_steps(dev, lib.np_real(dt), steps)
        dev.periodic()
        out = stored(lib, info, dev)
    model = data.astype(np.float64)
    cfg = O.config_from_info(info)
    for _ in range(steps):
        O.integrate_step(model, cfg, dt)
    O.periodic_fill(model, cfg)
    # the bounds of the solve kernels' tests on the same kind of state
    for q, e in enumerate(O.field_errors(model, out)):
        assert e["maxrel"] < (2e-5 if lib.precision == "fp32" else 1e-12), (q, e)


def test_separate_calls_equal_whole_steps_256(lib):
    print(f"case separate calls against whole steps {lib.precision} 256^3", flush=True)
    info = config(lib, (256, 256, 256))
    mesh = ac.HostMesh(lib, info)
    assert lib.acHostMeshInitFourier(ctypes.byref(mesh.struct), 2024, 16, 4, 0.05, 0.0) == 0
    dt = lib.np_real(1e-3)
    with ac.Device(lib, info) as dev:  # one device, so that both run the kernel that its autotuner took
        dev.load_mesh(mesh)
        separate_steps(dev, dt, 2)
        separate = stored(lib, info, dev)
        dev.load_mesh(mesh)
        for _ in range(2):
            dev.step(dt)
        whole = stored(lib, info, dev)
    assert np.isfinite(separate).all()
    assert np.array_equal(separate, whole)
    assert not np.array_equal(separate, mesh.data)
