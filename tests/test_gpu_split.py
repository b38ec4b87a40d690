"""The role-split solve kernel (solve_split.hip, AC_solve_kernel = 2) at the edges of its column blocks
and z-chunks: grids smaller than a block, one column or plane past a block, chunks of one plane and
ragged last chunks; against the oracle, and its periodic-image reads (multi-step path) against
fill + substep + swap bit for bit with every compensation width."""
import ctypes
import sys

import numpy as np
import pytest

from astaroth_amd import astaroth as ac
import oracle.oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=["fp32", "fp64"])
def lib(request, require_gpu):
    return ac.load(request.param)


def config(lib, n, shape, **over):
    if lib.precision == "fp64" and shape[:2] == (64, 4):
        pytest.skip("64 x 4 column blocks exist in FP32 only")
    p = dict(AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3,
             AC_eta=5e-3, AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=True, AC_lentropy=True,
             AC_solve_tile_x=shape[0], AC_solve_tile_y=shape[1], AC_solve_zchunk=shape[2],
             AC_solve_kernel=2)
    p.update(over)
    return lib.config(n, **p)


def initial(lib, info, seed=7):
    mesh = ac.HostMesh(lib, info)
    assert lib.acHostMeshInitFourier(ctypes.byref(mesh.struct), seed, 16, 4, 0.05, 0.0) == 0
    data = mesh.data.copy()
    rng = np.random.default_rng(seed)
    data[0] += 0.01 * rng.standard_normal(data[0].shape).astype(data.dtype)
    data[7] += 0.01 * rng.standard_normal(data[7].shape).astype(data.dtype)
    O.periodic_fill(data, O.config_from_info(info))
    return data


CASES = [((32, 4, 8), (32, 4, 8)), ((33, 5, 7), (32, 4, 3)), ((5, 3, 4), (32, 4, 1)),
         ((31, 11, 9), (32, 4, 9)), ((17, 9, 12), (16, 8, 5)), ((16, 8, 6), (16, 8, 6)),
         ((64, 4, 16), (64, 4, 16)), ((65, 7, 10), (64, 4, 4)), ((70, 13, 8), (64, 4, 1))]


@pytest.mark.parametrize("n,shape", CASES)
@pytest.mark.parametrize("upwd,entropy", [(True, True), (False, False), (True, False), (False, True)])
def test_split_vs_oracle(lib, n, shape, upwd, entropy):
    print(f"case split vs oracle {lib.precision} n={n} shape={shape} {upwd} {entropy}", flush=True)
    info = config(lib, n, shape, AC_lupwd=upwd, AC_lentropy=entropy)
    data = initial(lib, info)
    dt, steps = 2e-3, 2
    kind = ctypes.c_int()
    with ac.Device(lib, info) as dev:
        lib.acDeviceGetSolveKernel(dev.handle, ctypes.byref(kind))
        assert kind.value == 2
        dev.load_mesh(ac.HostMesh(lib, info, data))
        for _ in range(steps):
            dev.step(lib.np_real(dt))
        dev.periodic()
        out = ac.HostMesh(lib, info)
        dev.store_mesh(out)
    model = data.astype(np.float64)
    cfg = O.config_from_info(info)
    for _ in range(steps):
        O.integrate_step(model, cfg, dt)
    O.periodic_fill(model, cfg)
    # the bounds of the delay-line kernel's test of the same kind of state
    tol = 2e-5 if lib.precision == "fp32" else 1e-12
    for q, e in enumerate(O.field_errors(model, out.data)):
        assert e["maxrel"] < tol, (q, e)


@pytest.mark.parametrize("n,shape", [((33, 5, 7), (32, 4, 3)), ((19, 10, 5), (16, 8, 2)),
                                     ((65, 6, 9), (64, 4, 9))])
@pytest.mark.parametrize("kb,entropy", [(0, True), (8, True), (16, False), (32, True), (32, False)])
def test_split_fused_periodic_steps(lib, n, shape, kb, entropy):
    if kb and lib.precision == "fp64":
        pytest.skip("compensation is FP32 only")
    print(f"case split fused {lib.precision} n={n} shape={shape} kahan={kb} {entropy}", flush=True)
    info = config(lib, n, shape, AC_kahan_bits=kb, AC_lentropy=entropy)
    data = initial(lib, info, seed=11)
    courant = lib.np_real(0.3)
    outs = []
    for fused in (True, False):
        with ac.Device(lib, info) as dev:
            dev.load_mesh(ac.HostMesh(lib, info, data))
            ac.check(lib.acDeviceUpdateTimestepCFL(dev.handle, 0, courant), "cfl")
            if fused:
                ac.check(lib.acDeviceIntegrateStepsCFL(dev.handle, 0, 2, courant, None), "steps")
            else:
                for s in (0, 1, 2, 0, 1, 2):
                    dev.periodic()
                    ac.check(lib.acDeviceIntegrateSubstepDeviceDt(dev.handle, 0, s, courant), "substep")
                    dev.swap()
            dev.periodic()
            out = ac.HostMesh(lib, info)
            dev.store_mesh(out)
            outs.append(out.data.copy())
    assert np.isfinite(outs[0]).all()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("n", [(64, 32, 32), (45, 33, 26)])
def test_gradient_runner_keeps_to_column_kernels(lib, n):
    """FP32 gradients are taken with the kernels that hold a cell per thread; FP64 ones with any."""
    from astaroth_amd import adjoint as AD
    print(f"case gradient kernels {lib.precision} n={n}", flush=True)
    kind = ctypes.c_int()
    kinds = []
    for make in (lambda i: AD.MHDAdjoint(lib, i, 1, 1e-3).dev, lambda i: ac.Device(lib, i)):
        with make(config(lib, n, (0, 0, 0), AC_solve_kernel=0)) as dev:
            dev.step(lib.np_real(1e-3))
            dev.sync()
            ac.check(lib.acDeviceGetSolveKernel(dev.handle, ctypes.byref(kind)), "kind")
            kinds.append(kind.value)
    assert kinds[1] == 2  # both grids are past the 32^3 cells up to which the direct kernel is tried
    assert kinds[0] == 2 if lib.precision == "fp64" else kinds[0] in (-1, 0, 1)
