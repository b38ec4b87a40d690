"""Whole-step calls against the separate ones, bit for bit: acDeviceIntegrateStep (halos of the returned
state included) for each kind of solve kernel, the direct kernel's periodic-image reads, and
acDeviceIntegrateStepAdjoint against recomputation and adjoint substeps one by one."""
import ctypes

import numpy as np
import pytest

from astaroth_amd import astaroth as ac
from astaroth_amd import adjoint as AD
import oracle.oracle as O

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", params=["fp32", "fp64"])
def lib(request, require_gpu):
    return ac.load(request.param)


def config(lib, n, shape, kind, **over):
    p = dict(AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_gamma=5.0 / 3.0, AC_nu_visc=5e-3, AC_eta=5e-3,
             AC_chi=5e-3, AC_K_heatcond=5e-3, AC_lupwd=True, AC_lentropy=True, AC_solve_tile_x=shape[0],
             AC_solve_tile_y=shape[1], AC_solve_zchunk=shape[2], AC_solve_kernel=kind)
    p.update(over)
    return lib.config(n, **p)


def initial(lib, info, seed):
    mx, my, mz = info["AC_mlocal"]
    rng = np.random.default_rng(seed)
    return (0.02 * rng.standard_normal((ac.NUM_VTXBUF_HANDLES, mz, my, mx))).astype(lib.np_real)


def separate_step(dev, dt):
    for s in range(3):
        dev.periodic()
        dev.substep(s, dt)
        dev.swap()


# split (autotuned), delay-line, ring, direct from LDS blocks and from the caches, narrower than the halo
@pytest.mark.parametrize("n,shape,kind", [((37, 21, 18), (0, 0, 0), 0), ((64, 8, 16), (64, 4, 16), 0),
                                          ((32, 8, 32), (32, 8, 32), 0), ((45, 30, 41), (-1, 0, 0), 0),
                                          ((17, 9, 6), (-1, 0, 0), 0), ((2, 5, 4), (0, 0, 0), 0)])
def test_step_equals_separate_calls(lib, n, shape, kind):
    print(f"case step {lib.precision} n={n} shape={shape} kind={kind}", flush=True)
    info = config(lib, n, shape, kind)
    data = initial(lib, info, 1)
    dt = lib.np_real(1e-3)
    outs = []
    for whole in (True, False):
        with ac.Device(lib, info) as dev:
            dev.load_mesh(ac.HostMesh(lib, info, data))
            for _ in range(2):
                dev.step(dt) if whole else separate_step(dev, dt)
            out = ac.HostMesh(lib, info)
            dev.store_mesh(out)
            outs.append(out.data.copy())
    assert np.isfinite(outs[0]).all()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("kb", [0, 16, 32])
def test_direct_periodic_reads(lib, kb):
    if kb and lib.precision == "fp64":
        pytest.skip("compensation is FP32 only")
    n = (45, 30, 41)
    print(f"case direct periodic reads {lib.precision} kahan={kb}", flush=True)
    info = config(lib, n, (-1, 0, 0), 0, AC_kahan_bits=kb)
    data = initial(lib, info, 2)
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
            out = ac.HostMesh(lib, info)
            dev.periodic()
            dev.store_mesh(out)
            outs.append(out.data.copy())
    assert np.isfinite(outs[0]).all()
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("n", [(64, 8, 12), (29, 20, 17)])
def test_step_adjoint_equals_substeps(lib, n):
    print(f"case step adjoint {lib.precision} n={n}", flush=True)
    info = config(lib, n, (0, 0, 0), 0)
    data = initial(lib, info, 3)
    O.periodic_fill(data, O.config_from_info(info))
    runner = AD.MHDAdjoint(lib, info, 1, 1e-3)
    f = torch.from_numpy(data).to(runner.tdev)
    g = torch.Generator(device="cpu").manual_seed(5)
    lam = [torch.randn(runner.shape, generator=g, dtype=torch.float64).to(runner.tdtype).to(runner.tdev)
           for _ in range(2)]
    results = []
    for whole in (True, False):
        lf, lw = lam[0].clone(), lam[1].clone()
        runner.param_grad.zero_()
        runner.load(f)
        if whole:
            runner.reverse_step(lf, lw)
        else:
            states = []
            for s in range(3):
                runner.dev.periodic()
                t = runner.empty()
                runner.store(t)
                states.append(t)
                if s < 2:
                    runner.dev.substep(s, runner.dt)
                    runner.dev.swap()
            for s in (2, 1, 0):
                runner.load(states[s])
                ac.check(lib.acDeviceIntegrateSubstepAdjoint(
                    runner.dev.handle, 0, s, runner.dt, ctypes.c_void_p(lf.data_ptr()), ctypes.c_void_p(lw.data_ptr()),
                    ctypes.c_void_p(runner.workspace.data_ptr()), ctypes.c_void_p(runner.param_grad.data_ptr())), "adj")
        runner._sync()
        torch.cuda.synchronize()
        results.append([x.cpu().numpy() for x in (lf[:, 3:-3, 3:-3, 3:-3], lw[:, 3:-3, 3:-3, 3:-3], runner.param_grad)])
    runner.close()
    for a, b in zip(*results):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
