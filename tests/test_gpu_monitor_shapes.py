"""Reductions, diagnostics, the reference timestep's maxima and the forcing on grids that their column
blocks, plane chunks and unrolled loads do not divide, against numpy in float64 (the tolerances of the
same checks on even grids: FP32 derivatives round at 2e-5 of the largest |B|, FP64 at 1e-11)."""
import ctypes

import numpy as np
import pytest

from astaroth_amd import astaroth as ac
import oracle.oracle as O
from tests.test_gpu_forcing import forced_info, oracle_step_with_forcing, run_steps
from tests.test_gpu_parity import curl_6th, reference_dt_numpy

pytestmark = pytest.mark.gpu
GRIDS = [(5, 4, 3), (65, 17, 9), (255, 3, 8), (30, 31, 70), (300, 40, 33)]


@pytest.fixture(scope="module", params=["fp32", "fp64"])
def lib(request, require_gpu):
    return ac.load(request.param)


@pytest.mark.parametrize("n", GRIDS)
def test_monitoring_on_any_grid(lib, n):
    print(f"case monitoring shapes {lib.precision} n={n}", flush=True)
    info = lib.config(n, AC_len=(2 * np.pi,) * 3, AC_cs_sound=1.0, AC_nu_visc=5e-3, AC_eta=5e-3)
    cfg = O.config_from_info(info)
    rng = np.random.default_rng(n[0])
    data = (0.3 * rng.standard_normal((ac.NUM_VTXBUF_HANDLES, n[2] + 6, n[1] + 6, n[0] + 6))).astype(lib.np_real)
    O.periodic_fill(data, cfg)
    sl = O.interior_slices(data.shape[1:])
    f = [data[q][sl].astype(np.float64) for q in range(8)]
    b2 = sum(c * c for c in curl_6th(data[4:7], [float(v) for v in info["AC_ds"]]))
    u2 = f[1] ** 2 + f[2] ** 2 + f[3] ** 2
    va2 = b2 / np.exp(f[0])
    tol, eps = (2e-5, 1e-6) if lib.precision == "fp32" else (1e-11, 1e-13)
    with ac.Device(lib, info) as dev:
        dev.load_mesh(ac.HostMesh(lib, info, data))
        d = dev.diagnostics()
        for q in range(8):
            assert d.min[q] == f[q].min() and d.max[q] == f[q].max()
            assert d.rms[q] == pytest.approx(np.sqrt((f[q] ** 2).mean()), rel=1e-13)
        for name, v2, t in (("uu", u2, 1e-13), ("bb", b2, tol), ("va", va2, tol)):
            for kind, want in (("min", v2.min()), ("max", v2.max()), ("rms", v2.mean())):
                got = getattr(d, f"{name}_{kind}")
                assert got == pytest.approx(np.sqrt(want), rel=t, abs=t * np.sqrt(v2.max())), (name, kind)
        for q in (0, 7):
            assert dev.reduce_scal("RTYPE_MAX", q) == f[q].max()
            assert dev.reduce_scal("RTYPE_MIN", q) == f[q].min()
            assert dev.reduce_scal("RTYPE_RMS", q) == pytest.approx(np.sqrt((f[q] ** 2).mean()), rel=eps)
        assert dev.reduce_vec("RTYPE_MAX", 1, 2, 3) == pytest.approx(np.sqrt(u2.max()), rel=eps)
        assert dev.reduce_vec("RTYPE_RMS", 1, 2, 3) == pytest.approx(np.sqrt(u2.mean()), rel=eps)
        got = dev.reduce_vec_scal("RTYPE_ALFVEN_RMS", 1, 2, 3, 0)
        assert got == pytest.approx(np.sqrt((u2 / np.exp(f[0])).mean()), rel=eps)
        dt = ctypes.c_double()
        for mode in (0, 1):
            ac.check(lib.acDeviceSetTimestepMode(dev.handle, mode), "mode")
            ac.check(lib.acDeviceUpdateTimestepCFL(dev.handle, 0, lib.np_real(0.5)), "cfl")
            ac.check(lib.acDeviceGetTimestep(dev.handle, 0, ctypes.byref(dt)), "dt")
            if mode == 0:
                want = 0.5 * float(min(info["AC_ds"])) / (1.0 + np.sqrt(u2.max()))
                assert dt.value == pytest.approx(want, rel=1e-6)
            else:
                assert dt.value == pytest.approx(reference_dt_numpy(data, info, False), rel=max(tol, 1e-6))


@pytest.mark.parametrize("n", [(65, 17, 9), (20, 31, 40)])
def test_forcing_on_any_grid(lib, n):
    print(f"case forcing shapes {lib.precision} n={n}", flush=True)
    info, fp = forced_info(lib, n, (0, 0, 0), relhel=0.5)
    rng = np.random.default_rng(3)
    data = (0.01 * rng.standard_normal((ac.NUM_VTXBUF_HANDLES, n[2] + 6, n[1] + 6, n[0] + 6))).astype(lib.np_real)
    O.periodic_fill(data, O.config_from_info(info))
    dt = 2e-3
    model = oracle_step_with_forcing(lib, info, data, fp, dt)
    for q, e in enumerate(O.field_errors(model, run_steps(lib, info, data, dt, 1))):
        assert e["maxrel"] < (2e-5 if lib.precision == "fp32" else 1e-12), (q, e)
