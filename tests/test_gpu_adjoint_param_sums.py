"""The adjoint's parameter sums on both sides of the line where they take a second stage (4096 block partials).
With lambda_w = dw', the tangent of the substep in the direction of one parameter, the adjoint's sum for that
parameter is <dw', dw'>, in which nothing cancels: each cell's term agrees to FP32's rounding of a second
derivative (about 3e-5 of it at these spacings, of either sign, so far less in the sum over 1e5 cells or more); a
lost range of partials would take out 1/256 of it or more."""
import ctypes

import pytest

from astaroth_amd import astaroth as ac
from tests.test_gpu_adjoint import idot, initial, physics_info, say

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", params=["fp64", "fp32"])
def lib(request, require_gpu):
    return ac.load(request.param)


# 4600 block partials (two stages), 4032, 4096 (in FP64; FP32 takes columns there), 4160, 825 of ragged blocks
@pytest.mark.parametrize("n", [(160, 80, 90), (144, 128, 56), (256, 64, 64), (80, 64, 205), (72, 60, 41)])
@pytest.mark.parametrize("param", [0, 1])
def test_parameter_sum_of_its_own_tangent(lib, n, param):
    say(f"case parameter sums {lib.precision} n={n} param={param}")
    info = physics_info(lib, n)
    f = initial(lib, info, 5)
    tdt = torch.float32 if lib.precision == "fp32" else torch.float64
    dt, step = lib.np_real(0.5), 1
    with ac.Device(lib, info) as dev:
        ft = torch.from_numpy(f).cuda()
        torch.cuda.synchronize()
        ac.check(lib.acDeviceLoadMeshFromDevicePtr(dev.handle, 0, ft.data_ptr()), "load")
        dev.periodic()
        dev.sync()
        df, df_out, dw, lf = (torch.zeros(f.shape, dtype=tdt, device="cuda") for _ in range(4))
        ws = torch.full((int(lib.acAdjointWorkspaceBytes(dev.handle)),), 0xFF, dtype=torch.uint8, device="cuda")
        sums = torch.zeros(2, dtype=torch.float64, device="cuda")
        direction = (ctypes.c_double * 2)(*(1.0 if p == param else 0.0 for p in range(2)))
        torch.cuda.synchronize()
        ac.check(lib.acDeviceIntegrateSubstepTangent(dev.handle, 0, step, dt, df.data_ptr(), df_out.data_ptr(),
                                                     dw.data_ptr(), direction), "tangent")
        dev.sync()
        want = idot(dw, dw)
        ac.check(lib.acDeviceIntegrateSubstepAdjoint(dev.handle, 0, step, dt, lf.data_ptr(), dw.data_ptr(),
                                                     ws.data_ptr(), sums.data_ptr()), "adjoint")
        dev.sync()
        got = float(sums[param])
    say(f"  sum {got:.12g}  <dw', dw'> {want:.12g}  rel {abs(got - want) / want:.3g}")
    assert want > 0
    assert abs(got - want) < (1e-12 if lib.precision == "fp64" else 1e-5) * want
