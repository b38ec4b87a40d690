"""The column form of the adjoint's local stage in FP64, on grids that 64 x 4 columns divide: at its shortest chunk
(8 planes), at one of 10, beside the line (4 planes, where blocks run), and on the smallest grid where it also takes
upwinding with entropy: <T(dx), y> = <dx, A(y)> with the tangent substep, and repeated runs bit for bit."""
import pytest

from astaroth_amd import astaroth as ac
from tests.test_gpu_adjoint import initial, physics_info, say, substep_dot_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(128, 64, 64), (64, 256, 40), (64, 64, 64), (256, 64, 216)])
@pytest.mark.parametrize("upwd,entropy,step", [(False, True, 0), (True, False, 1), (False, False, 2), (True, True, 1)])
def test_columns_in_fp64(n, upwd, entropy, step, require_gpu):
    say(f"case adjoint columns fp64 n={n} upwd={upwd} entropy={entropy} step={step}")
    lib = ac.load("fp64")
    info = physics_info(lib, n, AC_lupwd=upwd, AC_lentropy=entropy)
    f = initial(lib, info, 3 + step)
    runs = [substep_dot_product(lib, info, f, step, entropy, 7 + step) for _ in range(2)]
    assert runs[0][2] < 1e-12
    assert runs[0][:3] == runs[1][:3] and bool((runs[0][3] == runs[1][3]).all())
