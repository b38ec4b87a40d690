"""The monitoring of test_gpu_monitor_shapes.py on grids whose columns fill the chip's workgroups one and a bit times,
where the marching kernels split their planes into more chunks: FP64 517 columns, 66 planes in two chunks; FP32
422 columns, 128 planes in three ragged chunks."""
import pytest

from astaroth_amd import astaroth as ac
from tests import test_gpu_monitor_shapes as shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,n", [("fp64", (363, 364, 66)), ("fp32", (360, 300, 128))])
def test_monitoring_with_split_chunks(prec, n, require_gpu):
    shapes.test_monitoring_on_any_grid(ac.load(prec), n)
