"""What a run keeps per edge.  cvg_run_device_noalloc shows it: its scratch array
takes maps up to a number of edges that follows from the buffers' sizes."""
import numpy as np
import pytest

from curvelet_construction_on_gpu_amd import Context, CurveletParams
from curvelet_construction_on_gpu_amd.hip import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [180_000, 257_400])
def test_sparse_map_of_one_orientation_cell(n):
    """No neighbours and the smallest grid: the anchor lists are most of what is
    kept (256 bytes of 372 an edge, when each list had places for all anchors)."""
    i = np.arange(n)
    e = np.ascontiguousarray(np.stack([(i % 500) * 1.0, (i // 500) * 1.0, np.zeros(n), np.ones(n)], axis=1))
    with Context(0) as ctx:
        d = ctx.upload(e)
        chains, info = DeviceArray((16, 5), np.uint32), DeviceArray((16, 10), np.float64)
        assert ctx.run_device_noalloc(d, n, 4, CurveletParams(st=10.0, nrad=0.5), chains.ptr, info.ptr, 16) == (0, 0)
