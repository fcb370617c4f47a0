"""The helper threads of large downloads into pageable memory: they leave a
context that makes no more of them, and a later download is whole again."""
import os
import time

import numpy as np
import pytest

from curvelet_construction_on_gpu_amd import Context, CurveletParams, synth_edges

pytestmark = pytest.mark.gpu


def threads():
    return len(os.listdir("/proc/self/task"))


def test_helpers_leave_an_idle_context():
    e, p = synth_edges("C3", 1003), CurveletParams(group_max_sz=7)
    with Context(0) as ctx:
        ctx.run(e, p)
        before = threads()
        chains, info = ctx.curvelets()
        assert chains.nbytes > 1 << 20
        held = threads() - before
        deadline = time.monotonic() + 10.0
        while threads() > before and time.monotonic() < deadline:
            time.sleep(0.1)
        assert held > 0 and threads() <= before
        for _ in range(3):
            again, info2 = ctx.curvelets()
            assert np.array_equal(again, chains)
            assert np.array_equal(info2.view(np.uint64), info.view(np.uint64))
