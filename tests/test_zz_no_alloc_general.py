"""cvg_run_device_noalloc where the general curvelet kernel runs (orientations
beyond the fused kernel's error bound, long chains): its per-wave buffers fit
what the scratch array has left, and the bits are the pooled run's."""
import numpy as np
import pytest

from curvelet_construction_on_gpu_amd import Context, CurveletParams
from tests._inputs import edges_for
from tests.test_zz_no_alloc import bits, noalloc, pooled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turns,group", [(16, 4), (-16, 7), (0, 65)])
def test_noalloc_on_the_general_kernel(turns, group):
    e = np.array(edges_for("synth:C1:1001"))
    e[:, 2] += 2 * np.pi * turns
    if group > 64:
        e = e[:2500]
    e = np.ascontiguousarray(e)
    p = CurveletParams(group_max_sz=group)
    ctx = Context(0)
    want_c, want_i, want_v = pooled(ctx, e, p)
    got_c, got_i, got_v = noalloc(ctx, e, p, len(want_c) + 3)
    assert got_v == want_v
    assert np.array_equal(got_c, want_c)
    assert np.array_equal(bits(got_i), bits(want_i))
    ctx.close()
