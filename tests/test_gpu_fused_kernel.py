"""The fused curvelet kernel (approximate bounds with certified comparisons,
mask growth for short runs) where its branches meet, bit for bit against the
oracle with correctly rounded sin/cos: run lengths around the 8 of the mask
growth, the 14 bundle slots in LDS and the 64 seeds of a word; neighbour
lists around the 64 of the main kernel; one, two and four cells per lane;
lattices, whose comparisons are equalities in exact arithmetic and go to the
exact bounds; orientations on both sides of the error bound's range, beyond
which the general kernel runs.  Whole numbers and bits are compared: there is
no tolerance."""
import numpy as np
import pytest

from curvelet_construction_on_gpu_amd import Context, CurveletParams
from oracle import OracleF32

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def both():
    """The context under test and one on the general kernel."""
    with pytest.MonkeyPatch.context() as m:
        fused = Context()
        m.setenv("CVG_GENERIC_KERNEL", "1")
        general = Context()
    return fused, general


def same_bits(both, oracle_cr, edges, p):
    want = oracle_cr.run(edges, p)
    counts = []
    for ctx in both:
        stats = ctx.run(edges, p)
        chains, info = ctx.curvelets()
        assert stats["valid_pairs"] == want["valid_pairs"]
        assert np.array_equal(chains, want["chains"])
        assert np.array_equal(info.view(np.uint64), want["info"].view(np.uint64))
        counts.append(stats["intersections"])
    if p.group_max_sz > 2:  # (below, no chain can be long enough and the fused kernel tests none)
        assert counts[0] == counts[1]
    return stats


def lines(run, seed, rows=3):
    """Rows of edges along x, `run` of them within the radius on either side
    of an inner edge, close to a common curve (so that most pairs hold)."""
    rng = np.random.default_rng(seed)
    step = 3.4 / run
    m = 2 * run + 3
    out = []
    for r in range(rows):
        x = 5.0 + np.arange(m) * step
        y = 5.0 + 20.0 * r + 0.01 * (x - 5.0) ** 2 + rng.uniform(-0.04, 0.04, m)
        th = np.arctan(0.02 * (x - 5.0)) + rng.uniform(-0.05, 0.05, m) + (np.pi if r == 1 else 0.0)
        out.append(np.stack([x, y, th, np.ones(m)], axis=1))
    return np.concatenate(out)


@pytest.mark.parametrize("group", [2, 3, 7, 12])
@pytest.mark.parametrize("run", [1, 2, 7, 8, 9, 13, 14, 15, 31, 32, 33, 63, 64, 65, 100])
def test_run_lengths(both, oracle_cr, run, group):
    stats = same_bits(both, oracle_cr, lines(run, seed=run), CurveletParams(group_max_sz=group, max_candidates=256))
    assert stats["max_num_of_neighbors"] >= run


@pytest.mark.parametrize("sx,st", [(0.1, 0.08), (0.05, 0.08), (0.05, 0.04)])  # 1, 2 and 4 cells per lane
@pytest.mark.parametrize("cand", [64, 65, 128, 129])
def test_list_lengths_and_cells(both, oracle_cr, sx, st, cand):
    rng = np.random.default_rng(cand)
    e = np.stack([rng.uniform(0, 10, 420), rng.uniform(0, 10, 420), rng.uniform(0, 0.8, 420), np.ones(420)], axis=1)
    stats = same_bits(both, oracle_cr, e, CurveletParams(sx=sx, st=st, group_max_sz=6, max_candidates=cand))
    assert stats["max_num_of_neighbors"] >= min(cand, 100)


@pytest.mark.parametrize("angle", [0.0, np.pi / 2, np.pi / 4])
@pytest.mark.parametrize("sx,st", [(0.1, 0.08), (0.05, 0.04)])
def test_equal_bounds(both, oracle_cr, angle, sx, st):
    xs, ys = np.meshgrid(np.arange(12) * 1.0, np.arange(9) * 1.0)
    e = np.stack([xs.ravel(), ys.ravel(), np.full(xs.size, angle), np.ones(xs.size)], axis=1)
    same_bits(both, oracle_cr, e, CurveletParams(sx=sx, st=st, group_max_sz=5))


@pytest.mark.parametrize("top", [63.9, 64.0, 64.1, 500.0, 4095.9, 4096.0, 4096.1, 1e5])
def test_orientation_range(both, oracle_cr, top):
    e = lines(6, seed=3)
    e[:, 2] += 2 * np.pi * np.floor((top - e[:, 2].max()) / (2 * np.pi))
    e[0, 2] = top
    same_bits(both, oracle_cr, e, CurveletParams(group_max_sz=7))


@pytest.mark.parametrize("dx,dt,max_k,nrad", [(0.4, 15.0, 0.3, 3.5), (0.2, 2.0, 2.0, 3.0), (1.5, 40.0, 0.05, 5.0),
                                              (0.4, 15.0, 1e-6, 3.5), (0.4, 15.0, 1e-3, 3.5),
                                              (0.4, 15.0, 1e4, 3.5)])
def test_parameter_range(both, oracle_cr, dx, dt, max_k, nrad):
    rng = np.random.default_rng(7)
    e = np.stack([rng.uniform(0, 30, 500), rng.uniform(0, 30, 500), rng.uniform(-3, 3, 500), np.ones(500)], axis=1)
    same_bits(both, oracle_cr, e, CurveletParams(dx=dx, dt_deg=dt, max_k=max_k, nrad=nrad, sx=dx / 4))


@pytest.fixture(scope="module")
def oracle_f32_cr():
    return OracleF32(cr=True)


def same_bits_float(both, oracle_f32_cr, edges, p):
    e = np.ascontiguousarray(edges, dtype=np.float32)
    want = oracle_f32_cr.run(e, p)
    counts = []
    for ctx in both:
        stats = ctx.run_f32(e, p)
        chains, info = ctx.curvelets()
        assert stats["valid_pairs"] == want["valid_pairs"]
        assert np.array_equal(chains, want["chains"])
        assert np.array_equal(info.view(np.uint64), want["info"].view(np.uint64))
        counts.append(stats["intersections"])
    assert counts[0] == counts[1]


@pytest.mark.parametrize("group", [2, 3, 7, 12])
@pytest.mark.parametrize("run", [1, 2, 8, 9, 14, 15, 32, 33, 65])
def test_float_run_lengths(both, oracle_f32_cr, run, group):
    same_bits_float(both, oracle_f32_cr, lines(run, seed=run), CurveletParams(group_max_sz=group, max_candidates=256))


@pytest.mark.parametrize("sx,st", [(0.1, 0.08), (0.05, 0.08), (0.05, 0.04)])
@pytest.mark.parametrize("cand", [64, 65])
def test_float_list_lengths_and_cells(both, oracle_f32_cr, sx, st, cand):
    rng = np.random.default_rng(cand)
    e = np.stack([rng.uniform(0, 10, 420), rng.uniform(0, 10, 420), rng.uniform(0, 0.8, 420), np.ones(420)], axis=1)
    same_bits_float(both, oracle_f32_cr, e, CurveletParams(sx=sx, st=st, group_max_sz=6, max_candidates=cand))


@pytest.mark.parametrize("angle", [0.0, np.pi / 2, np.pi / 4])
def test_float_equal_bounds(both, oracle_f32_cr, angle):
    xs, ys = np.meshgrid(np.arange(12) * 1.0, np.arange(9) * 1.0)
    e = np.stack([xs.ravel(), ys.ravel(), np.full(xs.size, angle), np.ones(xs.size)], axis=1)
    same_bits_float(both, oracle_f32_cr, e, CurveletParams(group_max_sz=5))


@pytest.mark.parametrize("top", [63.9, 64.0, 64.1, 1e5])
def test_float_orientation_range(both, oracle_f32_cr, top):
    e = lines(6, seed=3)
    e[:, 2] += 2 * np.pi * np.floor((top - e[:, 2].max()) / (2 * np.pi))
    e[0, 2] = top
    same_bits_float(both, oracle_f32_cr, e, CurveletParams(group_max_sz=7))


@pytest.mark.parametrize("dx,dt,max_k,nrad", [(0.2, 2.0, 2.0, 3.0), (1.5, 40.0, 0.05, 5.0), (0.4, 15.0, 1e-6, 3.5),
                                              (0.4, 15.0, 1e4, 3.5), (12.0, 15.0, 0.3, 3.5)])
def test_float_parameter_range(both, oracle_f32_cr, dx, dt, max_k, nrad):
    rng = np.random.default_rng(7)
    e = np.stack([rng.uniform(0, 30, 500), rng.uniform(0, 30, 500), rng.uniform(-3, 3, 500), np.ones(500)], axis=1)
    same_bits_float(both, oracle_f32_cr, e, CurveletParams(dx=dx, dt_deg=dt, max_k=max_k, nrad=nrad, sx=dx / 4))
