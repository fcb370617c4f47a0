"""Maps whose anchors all take their own bounds (orientations or parameters
outside the approximate bounds' range): bit for bit against the oracle with
correctly rounded sin/cos and against the general kernel, at the edges of the
kernel's pieces: runs of 8 (mask growth, and the bundle slots in LDS), 16 pair
records, lists of 64 and 65 neighbours, one, two and four cells per lane, sines
in groups of 16 pairs down to one, offsets up to and beyond the 32 that share a
call with the first records.  There is no tolerance."""
import numpy as np
import pytest

from curvelet_construction_on_gpu_amd import Context, CurveletParams
from tests._inputs import edges_for
from tests.test_gpu_fused_kernel import lines
from tests.test_zz_no_alloc import bits, noalloc, pooled

pytestmark = pytest.mark.gpu

FAR = 2 * np.pi * 2.0 ** 20


@pytest.fixture(scope="module")
def both():
    """The context under test and one on the general kernel."""
    with pytest.MonkeyPatch.context() as m:
        under_test = Context()
        m.setenv("CVG_GENERIC_KERNEL", "1")
        general = Context()
    return under_test, general


def same_bits(both, oracle_cr, edges, p, route="direct"):
    want = oracle_cr.run(edges, p)
    counts = []
    for ctx, took in zip(both, (route, "general")):
        stats = ctx.run(edges, p)
        chains, info = ctx.curvelets()
        assert ctx.debug_route() == took
        assert stats["valid_pairs"] == want["valid_pairs"]
        assert np.array_equal(chains, want["chains"])
        assert np.array_equal(info.view(np.uint64), want["info"].view(np.uint64))
        counts.append(stats["intersections"])
    if p.group_max_sz > 2:
        assert counts[0] == counts[1]
    return stats


@pytest.mark.parametrize("group", [2, 3, 7, 12])
@pytest.mark.parametrize("run", [1, 2, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 100])
def test_run_lengths(both, oracle_cr, run, group):
    e = lines(run, seed=run)
    e[:, 2] += FAR
    same_bits(both, oracle_cr, e, CurveletParams(group_max_sz=group, max_candidates=256))


@pytest.mark.parametrize("group", [4, 9])
@pytest.mark.parametrize("run", [7, 8, 9, 16, 17, 40, 65, 100])
def test_run_lengths_on_larger_maps(both, oracle_cr, run, group):
    """More than four anchors a CU: eight slots in LDS, the other bundles in
    device memory (smaller maps have slots for whole lists)."""
    e = lines(run, seed=run, rows=2100 // (2 * run + 3))
    e[:, 2] += FAR
    assert len(e) > 1900
    same_bits(both, oracle_cr, e, CurveletParams(group_max_sz=group, max_candidates=256))


# kt = 1, 3, 7, 13, 31, 33, 45, 131
@pytest.mark.parametrize("sx,st", [(0.1, 10.0), (0.1, 0.16), (0.1, 0.08), (0.05, 0.08), (0.05, 0.04), (0.2, 0.0175),
                                   (0.2, 0.016), (0.4, 0.0117), (1.0, 0.004)])
@pytest.mark.parametrize("cand", [64, 65, 129])
def test_list_lengths_and_cells(both, oracle_cr, sx, st, cand):
    rng = np.random.default_rng(cand)
    e = np.stack([rng.uniform(0, 10, 420), rng.uniform(0, 10, 420), FAR + rng.uniform(0, 0.8, 420), np.ones(420)],
                 axis=1)
    same_bits(both, oracle_cr, e, CurveletParams(sx=sx, st=st, group_max_sz=6, max_candidates=cand))


@pytest.mark.parametrize("top", [4200.0, 1e6, 1e9, 1e15, 1e300])
def test_mixed_orientations(both, oracle_cr, top):
    """Neighbours at +top and -top, whose differences round the most."""
    e = lines(9, seed=5)
    e[::2, 2] += 2 * np.pi * np.floor(top / (2 * np.pi))
    e[1::2, 2] -= 2 * np.pi * np.floor(top / (2 * np.pi))
    same_bits(both, oracle_cr, e, CurveletParams(group_max_sz=7))


@pytest.mark.parametrize("dx,dt,max_k", [(0.4, 15.0, 1e5), (0.4, 15.0, np.inf), (0.4, 15.0, np.nan), (0.4, 15.0, 0.0),
                                         (0.4, 15.0, -0.3), (0.0, 15.0, 0.3),
                                         (-0.02, 15.0, 0.3), (1e-70, 15.0, 0.3), (0.4, 600.0, 0.3)])
def test_parameters(both, oracle_cr, dx, dt, max_k):
    rng = np.random.default_rng(7)
    e = np.stack([rng.uniform(0, 30, 500), rng.uniform(0, 30, 500), rng.uniform(-3, 3, 500), np.ones(500)], axis=1)
    e[1::25, :2] = e[::25, :2]  # some at the same place
    e[:, 2] += FAR if dx >= 0.0 and dt < 100.0 and 0.0 < max_k < 1.0 else 0.0
    same_bits(both, oracle_cr, e, CurveletParams(dx=dx, dt_deg=dt, max_k=max_k, st=0.08 if dt < 100.0 else 1.5))


@pytest.mark.parametrize("angle", [0.0, np.pi / 2, np.pi / 4])
def test_lattice(both, oracle_cr, angle):
    xs, ys = np.meshgrid(np.arange(12) * 1.0, np.arange(9) * 1.0)
    e = np.stack([xs.ravel(), ys.ravel(), np.full(xs.size, angle), np.ones(xs.size)], axis=1)
    for max_k in (1e5, 0.0):
        same_bits(both, oracle_cr, e, CurveletParams(max_k=max_k, group_max_sz=5))


@pytest.mark.parametrize("max_k,turns,route", [(1e-305, 0, "direct"), (5e-31, 0, "direct"),
                                               (1e-30, 0, "fused"), (1e-9, 0, "fused"), (1e-6, 0, "fused"), (1e-3, 100, "fused"),
                                               (0.05, 0, "fused"), (3000.0, 0, "fused"), (8000.0, 0, "direct"),
                                               (0.3, 650, "fused"), (0.3, 653, "direct")])
def test_where_the_route_changes(both, oracle_cr, max_k, turns, route):
    """On either side of the approximate bounds' range, on a map and on a
    lattice of it, whose bounds are often equal."""
    rng = np.random.default_rng(11)
    e = np.stack([rng.uniform(0, 30, 600), rng.uniform(0, 30, 600), rng.uniform(-3, 3, 600), np.ones(600)], axis=1)
    q = np.unique(np.rint(e[:, :2]), axis=0)
    lattice = np.concatenate([q, np.rint(e[:len(q), 2:3] * 4) / 4, np.ones((len(q), 1))], axis=1)
    for m in (e, lattice):
        m[:, 2] += 2 * np.pi * turns
        same_bits(both, oracle_cr, m, CurveletParams(max_k=max_k, group_max_sz=5), route)


@pytest.mark.parametrize("group", [4, 7])
def test_noalloc(group):
    e = np.array(edges_for("synth:C1:1001"))
    e[:, 2] += FAR
    p = CurveletParams(group_max_sz=group)
    with Context(0) as ctx:
        want_c, want_i, want_v = pooled(ctx, e, p)
        got_c, got_i, got_v = noalloc(ctx, e, p, len(want_c) + 3)
        assert ctx.debug_route() == "direct"
    assert got_v == want_v
    assert np.array_equal(got_c, want_c)
    assert np.array_equal(bits(got_i), bits(want_i))


def test_batch():
    """Each map of a batch that takes the direct kernel equals its lone run."""
    far = np.array(edges_for("synth:C1:1001"))
    far[:, 2] += FAR
    maps = [lines(9, seed=2), far, lines(70, seed=4)]
    p = CurveletParams(group_max_sz=6, max_candidates=256)
    with Context(0) as ctx:
        lone = []
        for m in maps:
            ctx.run(m, p)
            lone.append(ctx.curvelets())
        ctx.run_batch(maps, p)
        assert ctx.debug_route() == "direct"
        for k, (chains, info) in enumerate(lone):
            got_c, got_i = ctx.batch_curvelets(k)
            assert np.array_equal(got_c, chains)
            assert np.array_equal(bits(got_i), bits(info))
