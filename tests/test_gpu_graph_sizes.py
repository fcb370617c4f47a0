"""The neighbour graph on guessed sizes, where a map counts its lists in the
fill (up to 65,536 edges) or before it, and the list ranks with and without
exact distance ties: the same CSR and curvelets, bit for bit, as a context
that reads every size first; repeated maps, a denser map after a sparse one
(whose guess misses) and lists of more than 16 entries."""
import numpy as np
import pytest

from curvelet_construction_on_gpu_amd import Context, CurveletParams, synth_edges

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def both():
    """A context that guesses sizes and one that reads them."""
    with pytest.MonkeyPatch.context() as m:
        guessing = Context()
        m.setenv("CVG_SPECULATE", "0")
        reading = Context()
    return guessing, reading


def same(both, edges, p):
    got = []
    for ctx in both:
        ctx.run(edges, p)
        g = ctx.graph()
        chains, info = ctx.curvelets()
        got.append((np.array(g.neighbor_offsets), np.array(g.neighbor_ids), g.neighbor_dist2.view(np.uint64), chains,
                    info.view(np.uint64)))
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def tiled(n, seed):
    base = synth_edges("C2", 1000 + seed)
    reps = -(-n // len(base))
    out = np.concatenate([base + np.array([700.0 * (k % 3), 520.0 * (k // 3), 0.0, 0.0]) for k in range(reps)])
    return np.ascontiguousarray(out[:n])


@pytest.mark.parametrize("n", [63, 65535, 65536, 65537, 90001])
def test_sizes(both, n):
    p = CurveletParams(group_max_sz=4)
    same(both, tiled(n, 1), p)
    same(both, tiled(n, 1), p)
    same(both, tiled(n, 2), p)


@pytest.mark.parametrize("n", [300, 70000])
def test_denser_map_after_a_sparse_one(both, n):
    rng = np.random.default_rng(n)
    side = np.sqrt(n) * 2.0
    for scale in (1.0, 0.45, 1.0):
        e = np.stack([rng.uniform(0, side * scale, n), rng.uniform(0, side * scale, n), rng.uniform(0, 3.1, n),
                      np.ones(n)], axis=1)
        same(both, e, CurveletParams(group_max_sz=4))


@pytest.mark.parametrize("cand", [5, 16, 17, 128])
@pytest.mark.parametrize("nx,ny", [(40, 30), (270, 250)])
def test_tied_distances(both, nx, ny, cand):
    xs, ys = np.meshgrid(np.arange(nx) * 1.0, np.arange(ny) * 1.0)
    rng = np.random.default_rng(nx)
    e = np.stack([xs.ravel(), ys.ravel(), rng.uniform(0, 3.1, xs.size), np.ones(xs.size)], axis=1)
    e[::3, 0] += 0.25 * (rng.integers(0, 3, len(e[::3])))
    for _ in range(2):
        same(both, e, CurveletParams(group_max_sz=4, max_candidates=cand))
