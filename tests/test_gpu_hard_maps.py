"""Maps whose distances, bounds, orientations or parameters put the kernels on
their slower branches: the time stays of the order of an ordinary map's of the
same size (the shortest of several runs, against a factor far above what is
measured and far below what the fault behind each test cost)."""
import numpy as np
import pytest

from curvelet_construction_on_gpu_amd import Context, CurveletParams, synth_edges

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return Context()


@pytest.fixture(scope="module")
def frame():
    return synth_edges("C3", 1003)


def on_pixels(e):
    """The map at whole pixels, one edge each."""
    e = e.copy()
    e[:, :2] = np.rint(e[:, :2])
    _, first = np.unique(e[:, :2], axis=0, return_index=True)
    return np.ascontiguousarray(e[np.sort(first)])


def shortest(ctx, e, p, key, runs=7):
    return min(ctx.run(e, p)[key] for _ in range(runs))


def test_graph_of_tied_distances(ctx, frame):
    """Nearly every list has exact ties; the fill took 1,100 us of it (about
    100 without ties) while tied places were written twice."""
    p = CurveletParams()
    e = on_pixels(frame)
    apart = e.copy()
    apart[:, :2] += np.random.default_rng(1).uniform(-0.3, 0.3, (len(e), 2))
    assert shortest(ctx, e, p, "ms_graph") < 3.0 * shortest(ctx, apart, p, "ms_graph")


def theta_zero(e):
    e = on_pixels(e)
    e[:, 2] = 0.0
    return e


def sixteen_thetas(e):
    e = on_pixels(e)
    e[:, 2] = np.rint(e[:, 2] / (np.pi / 8)) * (np.pi / 8)
    return e


@pytest.mark.parametrize("make,changes", [(theta_zero, {}), (sixteen_thetas, {}), (np.copy, {"max_k": 1e-3}),
                                          (np.copy, {"max_k": 1e6})])
def test_curvelets_of_open_anchors(ctx, frame, make, changes):
    """Comparisons that the approximate bounds leave open, at most anchors.  256
    waves, one for each of them at a time, took 8 to 85 times an ordinary map's time."""
    ordinary = shortest(ctx, frame, CurveletParams(group_max_sz=7), "ms_curvelets")
    assert shortest(ctx, make(frame), CurveletParams(group_max_sz=7, **changes), "ms_curvelets") < 6.0 * ordinary


def test_float_curvelets_of_open_anchors(ctx, frame):
    """Sines of exactly zero: 13 times an ordinary map's time before."""
    p = CurveletParams()
    e = np.ascontiguousarray(frame[::2], dtype=np.float32)
    flat = e.copy()
    flat[:, 2] = 0.0
    run = lambda m: min(ctx.run_f32(m, p)["ms_curvelets"] for _ in range(7))
    assert run(flat) < 6.0 * run(e)


def turned(e):
    e = e.copy()
    e[:, 2] += 2 * np.pi * 1000
    return e


@pytest.mark.parametrize("make,changes", [(turned, {}), (np.copy, {"max_k": 1e-6}), (np.copy, {"max_k": 0.0})])
def test_curvelets_outside_the_approximations(ctx, frame, make, changes):
    """Orientations and parameters that the approximate bounds do not cover: 11
    to 18 times an ordinary map's time on the general kernel."""
    ordinary = shortest(ctx, frame, CurveletParams(group_max_sz=7), "ms_curvelets")
    assert shortest(ctx, make(frame), CurveletParams(group_max_sz=7, **changes), "ms_curvelets") < 6.0 * ordinary


@pytest.mark.parametrize("max_k", [0.02, 0.05, 0.1])
def test_bounds_beyond_a_small_max_k(ctx, frame, max_k):
    """Most bundles reach beyond max_k on both sides; none of those is close to
    anything.  Their anchors were all left open: 2.5 times the ordinary time."""
    ordinary = shortest(ctx, frame, CurveletParams(group_max_sz=7), "ms_curvelets")
    assert shortest(ctx, frame, CurveletParams(group_max_sz=7, max_k=max_k), "ms_curvelets") < 1.5 * ordinary


@pytest.mark.parametrize("max_k", [1e-4, 1e5])
def test_extreme_max_k(ctx, frame, max_k):
    """Small: the approximate bounds still settle most anchors.  Large: their
    units are too coarse, and the direct kernel takes all anchors at once."""
    ordinary = shortest(ctx, frame, CurveletParams(group_max_sz=7), "ms_curvelets")
    assert shortest(ctx, frame, CurveletParams(group_max_sz=7, max_k=max_k), "ms_curvelets") < 3.5 * ordinary
    assert ctx.debug_route() == ("fused" if max_k < 1.0 else "direct")


@pytest.mark.parametrize("make", [theta_zero, sixteen_thetas])
def test_curvelets_on_whole_pixels(ctx, frame, make):
    """Neighbours exactly across the anchor's direction: with none of their
    classes settled by the fused kernel, 2.0 and 1.0 times the ordinary time."""
    ordinary = shortest(ctx, frame, CurveletParams(group_max_sz=7), "ms_curvelets")
    assert shortest(ctx, make(frame), CurveletParams(group_max_sz=7), "ms_curvelets") < 0.9 * ordinary


def test_no_positive_max_k(ctx, frame):
    """No curvelet can exist: 1.4 times the ordinary time while bundles were formed."""
    ordinary = shortest(ctx, frame, CurveletParams(group_max_sz=7), "ms_curvelets")
    assert shortest(ctx, frame, CurveletParams(group_max_sz=7, max_k=0.0), "ms_curvelets") < ordinary
