"""Discretization with kept scratch and the guard's sums on the device: repeated
and mixed calls on one engine give what a fresh one gives, and the input guard
is the host restatement's at degenerate, NaN and one-segment inputs."""
import numpy as np
import pytest

flk = pytest.importorskip("fastlinkingnumbers_amd")

pytestmark = pytest.mark.gpu


def _rings(n, k, z):
    t = np.linspace(0, 2 * np.pi, n, endpoint=False)
    return [np.stack([i * 1.5 + np.cos(t), np.sin(t) * (1 if i % 2 else z), np.sin(t) * (z if i % 2 else 1)], 1)
            for i in range(k)]


@pytest.mark.parametrize("n,k", [(4, 2), (64, 3), (255, 5), (257, 4), (40, 300)])
def test_repeated_calls_match_a_fresh_engine(engine, n, k):
    curves = _rings(n, k, 0.01)
    pairs = [[i, i + 1] for i in range(k - 1)]
    engine.discretize(_rings(1000, 3, 0.1), flk.SEG_BSPLINE, True, [[0, 1]])  # larger scratch first
    for _ in range(2):
        for looped in (True, False):
            got, d = engine.discretize(curves, flk.SEG_BSPLINE, looped, pairs)
            fresh = flk.Engine(0)
            want, dw = fresh.discretize(curves, flk.SEG_BSPLINE, looped, pairs)
            fresh.close()
            assert d == dw
            assert all(np.array_equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("n", [3, 300, 70000])
def test_guard_names_the_first_smallest_segment(engine, n):
    t = np.linspace(0, 2 * np.pi, n, endpoint=False)
    a = np.stack([np.cos(t), np.sin(t), 0 * t], 1)
    bad = a.copy()
    bad[n // 2] = bad[n // 2 - 1]
    with pytest.raises(flk.FlkError, match="Smallest input segment"):
        engine.discretize([a, bad], flk.SEG_POLYLINE, True, [[0, 1]])
    # NaN: as the reference's loop, which takes it as smaller than anything
    nan = a.copy()
    nan[n - 1] = np.nan
    with pytest.raises(flk.FlkError, match="Smallest input segment"):
        engine.discretize([nan, a], flk.SEG_POLYLINE, True, [[0, 1]])
    # one unit above the threshold's order passes
    got, d = engine.discretize([a], flk.SEG_POLYLINE, True, np.zeros((0, 2), np.int32))
    assert d["segments"] == n and np.array_equal(got[0], a)


def test_scratch_beyond_the_kept_is_given_back(engine):
    """Two polylines of 2.5e6 segments take more than 1 GiB, which is given back,
    also when the input guard throws: the calls behind are a fresh engine's."""
    n = 2500000
    t = 2 * np.pi * np.arange(n) / n
    large = [np.stack([x + np.cos(t), np.sin(t), 0 * t], 1) for x in (0.0, 5.0)]
    none = np.zeros((0, 2), np.int32)
    small = _rings(300, 6, 0.01)
    pairs = [[i, i + 1] for i in range(5)]
    fresh = flk.Engine(0)
    want, dw = fresh.discretize(small, flk.SEG_BSPLINE, True, pairs)
    want_boxes = fresh.curve_boxes()
    fresh.close()
    bad = [large[0], large[1].copy()]
    bad[1][7] = bad[1][6]
    for attempt in ("whole", "guard"):
        if attempt == "whole":
            got, d = engine.discretize(large, flk.SEG_POLYLINE, True, none)
            assert d["segments"] == d["pieces"] == 2 * n
            assert all(np.array_equal(g, c) for g, c in zip(got, large))
        else:
            with pytest.raises(flk.FlkError, match="Smallest input segment"):
                engine.discretize(bad, flk.SEG_POLYLINE, True, none)
        got, d = engine.discretize(small, flk.SEG_BSPLINE, True, pairs)
        assert d == dw and all(np.array_equal(g, w) for g, w in zip(got, want)), attempt
        engine.set_curves(small)
        d = engine.discretize_current(flk.SEG_BSPLINE, True, pairs)
        assert d["pieces"] == dw["pieces"] and np.array_equal(engine.curve_boxes(), want_boxes), attempt
