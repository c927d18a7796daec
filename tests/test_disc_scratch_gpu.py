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
