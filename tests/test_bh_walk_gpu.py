"""The depth-first walk of batches with few segments a pair, against the
host-driven level-by-level schedule (timing = 1): the same node pairs visited,
far fields, leaf pairs and re-runs, and the same FP32 terms summed in another
order in FP64 (1e-9, as the other schedules' tests)."""
import numpy as np
import pytest

flk = pytest.importorskip("fastlinkingnumbers_amd")
from fastlinkingnumbers_amd import workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu

COUNTS = ("bh_visits", "bh_far", "bh_leaf_pairs", "retries")


def _check(engine, pairs, **kw):
    kw = dict(method="barneshut", fallback_tol=0.0, **kw)
    walked = engine.linking_numbers(pairs, **kw)
    levels = engine.linking_numbers(pairs, timing=1, **kw)
    assert walked.stats["bh_host_passes"] == 0 and levels.stats["bh_host_passes"] >= 1
    for key in COUNTS:
        assert walked.stats[key] == levels.stats[key], key
    np.testing.assert_allclose(walked.lk, levels.lk, rtol=0, atol=1e-9)
    np.testing.assert_allclose(walked.err, levels.err, rtol=1e-9, atol=1e-300)
    assert np.array_equal(walked.flags, levels.flags)
    return walked


@pytest.mark.parametrize("n,m", [(2, 2), (2, 3), (5, 4), (63, 65), (64, 1000), (1023, 1025), (9000, 700),
                                 (20000, 12000)])
def test_one_pair(engine, n, m):
    t, u = 2 * np.pi * np.arange(n) / n, 2 * np.pi * np.arange(m) / m
    a = np.stack([np.cos(t), np.sin(t), 0.05 * np.sin(5 * t)], 1)
    b = np.stack([1 + np.cos(u), 0.05 * np.cos(3 * u), np.sin(u)], 1)
    engine.set_curves([a, b])
    for leaf in (1, 4):
        _check(engine, [[0, 1], [1, 0]], leaf_size=leaf)


def test_tangled_pair_is_re_run(engine):
    """One root pair with much work: it spreads over every wave through the
    queues, and the adaptive re-run walks again."""
    engine.set_curves(W.random_walk_pair(seed=3, n=16000, rg=25.0, workload=3))
    assert _check(engine, [[0, 1]]).stats["retries"] == 1


@pytest.mark.parametrize("copies", [8, 1])
def test_many_pairs(engine, copies):
    """Chain mail; with every pair of curves (more than 4,096) the sums have one
    copy instead of eight."""
    curves = W.chainmail(seed=5, grid=10, nmin=16, nmax=700)
    engine.set_curves(curves)
    pairs = engine.potential_links() if copies == 8 else np.array(
        [(i, j) for i in range(100) for j in range(i + 1, 100)], dtype=np.int32)
    assert (len(pairs) <= 4096) == (copies == 8)
    _check(engine, pairs)


def test_overflow_goes_to_the_host(engine):
    engine.set_curves(W.random_walk_pair(seed=1, n=15000, rg=25.0, workload=3))
    kw = dict(method="barneshut", fallback_tol=0.0)
    base = engine.linking_numbers([[0, 1]], **kw)
    assert base.stats["bh_host_passes"] == 0
    for capacity in (64, 4096):
        engine.set_tune(bh_level_capacity=capacity)
        small = engine.linking_numbers([[0, 1]], **kw)
        assert small.stats["bh_host_passes"] >= 1
        for key in COUNTS:
            assert small.stats[key] == base.stats[key], key
        np.testing.assert_allclose(small.lk, base.lk, rtol=0, atol=1e-9)


def test_deep_stacks_stay_in_the_walk(engine):
    """Twenty tangled pairs, 360 node pairs a segment: in the last round the waves'
    stacks fill to the end and the steps narrow; nothing goes to the host."""
    curves = []
    for k in range(20):
        curves += [c + np.array([100.0 * k, 0, 0]) for c in W.random_walk_pair(seed=k, n=16000, rg=9.0, workload=3)]
    engine.set_curves(curves)
    pairs = [[2 * k, 2 * k + 1] for k in range(20)]
    first = _check(engine, pairs)
    for _ in range(3):
        again = engine.linking_numbers(pairs, method="barneshut", fallback_tol=0.0)
        assert again.stats["bh_host_passes"] == 0
        np.testing.assert_allclose(again.lk, first.lk, rtol=0, atol=1e-9)


def _rings(n, count, at):
    t = 2 * np.pi * np.arange(n) / n
    flat, tilted = (np.stack([np.cos(t), np.sin(t), 0 * t], 1), np.stack([np.cos(t), 0 * t, np.sin(t)], 1))
    return [(tilted if k % 2 else flat) + np.array([at + 1.4 * k, 0.0, 0.0]) for k in range(count)]


@pytest.mark.parametrize("n", [300000, 1500])
def test_one_large_pair_among_many_small(engine, n):
    """A dominant tangled pair takes the rounds it needs to spread over the chip:
    the batch costs little more than the pair and the rings by themselves (in six
    rounds 13 times as much for 300,000 segments a curve)."""
    curves = W.random_walk_pair(seed=7, n=n, rg=100.0 * np.sqrt(n / 2e6), workload=3) + _rings(200, 380, 1000.0)
    engine.set_curves(curves)
    pairs = engine.potential_links()
    assert len(pairs) > 300 and list(pairs[0]) == [0, 1]
    _check(engine, pairs)

    def fastest(p):
        return min(engine.linking_numbers(p, method="barneshut", fallback_tol=0.0).stats["ms_total"] for _ in range(5))

    parts, whole = fastest(pairs[:1]) + fastest(pairs[1:]), fastest(pairs)
    print(n, "parts", parts, "whole", whole)
    assert whole < 5 * parts


def test_the_leaf_list_is_used_up(engine):
    """A leaf list with room for every item holds them, though the segments' shares
    of it fill unevenly (some 20% over the mean here); one with too little goes to
    the host.  One pass: beta_limit leaves nothing to re-run."""
    curves = []
    for k in range(20):
        curves += [c + np.array([100.0 * k, 0, 0]) for c in W.random_walk_pair(seed=k, n=8000, rg=6.3, workload=3)]
    engine.set_curves(curves)
    pairs = [[2 * k, 2 * k + 1] for k in range(20)]
    kw = dict(method="barneshut", fallback_tol=0.0, beta_limit=2.0)
    base = engine.linking_numbers(pairs, **kw)
    leaves = base.stats["bh_leaf_pairs"]
    assert base.stats["retries"] == base.stats["bh_host_passes"] == 0 and leaves > 100000
    for room, passes in ((1.01, 0), (0.95, 1)):
        engine.set_tune(bh_level_capacity=int(room * leaves))
        for _ in range(3):
            got = engine.linking_numbers(pairs, **kw)
            assert got.stats["bh_host_passes"] == passes, room
            for key in COUNTS:
                assert got.stats[key] == base.stats[key], key
            np.testing.assert_allclose(got.lk, base.lk, rtol=0, atol=1e-9)
