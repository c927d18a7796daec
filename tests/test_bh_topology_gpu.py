"""The device trees' shape (segment ranges and children, computed for every node
at once from its curve's segment count) against the construction it stands for:
level by level, every range of more than `leaf` segments split into the lower
half, rounded down, and the rest, nodes numbered as they come (reference
src/compute_link.cpp:294-332 splits its ranges the same way)."""
import numpy as np
import pytest

flk = pytest.importorskip("fastlinkingnumbers_amd")

pytestmark = pytest.mark.gpu


def _level_by_level(n, leaf):
    ranges, children, level, total = [], [], [(0, n)], 1
    while level:
        below = []
        for lo, hi in level:
            ranges.append((lo, hi - lo))
            if hi - lo > leaf:
                mid = lo + (hi - lo) // 2
                children.append((total + len(below), total + len(below) + 1))
                below += [(lo, mid), (mid, hi)]
            else:
                children.append((-1, -1))
        total += len(below)
        level = below
    return np.array(ranges), np.array(children)


@pytest.mark.parametrize("leaf", [1, 2, 3, 5, 8])
def test_tree_shape_is_the_level_by_level_construction(engine, leaf):
    """Powers of two and their neighbours, odd sizes, curves that are one leaf;
    the trees of several curves in one batch are compared through their pairs'
    results elsewhere."""
    sizes = [2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 33, 100, 127, 128, 129, 255, 256, 257, 1000, 4097]
    rng = np.random.default_rng(leaf)
    engine.set_curves([rng.normal(size=(n, 3)) for n in sizes])
    for c, n in enumerate(sizes):
        nodes, _ = engine.tree_moments(c, leaf_size=leaf)
        ranges, children = _level_by_level(n, leaf)
        assert np.array_equal(np.stack([nodes["seg0"], nodes["nseg"]], 1), ranges), n
        assert np.array_equal(nodes["child"], children), n


@pytest.mark.parametrize("leaf", [1, 3])
def test_many_curves_in_one_batch(engine, leaf):
    """More than 256 curves, those of both sorts interleaved: a curve's tree is the
    same in any batch, so the batch's node pairs and values are those of its pairs
    built and walked one by one."""
    rng = np.random.default_rng(leaf)
    curves, pairs = [], []
    for k in range(150):
        sizes = rng.integers(2, 400, size=2)
        if k % 10 == 4:
            sizes[k // 10 % 2] = rng.choice([1024, 1025, 4097, 8192, 8193, 9000, 20000])
        t, u = (2 * np.pi * np.arange(n) / n for n in sizes)
        curves.append(np.stack([3.0 * k + np.cos(t), np.sin(t), 0.1 * np.sin(3 * t + k)], 1))
        curves.append(np.stack([3.0 * k + 1 + np.cos(u), 0.1 * np.cos(2 * u), np.sin(u)], 1))
        pairs.append((2 * k, 2 * k + 1) if k % 3 else (2 * k + 1, 2 * k))
    engine.set_curves(curves)
    kw = dict(method="barneshut", fallback_tol=0.0, leaf_size=leaf)
    batch = engine.linking_numbers(pairs, **kw)
    single = [engine.linking_numbers([p], graph=0, **kw) for p in pairs]
    for key in ("bh_visits", "bh_far", "bh_leaf_pairs", "retries"):
        assert batch.stats[key] == sum(s.stats[key] for s in single), key
    np.testing.assert_allclose(batch.lk, [s.lk[0] for s in single], rtol=0, atol=1e-9)
    np.testing.assert_allclose(batch.err, [s.err[0] for s in single], rtol=1e-9, atol=1e-300)
