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
