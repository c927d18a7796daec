"""The one-block sort of short curves' segments: at the edges of its runs, classes
and range (64, 1,024 and 8,192 segments) a tree's order is numpy's stable argsort
of the segments' Morton keys, as the segmented sort's is beyond it."""
import numpy as np
import pytest

flk = pytest.importorskip("fastlinkingnumbers_amd")

pytestmark = pytest.mark.gpu


def _spread(v):
    v = v & np.uint64(0x3FF)
    for shift, mask in ((16, 0x0000FF0000FF), (8, 0x00F00F00F00F), (4, 0x0C30C30C30C3), (2, 0x249249249249)):
        v = (v | (v << np.uint64(shift))) & np.uint64(mask)
    return v


@pytest.mark.parametrize("exact", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("sizes", [[2, 3, 63, 64, 65, 127, 128, 129], [1000, 1023, 1024, 1025, 2048, 2049],
                                   [8191, 8192, 100], [8193, 20000, 8192, 65]], ids=str)
def test_order_is_the_stable_sort_of_the_keys(engine, sizes, exact):
    """Points on a coarse grid, so that many keys are equal; the last set has
    curves of both sorts, each in a tree build of its own."""
    rng = np.random.default_rng(len(sizes))
    curves = [np.round(rng.normal(size=(n, 3)) * 6) / 8 + (0 if exact else rng.normal(size=(n, 3)) * 1e-13)
              for n in sizes]
    engine.set_curves(curves)
    largest = max(float(np.linalg.norm(c.max(0) - c.min(0))) for c in curves)
    scale = 2.0 ** -np.ceil(np.log2(2.0 * largest))
    for k, c in enumerate(curves):
        _, order = engine.tree_moments(k, leaf_size=1)
        p = c * scale
        m = 0.5 * (p + np.roll(p, -1, axis=0))
        lo, hi = p.min(0), p.max(0)
        inv = np.where(hi > lo, 1024.0 / np.where(hi > lo, hi - lo, 1.0), 0.0)
        cell = np.clip((m - lo) * inv, 0.0, 1023.0).astype(np.uint64)
        key = (_spread(cell[:, 0]) << np.uint64(2)) | (_spread(cell[:, 1]) << np.uint64(1)) | _spread(cell[:, 2])
        assert np.array_equal(order, np.argsort(key, kind="stable")), sizes[k]


def test_both_sorts_in_one_batch(engine):
    """A certificate over curves of both sorts: the integers of the direct sum."""
    t = lambda n: 2 * np.pi * np.arange(n) / n  # noqa: E731
    ring = lambda n, x: np.stack([np.cos(t(n)) + x, np.sin(t(n)), 0 * t(n)], 1)  # noqa: E731
    tilted = lambda n, x: np.stack([np.cos(t(n)) + x, 0 * t(n), np.sin(t(n))], 1)  # noqa: E731
    engine.set_curves([ring(500, 0.0), tilted(20000, 1.0), ring(5000, 2.0), tilted(64, 3.0)])
    pairs = engine.potential_links()
    ds = engine.linking_numbers(pairs, method="directsum")
    bh = engine.linking_numbers(pairs, method="barneshut", fallback_tol=0.0)
    assert np.array_equal(np.round(ds.lk), np.round(bh.lk)) and np.abs(np.round(ds.lk)).sum() == 3
