"""An upload's boxes and vertices at the edges of their kernels: curves of one and
of several box chunks (4,096 vertices), empty and short ones among them, and
the one-block potential-link search at the ends of its range."""
import numpy as np
import pytest

flk = pytest.importorskip("fastlinkingnumbers_amd")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("sizes", [[1, 0, 2, 16384, 3], [16385, 0, 5], [0, 40000, 1, 16384], [0, 0]], ids=str)
def test_boxes_and_direct_sums(engine, sizes, dtype):
    """The boxes are the vertices' extrema exactly; a Hopf link appended behind
    the curves has its integer by either precision."""
    rng = np.random.default_rng(len(sizes))
    t = 2 * np.pi * np.arange(300) / 300
    ring = np.stack([np.cos(t), np.sin(t), 0 * t], 1) + 20
    curves = [rng.normal(size=(n, 3)) for n in sizes] + [ring, ring[:, [0, 2, 1]] * [1, 1, 1] + [1, 0, 0]]
    packed = np.concatenate(curves).astype(dtype)
    offsets = np.concatenate([[0], np.cumsum([len(c) for c in curves])])
    engine.set_curves_packed(packed, offsets)
    boxes = engine.curve_boxes()
    for k, (a, b) in enumerate(zip(offsets[:-1], offsets[1:])):
        if b > a:
            v = packed[a:b].astype(np.float64)
            assert np.array_equal(boxes[k], np.concatenate([v.min(0), v.max(0)])), k
    n = len(sizes)
    for fp64 in (0, 1):
        lk = engine.linking_numbers([[n, n + 1]], method="directsum", fp64=fp64, fallback_tol=0.0).lk[0]
        assert abs(abs(lk) - 1) < 1e-4, lk


@pytest.mark.parametrize("n", [2, 63, 64, 65, 128, 255, 256, 257])
def test_one_block_search_is_every_overlapping_pair(engine, n):
    """All pairs in ascending order; touching, empty and all-overlapping boxes,
    more pairs than the first pinned array holds among them."""
    rng = np.random.default_rng(n)
    lo = np.round(rng.uniform(0, 4, size=(n, 3)))
    for size in (0.0, 1.0, 10.0):
        boxes = np.concatenate([lo, lo + size], 1)
        boxes[n // 2] = [1, 1, 1, 0, 0, 0]  # empty
        i, j = np.triu_indices(n, 1)
        near = np.all((boxes[i, :3] <= boxes[j, 3:]) & (boxes[j, :3] <= boxes[i, 3:]), axis=1)
        assert np.array_equal(engine.potential_links(boxes), np.stack([i[near], j[near]], 1)), size


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("sizes", [[4096, 0, 4095, 1], [4097, 1, 0, 8193], [1024, 1025, 3]], ids=str)
def test_boxes_around_a_chunk(engine, sizes, dtype):
    """Curves within and beyond one chunk of 4,096 vertices, in whole and part
    rounds of a block's 1,024 threads; extrema at the ends."""
    rng = np.random.default_rng(sum(sizes))
    packed = rng.normal(size=(sum(sizes), 3)).astype(dtype)
    offsets = np.concatenate([[0], np.cumsum(sizes)])
    for a, b in zip(offsets[:-1], offsets[1:]):
        if b > a:
            packed[a], packed[b - 1] = -9, 9
    engine.set_curves_packed(packed, offsets)
    boxes = engine.curve_boxes()
    for k, (a, b) in enumerate(zip(offsets[:-1], offsets[1:])):
        if b > a:
            v = packed[a:b].astype(np.float64)
            assert np.array_equal(boxes[k], np.concatenate([v.min(0), v.max(0)])), k


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("mean", [3, 256, 257, 1000, 1100])
@pytest.mark.parametrize("longest", [0, 9000])
def test_boxes_of_many_curves(engine, mean, longest, dtype):
    """More than 1,024 curves: blocks of a wave, of four and of sixteen by the
    mean chunk, each over curves shorter and longer than its rounds (and, with
    one beyond a chunk, through the merge); empty ones among them."""
    rng = np.random.default_rng(mean + longest)
    sizes = rng.integers(0, 2 * mean, size=1300)
    sizes[:6] = [0, 1, 2 * mean, 255, 4 * 255 + 1, longest]
    packed = rng.normal(size=(sizes.sum(), 3)).astype(dtype)
    offsets = np.concatenate([[0], np.cumsum(sizes)])
    full = sizes > 0
    packed[offsets[:-1][full]], packed[offsets[1:][full] - 1] = -9, 9
    engine.set_curves_packed(packed, offsets)
    boxes = engine.curve_boxes()
    want = np.array([np.concatenate([v.min(0), v.max(0)]) for v in np.split(packed.astype(np.float64), offsets[1:-1])
                     if len(v)])
    assert np.array_equal(boxes[full], want)
    assert np.array_equal(engine.linking_numbers([[2, 3]], method="directsum", fp64=1).lk,
                          engine.linking_numbers([[2, 3]], method="directsum", fp64=1, graph=0).lk)
