"""The discretization's walk for overlapping pieces: what it finds does not
depend on where the model lies, how large it is, or the curves' order."""
import re
import time

import numpy as np
import pytest

import oracle as O

flk = pytest.importorskip("fastlinkingnumbers_amd")

pytestmark = pytest.mark.gpu


def _polygons(na, nb):
    """Two linked polygons whose first segments each span most of the model on
    every axis, 0.4 apart where they cross."""
    a = np.array([[-1, -1, -1], [1, 1, 1]], float)
    b = np.array([[-1, 1, 0.8], [1, -1, -1.1]], float) + [0.3, 0.3, 0]
    arc = lambda p, q, n, bend: [p + (q - p) * t + bend * np.sin(np.pi * t)  # noqa: E731
                                 for t in np.arange(n) / n]
    return [np.array([a[0], *arc(a[1], a[0], na - 1, np.array([2.0, -2.0, 0.3]))]),
            np.array([b[0], *arc(b[1], b[0], nb - 1, np.array([-1.5, -1.5, 0.4]))])]


# numbers of pieces that are not powers of two, so the tree has padding; beyond
# 2^128 a box that holds the origin is every FP32 number once rounded outward
@pytest.mark.parametrize("na,nb", [(3, 4), (5, 6), (60, 201)])
def test_models_beyond_fp32(engine, na, nb):
    curves = _polygons(na, nb)
    ref = O.Model.from_curves(curves).discretize().curves()
    unit, du = engine.discretize(curves, flk.SEG_POLYLINE, True, [[0, 1]])
    assert du["rounds"] > 1 and du["overlaps"][0] > 0 and du["overlaps"][-1] == 0
    assert [len(c) for c in unit] == [len(c) for c in ref]
    for u, r in zip(unit, ref):
        np.testing.assert_allclose(u, r, rtol=0, atol=1e-12)
    big, db = engine.discretize([2.0 ** 130 * c for c in curves], flk.SEG_POLYLINE, True, [[0, 1]])
    assert db == du
    for u, b in zip(unit, big):  # a power of two changes no rounding
        np.testing.assert_array_equal(b, 2.0 ** 130 * u)


def _rings(n, rows, columns):
    """Chain mail of rows x columns rings of n points, on a grid of 2^-20."""
    t = 2 * np.pi * np.arange(n) / n
    out = []
    for k in range(rows * columns):
        i, j = divmod(k, columns)
        s = 1 if (i + j) % 2 else -1
        x = np.stack([1.5 * i + np.cos(t), 1.5 * j + 0.7 * np.sin(t), 0.7 * s * np.sin(t) + 0.05 * np.sin(3 * t + k)], 1)
        out.append(np.round(x * 2.0 ** 20) / 2.0 ** 20)
    return out


def _timed(engine, curves, seg_type=None):
    """The discretization of curves that are on the device, and the fastest of five."""
    best = np.inf
    for _ in range(5):
        engine.set_curves(curves)
        pairs = engine.potential_links()
        start = time.perf_counter()
        d = engine.discretize_current(flk.SEG_POLYLINE if seg_type is None else seg_type, True, pairs)
        best = min(best, time.perf_counter() - start)
    return d, best


def test_model_far_from_the_origin(engine):
    """At 2^23 an FP32 number is 1 from the next, more than a hundred segments'
    length: the same rounds, and no longer than at the origin (17 times as long
    with boxes about 0)."""
    curves = _rings(400, 16, 16)
    near, t_near = _timed(engine, curves)
    far, t_far = _timed(engine, [c + 2.0 ** 23 for c in curves])
    print("near", t_near, "far", t_far)
    assert far == near
    assert t_far < 2 * t_near
    few = [c + 2.0 ** 23 for c in _rings(60, 3, 4)]
    m = O.Model.from_curves(few)
    got, _ = engine.discretize(few, flk.SEG_POLYLINE, True, m.pls())
    assert [len(c) for c in got] == [len(c) for c in m.discretize().curves()]


@pytest.mark.parametrize("rows,columns,n", [(5, 7, 33), (70, 70, 60)])
def test_order_of_the_curves(engine, rows, columns, n):
    """Curves in random order: the same rounds and polylines, and no longer (55
    times as long when a query walked every piece behind its curve)."""
    curves = _rings(n, rows, columns)
    perm = np.random.default_rng(1).permutation(len(curves))
    ordered, t_ordered = _timed(engine, curves)
    shuffled, t_shuffled = _timed(engine, [curves[k] for k in perm])
    print("ordered", t_ordered, "shuffled", t_shuffled, ordered["rounds"])
    assert shuffled == ordered
    assert t_shuffled < 3 * t_ordered
    if rows == 5:
        pairs = O.Model.from_curves(curves).pls()
        want, _ = engine.discretize(curves, flk.SEG_BSPLINE, True, pairs)
        back = np.argsort(perm)
        got, _ = engine.discretize([curves[k] for k in perm], flk.SEG_BSPLINE, True, back[pairs])
        assert all(np.array_equal(got[back[k]], w) for k, w in enumerate(want))


def _through_one_another(count, n):
    """Closed curves of two modes a coordinate, all about the origin."""
    t = 2 * np.pi * np.arange(n) / n
    out = []
    for k in range(count):
        g = np.random.default_rng([7, k])
        out.append(sum(g.normal(size=3) / m * np.cos(m * t[:, None] + g.uniform(0, 6.28, 3)) for m in (1, 2)))
    return out


# up to 32 partners of a curve are asked one by one, beyond that the pieces are sorted
@pytest.mark.parametrize("looped", [True, False])
@pytest.mark.parametrize("count,n", [(12, 100), (33, 40), (34, 40), (70, 25), (80, 23), (80, 150)])
def test_many_partners(engine, capfd, count, n, looped):
    curves = _through_one_another(count, n) + [c + [9.0, 0, 0] for c in _through_one_another(2, 9)]
    m = O.Model.from_curves(curves, looped=looped)
    pairs = m.pls()
    capfd.readouterr()
    ref = m.discretize().curves()
    overlaps = [int(x) for x in re.findall(r"Iteration \d+, (\d+) overlaps", capfd.readouterr().out)]
    got, d = engine.discretize(curves, flk.SEG_POLYLINE, looped, pairs)
    assert d["overlaps"] == overlaps
    assert [len(c) for c in got] == [len(c) for c in ref]
    for a, b in zip(got, ref):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-12)
