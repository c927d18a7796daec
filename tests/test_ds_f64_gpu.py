"""The FP64 tile kernel at the sizes where its rows (2 per lane, 128 per wave),
columns (two per iteration, chunks of a multiple of 64) and general path can go
wrong, against the FP64 oracle.

Tolerance 1e-12 per pair: a pair of at most 1,100 x 700 segments sums 8e5
angles.  An angle's rounding error is that of its triple product, about 1e-16
r^3 in the oracle (a product of three relative vectors), over x' ~ 8 r^3, so
below 1e-16, and 8e5 of them (random signs) stay below 1e-13 even times ten.
"""
import numpy as np
import pytest

import oracle as O

flk = pytest.importorskip("fastlinkingnumbers_amd")

pytestmark = pytest.mark.gpu


def _ring(n, centre, tilt, wobble, seed):
    g = np.random.default_rng(seed)
    t = 2 * np.pi * np.arange(n) / n
    r = 1 + wobble * np.cos(3 * t + g.uniform(0, 6))
    x = np.stack([r * np.cos(t), r * np.sin(t), wobble * np.sin(2 * t)], 1)
    c, s = np.cos(tilt), np.sin(tilt)
    return x @ np.array([[1, 0, 0], [0, c, s], [0, -s, c]]) + centre


@pytest.mark.parametrize("n,m", [(2, 2), (3, 2), (5, 4), (63, 64), (65, 3), (127, 31), (128, 33), (129, 128),
                                 (255, 63), (257, 65), (600, 511), (1100, 513), (1025, 700)])
def test_remainders_match_oracle(engine, n, m):
    a = _ring(n, [0, 0, 0], 0.0, 0.07, n)
    b = _ring(m, [0.9, 0.1, 0.2], 1.3, 0.05, m)
    engine.set_curves([a, b])
    got = engine.linking_numbers([[0, 1], [1, 0]], method="directsum", fp64=1).lk
    ref = O.ds(a, b)
    print(n, m, "got", got, "oracle", ref)
    assert np.abs(got - ref).max() < 1e-12


@pytest.mark.parametrize("gap", [1e-2, 1e-5, 1e-9])
def test_near_misses_take_the_general_path(engine, gap):
    """Curves passing each other at `gap` of their size: large angles and small
    denominators, mixed with the short path's columns in the same wave.  The
    oracle's triple products then err by 1e-16 of pairs whose angle is pi, over
    x' ~ gap^2 times the segments' squares: 1e-16 / gap."""
    a = _ring(300, [0, 0, 0], 0.0, 0.0, 1)
    b = _ring(211, [2.0 + gap, 0, 0], np.pi / 2, 0.0, 2)
    engine.set_curves([a, b])
    got = engine.linking_numbers([[0, 1]], method="directsum", fp64=1).lk[0]
    ref = O.ds(a, b)
    print(gap, "got", got, "oracle", ref)
    assert abs(got - ref) < 1e-12 + 1e-14 / gap


def test_planar_and_touching_curves_keep_their_signs(engine):
    """Coplanar curves have zero triple products, and so has a shared vertex:
    the sums are the oracle's, not noise over noise.  A shared vertex's sum
    depends on which curve comes first, in the oracle too (its two orders
    differ by 1/4 here): the engine's is one of them."""
    a = _ring(130, [0, 0, 0], 0.0, 0.0, 1)
    b = _ring(70, [3.0, 0, 0], 0.0, 0.0, 2)
    c = a[:40].copy()
    c[1:] += np.array([0.5, 0.25, 0.75])
    engine.set_curves([a, b, c])
    got = engine.linking_numbers([[0, 1], [0, 2]], method="directsum", fp64=1).lk
    print("got", got, "oracle", O.ds(a, b), O.ds(a, c), O.ds(c, a))
    assert abs(got[0] - O.ds(a, b)) < 1e-12
    assert min(abs(got[1] - O.ds(a, c)), abs(got[1] - O.ds(c, a))) < 1e-12


@pytest.mark.parametrize("gap", [1e3, 1e10, 1e11, 3e12, 1e13, 1e15])
@pytest.mark.parametrize("fp64", [1, 0])
def test_curves_far_apart_sum_to_zero(engine, gap, fp64):
    """Pairs that no search would list: the products of four denominators'
    x', r^24 for vectors of length r, stay finite (in FP32, whose own range ends
    first, the judge sums in FP64).  64 x 48 angles of at most 0.02 / r^2."""
    a = _ring(64, [0, 0, 0], 0.0, 0.05, 1)
    b = _ring(48, [gap, 0.3 * gap, -gap], 1.1, 0.05, 2)
    engine.set_curves([a, b])
    got = engine.linking_numbers([[0, 1]], method="directsum", fp64=fp64).lk[0]
    assert abs(got) < 3072 * 0.02 / gap ** 2 + 1e-15


@pytest.mark.parametrize("radius", [1.0, 1e-2, 1e-3, 1e-5, 1e-7, 1e-9])
def test_small_curves_beside_a_large_one(engine, radius):
    """The short path's limit follows the pair's own size, not that of the
    model's largest curve (radius 500): the sums keep the tolerance above."""
    a = radius * _ring(600, [0, 0, 0], 0.0, 0.07, 1)
    b = radius * _ring(511, [0.9, 0.1, 0.2], 1.3, 0.05, 2)
    c = radius * _ring(300, [2.0 + 1e-5, 0, 0], np.pi / 2, 0.0, 3)  # passes a at about 0.01 of its size
    engine.set_curves([a, b, c, 500 * _ring(64, [0, 0, 0], 0.0, 0.0, 4)])
    got = engine.linking_numbers([[0, 1], [0, 2]], method="directsum", fp64=1).lk
    ref = [O.ds(a, b), O.ds(a, c)]
    print(radius, "got", got, "oracle", ref)
    assert np.abs(got - ref).max() < 1e-12


def test_small_curves_take_no_longer_beside_a_large_one(engine):
    """The general path on every step took 3.1 times as long."""
    ring = [1e-2 * _ring(16384, [x, 0, 0], tilt, 0.05, 1) for x, tilt in ((0, 0.0), (0.9, 1.3))]
    large = 500 * _ring(64, [0, 0, 0], 0.0, 0.0, 4)
    ms = []
    for curves in (ring, ring + [large]):
        engine.set_curves(curves)
        times = []
        for _ in range(5):
            engine.linking_numbers([[0, 1]], method="directsum", fp64=1)
            times.append(engine.stats()["ms_ds_kernel"])
        ms.append(min(times))
    print("alone, beside", ms)
    assert ms[1] < 1.6 * ms[0]
