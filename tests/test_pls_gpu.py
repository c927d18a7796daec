"""Potential-link search over caller-given boxes against every pair tested on
the host: around the sizes where the device search changes its grid (waves of
four rows, 64-column steps, 1,024-column chunks) and its method (32,768
curves), with touching, empty and NaN boxes, and with more pairs than the
first result buffer holds."""
import numpy as np
import pytest

flk = pytest.importorskip("fastlinkingnumbers_amd")

pytestmark = pytest.mark.gpu


def _boxes(n, seed, size):
    g = np.random.default_rng(seed)
    # a coarse grid of corners, so that many boxes touch exactly
    lo = np.floor(g.uniform(0, 4 * n ** (1 / 3) + 2, size=(n, 3)) * 4) / 4
    b = np.concatenate([lo, lo + np.floor(g.uniform(0, size, size=(n, 3)) * 4) / 4], axis=1)
    if n > 8:
        b[n // 3] = [np.finfo(float).max] * 3 + [-np.finfo(float).max] * 3  # an empty curve
        b[n // 2, 4] = np.nan
        b[n - 2, :3] = -np.inf
    return b


def _brute(b):
    out = []
    for i in range(len(b) - 1):
        hit = np.all((b[i, :3] <= b[i + 1:, 3:]) & (b[i + 1:, :3] <= b[i, 3:]), axis=1)
        out += [(i, i + 1 + int(j)) for j in np.flatnonzero(hit)]
    return np.array(out, dtype=np.int32).reshape(-1, 2)


@pytest.mark.parametrize("n", [2, 3, 4, 5, 16, 17, 63, 64, 65, 257, 1023, 1024, 1025, 2049, 32768, 32769])
def test_pairs_equal_brute_force(engine, n):
    b = _boxes(n, n, 2.0)
    got = engine.potential_links(b)
    assert np.array_equal(got, _brute(b))
    if n < 4096:
        assert np.array_equal(engine.potential_links(b[::-1].copy()), _brute(b[::-1]))


@pytest.mark.parametrize("n", [47, 600])
def test_every_box_overlaps(engine, n):
    """n (n - 1) / 2 pairs: below and beyond the first buffer (1,024 pairs)."""
    b = np.tile([0.0, 0, 0, 1, 1, 1], (n, 1))
    i, j = np.triu_indices(n, 1)
    assert np.array_equal(engine.potential_links(b), np.stack([i, j], 1))
    assert engine.potential_links(b[:1]).shape == (0, 2)
