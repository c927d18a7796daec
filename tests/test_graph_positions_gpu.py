"""A captured certificate serves new positions of curves of the same sizes: after
each upload the results are those of the eager launch sequence on the new
coordinates, whatever changed with them (the scale, FP32-exactness, the
candidate pairs, one curve's size)."""
import numpy as np
import pytest

flk = pytest.importorskip("fastlinkingnumbers_amd")
from fastlinkingnumbers_amd import workloads as W  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(method="directsum"), dict(method="directsum", fp64=1), dict(method="barneshut"),
                                dict(method="barneshut", bh_direct_threshold=300 * 300)],
                         ids=["direct", "direct64", "tree", "hybrid"])
def test_captured_certificate_on_new_positions(engine, kw):
    base = W.workload(4, scale=0.006)
    rng = np.random.default_rng(3)
    steps = [base, [c + 0.01 * rng.normal(size=c.shape) for c in base], [1000.0 * c + 3e4 for c in base],
             [c.astype(np.float32).astype(np.float64) for c in base], [c[:, [1, 0, 2]] for c in base],
             base[:-1] + [base[-1][:-1]], base]
    for k, curves in enumerate(steps):
        engine.set_curves(curves)
        pairs = engine.potential_links()
        for _ in range(2):
            got = engine.linking_numbers(pairs, fallback_tol=0.0, **kw)
            want = engine.linking_numbers(pairs, fallback_tol=0.0, graph=0, **kw)
            # the eager and the captured hybrid split the direct sum alike; the
            # trees' sums differ by the order of FP64 additions
            np.testing.assert_allclose(got.lk, want.lk, rtol=0, atol=1e-9, err_msg=str(k))
            np.testing.assert_allclose(got.err, want.err, rtol=1e-9, atol=1e-15, err_msg=str(k))
            assert np.array_equal(got.flags, want.flags), k


def test_one_graph_with_and_without_re_runs(engine):
    """The re-runs' own graph is launched behind the first pass, at once, or not at
    all, as the positions of one key ask for them."""
    walks = W.random_walk_pair(seed=3, n=16000, rg=25.0, workload=3)
    t = 2 * np.pi * np.arange(16000) / 16000
    rings = [np.stack([np.cos(t), np.sin(t), 0 * t], 1), np.stack([1 + np.cos(t), 0.1 * np.cos(3 * t), np.sin(t)], 1)]
    rings = [r + 1e-9 * w for r, w in zip(rings, walks)]  # FP32 holds neither
    retries = []
    for curves in (rings, rings, walks, walks, rings, walks, rings, rings):
        engine.set_curves(curves)
        got = engine.linking_numbers([[0, 1]], method="barneshut", fallback_tol=0.0)
        want = engine.linking_numbers([[0, 1]], method="barneshut", fallback_tol=0.0, graph=0)
        retries.append(got.stats["retries"])
        for key in ("bh_visits", "bh_far", "bh_leaf_pairs", "retries"):
            assert got.stats[key] == want.stats[key], key
        np.testing.assert_allclose(got.lk, want.lk, rtol=0, atol=1e-9)
        np.testing.assert_allclose(got.err, want.err, rtol=1e-9)
        assert np.array_equal(got.flags, want.flags)
    assert retries == [0, 0, 1, 1, 0, 1, 0, 0]
