"""The curve seed search's two-level boxes: span counts at the edges of a box of kSupSpans = 8 spans, of
32 boxes and of the LDS limit, every degree, against the oracle's full scan.

Seeds are sample parameters, so they are equal or another sample's.  Where they differ, the two
samples must tie in the FP32 distances the search compares: each carries at most a few roundings
of coordinates below 8 (|d| <= 16, so 2 d eps 16 + ... < 1e-4 absolute on a squared distance), and
the samples themselves are rounded to FP32.
"""
import numpy as np
import pytest

import gnurbs as G
import oracle as O
from gnurbs import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spans,p", [(1, 1), (1, 7), (7, 2), (8, 3), (9, 4), (17, 5), (64, 6), (65, 3),
                                     (256, 3), (257, 2), (300, 3)])
def test_seeds_equal_full_scan(spans, p):
    rng = np.random.default_rng(1000 * spans + p)
    n = spans + p
    cd = synth.CurveDef(p, synth.clamped_knots(n, p, rng, jitter=0.3), rng.normal(size=(n, 3)),
                        rng.uniform(0.5, 2.0, n))
    g, o = G.Curve.from_def(cd), O.OCurve.from_def(cd)
    m = 3001
    P = o.eval(rng.uniform(0, 1, m)) + rng.normal(0, 0.05, (3, m))
    P[:, ::7] = rng.normal(0, 2.0, (3, P[:, ::7].shape[1]))  # far from the curve: wide bounds
    t, _ = g.Invert(*P, G.default_opts(max_iter=0))
    t, ref = t.cpu().numpy(), o.seed(*P)
    same = t == ref
    assert same.mean() > 0.999
    if not same.all():
        Pb = P[:, ~same]
        da = ((o.eval(t[~same]) - Pb) ** 2).sum(0)
        db = ((o.eval(ref[~same]) - Pb) ** 2).sum(0)
        assert np.all(np.abs(da - db) <= 1e-4)


def test_empty_spans_and_non_finite_queries():
    """A double interior knot leaves an empty span (its samples sit on the knot); queries without a
    finite distance to any sample end GN_PT_NONFINITE."""
    rng = np.random.default_rng(5)
    k = np.array([0, 0, 0, 0, 0.2, 0.5, 0.5, 0.7, 1, 1, 1, 1.0])
    cd = synth.CurveDef(3, k, rng.normal(size=(8, 3)), rng.uniform(0.5, 2.0, 8))
    g, o = G.Curve.from_def(cd), O.OCurve.from_def(cd)
    ts = rng.uniform(0, 1, 500)
    P = o.eval(ts)
    P[0, 3], P[1, 4], P[2, 5], P[0, 6] = np.nan, np.inf, -np.inf, 1e300
    for opts in (G.default_opts(newton=G.NEWTON_FP64), G.default_opts(precision=G.GN_MIXED, newton=3)):
        t, st = (a.cpu().numpy() for a in g.Invert(*P, opts))
        assert np.all(st[3:6] == G.PT_NONFINITE)
        good = np.ones(ts.size, dtype=bool)
        good[3:7] = False
        near = good & (np.abs(t - ts) < 1e-6)
        assert near.mean() > 0.9 and np.max(np.abs(t[near] - ts[near])) <= 1e-9
