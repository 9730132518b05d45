"""The global projection's chunks, pool and tree walk: a query's result and its count of leaves solved
are its own, so a call of any size gives each query the bits it gets in a call of its own.  Sizes at the
edges of chunks (16 .. 128 queries per wave), trees of every depth (a single leaf, one, two and three
levels of 8 x 8), queries near, far (many leaves each, so the pool fills) and non-finite."""
import numpy as np
import pytest

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("p,q,levels,n", [
    (3, 3, 1, 70), (3, 3, 2, 15), (2, 4, 2, 16), (3, 3, 3, 17), (5, 3, 3, 129), (5, 5, 3, 65), (1, 6, 3, 63),
    (3, 3, 4, 33), (3, 3, 3, 2500), (4, 4, 3, 300000),
])
def test_each_query_keeps_its_own_result(p, q, levels, n):
    sd = synth.surface_G(14, 13, p, q, seed=71, jitter=0.3)
    g = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    g.BuildTree(levels)
    rng = np.random.default_rng(n)
    P = _np(g.Evaluate(rng.uniform(0, 1, n), rng.uniform(0, 1, n), 0)) + rng.normal(0, 0.03, (3, n))
    far = slice(0, min(n // 2, 400))
    P[:, far] = P[:, far] * 4.0 - 1.5
    if n > 16:
        P[0, 7], P[1, 11], P[2, 13] = np.nan, np.inf, -np.inf
    o = G.default_opts(seed_mode=G.SEED_GLOBAL, max_iter=20)
    u, v, st, leaves, _ = (_np(t) for t in g.NewInverse(*P, o, iters=True))
    pick = np.unique(np.r_[0, n - 1, np.arange(min(n, 14)), rng.integers(0, n, 25)])
    for i in pick:
        one = [_np(t)[0] for t in g.NewInverse(*(P[k, i:i + 1].copy() for k in range(3)), o, iters=True)]
        assert one[0] == u[i] and one[1] == v[i] and one[2] == st[i] and one[3] == leaves[i], i
    if n > 16:
        assert np.all(st[[7, 11, 13]] == G.PT_NONFINITE)
    if levels == 1:
        assert np.all(leaves == 1)
