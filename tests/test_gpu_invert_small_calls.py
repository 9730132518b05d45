"""Calls small enough for one kernel from seed to result: each point gets the bits that the persistent
kernels give it as part of a large call.  Sizes at the edges of a wave and of the rule, every class of
patch, each seed, the option bits, points that do not converge, that are not finite, and no iterations."""
import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

LARGE = 700_001  # beyond the rule for every degree (at most three rounds of 7 waves on 256 CUs)
MIXED = dict(precision=G.GN_MIXED, fp32_iters=6, fp64_tail=3, tol_step32=3e-5, tol_step=1e-10, tol_quad=1e-10)


def _surface(p, q, nu, nv, levels=3):
    sd = synth.surface_G(nu, nv, p, q, seed=17, jitter=0.3)
    g = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    g.BuildTree(levels)
    if levels > 1:
        g.BuildSeedGrid(0)
    return g


def _same(g, P, o, n, given):
    """The first n points on their own, and in front of copies of themselves."""
    def call(pts, uv):
        out = [torch.empty(pts.shape[1], dtype=d, device="cuda") for d in (torch.float64, torch.float64, torch.uint8)]
        out[0].copy_(uv[0]), out[1].copy_(uv[1])
        return g.NewInverse(*pts, o, out=out, iters=True)
    uv = torch.rand(2, n, dtype=torch.float64, generator=torch.Generator().manual_seed(3)).cuda() if given else \
        torch.zeros(2, n, dtype=torch.float64, device="cuda")
    idx = torch.arange(LARGE, device="cuda") % n
    one = call(P[:, :n].contiguous(), uv)
    all_ = call(P[:, idx].contiguous(), uv[:, idx].contiguous())
    for a, b in zip(one, all_):
        assert torch.equal(a.view(torch.uint8), b[:n].contiguous().view(torch.uint8))
    return one


def _points(g, n, seed):
    gen = torch.Generator().manual_seed(seed)
    u, v = torch.rand(2, n, dtype=torch.float64, generator=gen).cuda()
    P = g.Evaluate(u, v, 0) + 0.02 * torch.randn(3, n, dtype=torch.float64, generator=gen).cuda()
    P[:, ::7] = P[:, ::7] * 3 - 1
    if n > 40:
        P[0, 11], P[1, 23], P[2, 37] = float("nan"), float("inf"), float("-inf")
    return P.contiguous()


SEEDS = [G.SEED_GREEDY_LEAF, G.SEED_GREEDY_STEP, G.SEED_GRID_STEP, G.SEED_NEAREST_LEAF, G.SEED_GIVEN]


@pytest.mark.parametrize("p,q,nu,nv", [(2, 2, 3, 4), (3, 3, 8, 8), (2, 5, 20, 9), (4, 3, 40, 40), (5, 5, 12, 13),
                                       (5, 5, 480, 480), (3, 2, 16, 700)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
def test_a_small_call_gives_the_large_calls_bits(p, q, nu, nv, n):
    g = _surface(p, q, nu, nv)
    P = _points(g, n, 5)
    for k, seed in enumerate(SEEDS):
        newton = k % 4
        _same(g, P, G.default_opts(seed_mode=seed, newton=newton, max_iter=30), n, seed == G.SEED_GIVEN)
        st = _same(g, P, G.default_opts(seed_mode=seed, newton=3 - newton, clamp=k % 2, **MIXED), n,
                   seed == G.SEED_GIVEN)[2]
        if n > 40:
            assert torch.all(st[[11, 23, 37]] == G.PT_NONFINITE)


@pytest.mark.parametrize("opts", [dict(max_iter=0), dict(fp32_iters=0), dict(fp64_tail=0), dict(max_iter=300),
                                  dict(tol_dist=5e-2), dict(fallback=1)])
def test_limits_and_tolerances(opts):
    g = _surface(3, 3, 12, 12)
    P = _points(g, 500, 9)
    _same(g, P, G.default_opts(**{**dict(newton=3, max_iter=25), **opts}), 500, False)
    _same(g, P, G.default_opts(**{**MIXED, **dict(newton=3), **opts}), 500, False)


@pytest.mark.parametrize("p,q,n", [(3, 3, 65536), (3, 3, 98305), (3, 3, 131073), (5, 5, 32769), (5, 5, 49153),
                                   (2, 2, 344065)])
def test_sizes_around_the_rule(p, q, n):
    g = _surface(p, q, 16, 16)
    P = _points(g, n, 6)
    _same(g, P, G.default_opts(newton=2), n, False)
    _same(g, P, G.default_opts(seed_mode=G.SEED_GRID_STEP, newton=3, **MIXED), n, False)


def test_a_tree_of_one_leaf():
    """The stepped seed of the only leaf starts from that leaf's centre, as gn_seed's does."""
    g = _surface(3, 3, 8, 8, levels=1)
    P = _points(g, 300, 4)
    _, su, sv = g.Seed(*P, exact="step")
    given = [su.clone(), sv.clone(), torch.empty(300, dtype=torch.uint8, device="cuda")]
    g.NewInverse(*P, G.default_opts(seed_mode=G.SEED_GIVEN, newton=2), out=given)
    got = g.NewInverse(*P, G.default_opts(seed_mode=G.SEED_GREEDY_STEP, newton=2))
    for a, b in zip(got, given):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    _same(g, P, G.default_opts(seed_mode=G.SEED_GREEDY_STEP, newton=2), 300, False)
