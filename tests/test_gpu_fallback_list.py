"""The fallback's launch is sized for its list, not for the call: a long call with no query listed hardly
pays for it, lists from one query to all of a call's give each query the result of a call of its own, and
a call of more than 2^30 queries is served."""
import time

import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

MIXED = dict(precision=G.GN_MIXED, newton=3, fp32_iters=6, fp64_tail=3, tol_step32=3e-5, tol_step=1e-10, tol_quad=1e-10)


@pytest.fixture(scope="module")
def surf():
    sd = synth.surface_G(32, 32, 3, 3, seed=1002)
    g = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    g.BuildTree(3)
    g.BuildSeedGrid(0)
    return g


def _points(g, n, far):
    """The queries numbered in far lie anywhere, the others within 1e-3 of the surface."""
    gen = torch.Generator(device="cuda").manual_seed(3)
    u, v = torch.rand(2, n, dtype=torch.float64, device="cuda", generator=gen)
    P = g.Evaluate(u, v, 0) + 1e-3 * torch.randn(3, n, dtype=torch.float64, device="cuda", generator=gen)
    P[:, far] = P[:, far] * 3 - 1
    return [t.contiguous() for t in P]


def test_an_empty_list_costs_little(surf):
    n = 16_000_000
    P = _points(surf, n, torch.arange(0, device="cuda"))
    out = [torch.empty(n, dtype=d, device="cuda") for d in (torch.float64, torch.float64, torch.uint8)]

    def best(o):
        t = []
        for _ in range(6):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            surf.NewInverse(*P, o, out=out)
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t[1:])

    plain, fb = (best(G.default_opts(seed_mode=G.SEED_GRID_STEP, fallback=f, **MIXED)) for f in (0, 1))
    assert fb < 1.25 * plain, (fb, plain)


@pytest.mark.parametrize("n", [1, 17, 64, 65, 4097, 300_000])
@pytest.mark.parametrize("listed", ["one", "some", "all"])
def test_listed_queries_get_their_own_results(surf, n, listed):
    """Iteration limits that leave a third, most or all of the queries to the fallback."""
    far = torch.arange(n, device="cuda")
    P = _points(surf, n, far[::3])
    o = G.default_opts(seed_mode=G.SEED_GRID_STEP, fallback=1, **{**MIXED, **dict(
        fp32_iters={"all": 0, "some": 2, "one": 20}[listed], fp64_tail={"all": 0, "some": 1, "one": 20}[listed])})
    out = surf.NewInverse(*P, o)
    pick = np.unique(np.random.default_rng(1).integers(0, n, 40))
    pick[0] = n - 1
    sel = torch.from_numpy(np.unique(pick)).cuda()
    one = surf.NewInverse(*(t[sel].contiguous() for t in P), o)
    for a, b in zip(out, one):
        assert torch.equal(a[sel], b)


def test_more_than_2_30_queries(surf):
    """Launches hold below 2^32 lanes."""
    n = (1 << 30) + 77
    few = _points(surf, 64, torch.arange(64, device="cuda"))
    uv = torch.full((2, 1), 0.3, dtype=torch.float64, device="cuda")
    Q = surf.Evaluate(uv[0], uv[1], 0)
    P = [Q[k, 0].expand(n).contiguous() for k in range(3)]
    at = torch.linspace(0, n - 1, 64, dtype=torch.float64, device="cuda").long()
    for k in range(3):
        P[k][at] = few[k]
    o = dict(seed_mode=G.SEED_GIVEN, fallback=1, **{**MIXED, **dict(fp32_iters=1, fp64_tail=1)})
    out = [torch.full((n,), 0.3, dtype=torch.float64, device="cuda") for _ in range(2)] + \
        [torch.empty(n, dtype=torch.uint8, device="cuda")]
    surf.NewInverse(*P, G.default_opts(**o), out=out)
    ref = [torch.full((64,), 0.3, dtype=torch.float64, device="cuda") for _ in range(2)] + \
        [torch.empty(64, dtype=torch.uint8, device="cuda")]
    surf.NewInverse(*few, G.default_opts(**o), out=ref)
    for a, b in zip(out, ref):
        assert torch.equal(a[at], b)
    mask = torch.ones(n, dtype=torch.bool, device="cuda")
    mask[at] = False
    assert bool(((out[2] == G.PT_CONVERGED) | ~mask).all())
    del P, out, mask
    torch.cuda.empty_cache()
