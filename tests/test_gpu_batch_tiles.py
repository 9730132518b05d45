"""Batched tiles: a point gets the bits of a call on its surface alone.  One surface of every degree class
and generic ones, segments of lengths at the edges of a wave, every seed, both precisions, the option
bits, tile sizes and occupancy caps, points that are not finite."""
import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

DEGREES = [(p, q) for p in range(2, 6) for q in range(2, 6)] + [(1, 3), (6, 2)]
COUNTS = [1, 63, 64, 65, 129, 200, 7]
SEEDS = [G.SEED_GREEDY_LEAF, G.SEED_GREEDY_STEP, G.SEED_GRID_STEP, G.SEED_NEAREST_LEAF, G.SEED_GIVEN]
MIXED = dict(precision=G.GN_MIXED, fp32_iters=6, fp64_tail=3, tol_step32=3e-5, tol_step=1e-10, tol_quad=1e-10)


@pytest.fixture(scope="module")
def batch():
    surfs = []
    for k, (p, q) in enumerate(DEGREES):
        sd = synth.surface_G(8 + k, 24 - k, p, q, seed=100 + k, jitter=0.3)
        g = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
        g.BuildTree(3)
        g.BuildSeedGrid(16)
        surfs.append(g)
    gen = torch.Generator().manual_seed(8)
    counts = [COUNTS[k % len(COUNTS)] for k in range(len(surfs))]
    P = []
    for g, n in zip(surfs, counts):
        u, v = torch.rand(2, n, dtype=torch.float64, generator=gen).cuda()
        pts = g.Evaluate(u, v, 0) + 0.02 * torch.randn(3, n, dtype=torch.float64, generator=gen).cuda()
        pts[:, ::7] = pts[:, ::7] * 3 - 1
        if n > 60:
            pts[0, 11], pts[1, 23], pts[2, 37] = float("nan"), float("inf"), float("-inf")
        P.append(pts)
    return surfs, G.Batch(surfs), counts, P


@pytest.mark.parametrize("seed", SEEDS)
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("shape", [(1024, 0), (64, 1), (100, 2)])
def test_a_point_gets_its_surfaces_bits(batch, seed, mixed, shape):
    surfs, b, counts, P = batch
    x, y, z = (torch.cat([p[i] for p in P]).contiguous() for i in range(3))
    n = x.numel()
    start = torch.rand(2, n, dtype=torch.float64, generator=torch.Generator().manual_seed(2)).cuda()
    b.set_shape(*shape)
    for newton in range(4):
        o = G.default_opts(seed_mode=seed, newton=newton, clamp=newton % 2, **(MIXED if mixed else dict(max_iter=25)))
        out = [start[0].clone(), start[1].clone(), torch.empty(n, dtype=torch.uint8, device="cuda")]
        b.invert(G.segments(np.arange(len(surfs)), counts), x, y, z, o, out=out)
        at = 0
        for g, c, pts in zip(surfs, counts, P):
            one = [start[0, at:at + c].clone(), start[1, at:at + c].clone(),
                   torch.empty(c, dtype=torch.uint8, device="cuda")]
            g.NewInverse(*(t.contiguous() for t in pts), o, out=one)
            for a, w in zip(out, one):
                assert torch.equal(a[at:at + c].contiguous().view(torch.uint8), w.view(torch.uint8)), (g.p, g.q, newton)
            at += c
