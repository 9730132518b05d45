"""Batches whose class groups take the persistent kernels: every point gets the bits of a call on its
surface alone, also from a graph replayed beside other persistent launches; and a group of large patches
is not held up by the few points that don't converge."""
import time

import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

DEGREES = [(p, q) for p in range(2, 6) for q in range(2, 6)] + [(1, 3), (6, 2)]
# points of group 0, 1 and 2 (patches of at most 16 entries, of at most 25, others): above the rule's
# bounds for PLAIN with a Newton bit and for MIXED (test_path_rules.py)
POINTS = [82_000, 72_003, 71_001]
PLAIN = dict(max_iter=25)
MIXED = dict(precision=G.GN_MIXED, fp32_iters=30, fp64_tail=40, tol_step32=3e-5, tol_step=1e-10, tol_quad=1e-10)
SEEDS = [G.SEED_GREEDY_LEAF, G.SEED_GREEDY_STEP, G.SEED_GRID_STEP, G.SEED_NEAREST_LEAF, G.SEED_GIVEN]


def group(p, q):
    if not (2 <= p <= 5 and 2 <= q <= 5):
        return 2
    e = (p + 1) * (q + 1)
    return 0 if e <= 16 else 1 if e <= 25 else 2


def counts():
    groups = [group(p, q) for p, q in DEGREES]
    w = np.array([1 + k % 3 for k in range(len(DEGREES))], dtype=np.float64)
    out = []
    for k, g in enumerate(groups):
        out.append(int(POINTS[g] * w[k] / sum(w[j] for j in range(len(w)) if groups[j] == g)) + 1)
    return out


def _far(P, share, gen):
    m = torch.rand(P.shape[1], generator=gen).cuda() < share
    return torch.where(m[None], P * 3 - 1 + torch.randn(*P.shape, dtype=torch.float64, generator=gen).cuda(), P)


@pytest.fixture(scope="module")
def batch():
    surfs, P = [], []
    gen = torch.Generator().manual_seed(8)
    for k, ((p, q), n) in enumerate(zip(DEGREES, counts())):
        sd = synth.surface_G(8 + k, 24 - k, p, q, seed=100 + k, jitter=0.3)
        g = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
        g.BuildTree(3)
        g.BuildSeedGrid(16)
        surfs.append(g)
        u, v = torch.rand(2, n, dtype=torch.float64, generator=gen).cuda()
        pts = g.Evaluate(u, v, 0) + 0.02 * torch.randn(3, n, dtype=torch.float64, generator=gen).cuda()
        pts = _far(pts, 0.03, gen)
        pts[0, 11], pts[1, 23], pts[2, 37] = float("nan"), float("inf"), float("-inf")
        P.append(pts)
    yield surfs, G.Batch(surfs), P


def _alone(surfs, P, o, start):
    at, res = 0, []
    for g, pts in zip(surfs, P):
        n = pts.shape[1]
        one = [start[0, at:at + n].clone(), start[1, at:at + n].clone(), torch.empty(n, dtype=torch.uint8, device="cuda")]
        g.NewInverse(*(t.contiguous() for t in pts), o, out=one)
        res.append(one)
        at += n
    return [torch.cat([r[k] for r in res]) for k in range(3)]


def _same(a, b):
    return all(torch.equal(x.view(torch.uint8), y.view(torch.uint8)) for x, y in zip(a, b))


@pytest.mark.parametrize("seed", SEEDS)
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("shape", [(1024, 0), (100, 2)])
def test_a_point_gets_its_surfaces_bits(batch, seed, mixed, shape):
    surfs, b, P = batch
    x, y, z = (torch.cat([p[i] for p in P]).contiguous() for i in range(3))
    n = x.numel()
    start = torch.rand(2, n, dtype=torch.float64, generator=torch.Generator().manual_seed(2)).cuda()
    b.set_shape(*shape)
    for newton in range(4):
        o = G.default_opts(seed_mode=seed, newton=newton, clamp=newton % 2, **(MIXED if mixed else PLAIN))
        out = [start[0].clone(), start[1].clone(), torch.empty(n, dtype=torch.uint8, device="cuda")]
        b.invert(G.segments(np.arange(len(surfs)), [p.shape[1] for p in P]), x, y, z, o, out=out)
        assert _same(out, _alone(surfs, P, o, start)), newton


def test_graph_replays_beside_persistent_calls(batch):
    """The graph's launches keep claim counters of their own: replayed on one stream while 300 persistent
    inversions (two counter slots each, so that the shared ring wraps twice) run on another."""
    surfs, b, P = batch
    b.set_shape(1024, 0)
    x, y, z = (torch.cat([p[i] for p in P]).contiguous() for i in range(3))
    n = x.numel()
    segs = G.segments(np.arange(len(surfs)), [p.shape[1] for p in P])
    o = G.default_opts(newton=3, **MIXED)
    ref = [t.clone() for t in b.invert(segs, x, y, z, o)]
    out = [torch.zeros(n, dtype=d, device="cuda") for d in (torch.float64, torch.float64, torch.uint8)]
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    g = b.graph(segs, x, y, z, *out, o, stream=s1)
    big = [P[0][k].repeat(60)[:130_001].contiguous() for k in range(3)]
    eref = [t.clone() for t in surfs[0].NewInverse(*big, o)]
    eout = [[torch.empty_like(t) for t in eref] for _ in range(8)]
    torch.cuda.synchronize()
    for i in range(300):
        if i % 15 == 0:
            g.launch(stream=s1)
        surfs[0].NewInverse(*big, o, out=eout[i % 8], stream=s2)
        if i % 100 == 99:
            torch.cuda.synchronize()
            assert _same(out, ref) and all(_same(e, eref) for e in eout), i
            for t in out:
                t.zero_()
            torch.cuda.synchronize()
    g.close()


def test_slow_points_do_not_hold_up_the_others():
    """2% of the points run to the iteration limit.  A surface's own call refills their lanes' neighbours;
    the batched call of as many points does too (three times as long where waves wait for them)."""
    sd = synth.surface_G(20, 20, 5, 5, seed=10, jitter=0.2)
    surfs = []
    for _ in range(4):
        s = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
        s.BuildTree(3)
        surfs.append(s)
    n = 1 << 20
    gen = torch.Generator().manual_seed(3)
    u, v = torch.rand(2, n, dtype=torch.float64, generator=gen).cuda()
    pts = surfs[0].Evaluate(u, v, 0) + 0.01 * torch.randn(3, n, dtype=torch.float64, generator=gen).cuda()
    P = [t.contiguous() for t in _far(pts, 0.02, gen)]
    o = G.default_opts(newton=G.NEWTON_FP64)
    b = G.Batch(surfs)
    segs = G.segments(np.arange(4), [n // 4] * 4)
    out = [torch.empty(n, dtype=d, device="cuda") for d in (torch.float64, torch.float64, torch.uint8)]

    def best(f):
        t = []
        for _ in range(6):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            f()
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t[1:])

    one = best(lambda: surfs[0].NewInverse(*P, o, out=out))
    many = best(lambda: b.invert(segs, *P, o, out=out))
    assert many < 2 * one, (many, one)
