"""Single-surface calls on the far side of the small-call rule: the persistent kernels give the points the
bits of small calls, keep their counters and lists apart on several streams, and the no-allocation entry
point's fixed array serves them; and a large call does not wait for the few points that run to the limit.
That every size here is beyond the rule is checked by test_path_rules.py."""
import time

import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

SHORT = dict(precision=G.GN_MIXED, fp32_iters=6, fp64_tail=3, tol_step32=3e-5, tol_step=1e-10, tol_quad=1e-10)
LONG = dict(SHORT, fp32_iters=30, fp64_tail=40)
DEFAULT = dict(precision=G.GN_MIXED, tol_step32=1e-4)  # 20 FP32 and 3 FP64 steps
# (p, q, options without the newton bits, points)
BITS = [(2, 2, dict(SHORT, fp32_iters=20), 850_003), (2, 2, LONG, 180_001), (2, 3, SHORT, 700_001), (3, 3, SHORT, 520_001),
        (3, 3, LONG, 100_003), (4, 4, SHORT, 330_001), (5, 5, SHORT, 230_001), (5, 5, LONG, 45_001)]
SMALL = 1000
NOALLOC = (600_001, 520_001)
STREAMS = 300_001
SLOW = 4_000_000


def _surface(p, q, net=20, seed=17):
    sd = synth.surface_G(net, net + 3, p, q, seed=seed, jitter=0.3)
    g = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    g.BuildTree(3)
    g.BuildSeedGrid(0)
    return g


def _points(g, n, seed, far=0.0):
    gen = torch.Generator().manual_seed(seed)
    u, v = torch.rand(2, n, dtype=torch.float64, generator=gen).cuda()
    P = g.Evaluate(u, v, 0) + 0.01 * torch.randn(3, n, dtype=torch.float64, generator=gen).cuda()
    m = torch.rand(n, generator=gen).cuda() < far
    return torch.where(m[None], P * 3 - 1, P).contiguous()


def _same(a, b):
    return all(torch.equal(x.contiguous().view(torch.uint8), y.contiguous().view(torch.uint8)) for x, y in zip(a, b))


@pytest.mark.parametrize("p,q,opts,n", BITS)
def test_a_large_call_gives_the_small_calls_bits(p, q, opts, n):
    g = _surface(p, q)
    few = _points(g, SMALL, 5, 0.1)
    few[0, 11], few[1, 23], few[2, 37] = float("nan"), float("inf"), float("-inf")
    P = few[:, torch.arange(n, device="cuda") % SMALL].contiguous()
    for seed, newton in ((G.SEED_GRID_STEP, 3), (G.SEED_GREEDY_LEAF, 2)):
        o = G.default_opts(seed_mode=seed, newton=newton, **opts)
        one = g.NewInverse(*few, o, iters=True)
        all_ = g.NewInverse(*P, o, iters=True)
        for k in (0, SMALL * (n // SMALL - 1)):
            assert _same([t[k:k + SMALL] for t in all_], one), (seed, k)


def test_noalloc_on_two_large_calls():
    """The second call is smaller: the array keeps the first's contents."""
    g = _surface(3, 3)
    for n in NOALLOC:
        P = _points(g, n, n, 0.01)
        o = G.default_opts(newton=3, **SHORT)
        assert _same(g.NewInverseNoAlloc(*P, o), g.NewInverse(*P, o)), n


def test_concurrent_calls_keep_counters_and_lists_apart():
    gs = [_surface(3, 3, seed=k) for k in (1, 2)]
    P = [_points(g, STREAMS, 7 + k, 0.01) for k, g in enumerate(gs)]
    o = G.default_opts(newton=3, **DEFAULT)
    alone = [g.NewInverse(*p, o) for g, p in zip(gs, P)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(4)]
    outs = [[torch.empty_like(t) for t in alone[0]] for _ in range(16)]
    torch.cuda.synchronize()
    for k, out in enumerate(outs):
        gs[k % 2].NewInverse(*P[k % 2], o, out=out, stream=streams[k % 4])
    torch.cuda.synchronize()
    for k, out in enumerate(outs):
        assert _same(out, alone[k % 2]), k


def test_slow_points_do_not_hold_up_the_others():
    """2% of the points run far longer than the rest: a point of a biquadratic patch still takes no longer
    than one of a bicubic patch (nearly twice as long where every wave waits for its slowest lane)."""
    o = G.default_opts(seed_mode=G.SEED_GRID_STEP, newton=3, **LONG)

    def per_point(p, n):
        g = _surface(p, p, net=24)
        P = _points(g, n, 5, 0.02)
        out = [torch.empty(n, dtype=d, device="cuda") for d in (torch.float64, torch.float64, torch.uint8)]
        t = []
        for _ in range(6):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            g.NewInverse(*P, o, out=out)
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t[1:]) / n

    two, three = per_point(2, SLOW), per_point(3, 1_000_000)
    assert two < 1.2 * three, (two, three)
