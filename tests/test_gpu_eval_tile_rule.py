"""Scattered evaluation: a count that is no multiple of a line costs what its partial lines cost, not what a
wrong number of tiles per wave adds; and the counts at which the rule changes its mind give the bits of
small calls."""
import time

import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

SMALL = 1000
FIELDS = (3, 9, 18, 30)


def _surface(p, q, net):
    sd = synth.surface_G(net, net, p, q, seed=41, jitter=0.3)
    return G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)


@pytest.mark.parametrize("p,q,order,dtype,n", [
    (2, 2, 3, torch.float64, 300_000), (2, 2, 2, torch.float64, 1_600_000), (3, 3, 3, torch.float64, 700_001),
    (4, 4, 3, torch.float64, 900_001), (3, 3, 1, torch.float64, 2_200_001), (2, 2, 3, torch.float32, 600_000),
    (2, 2, 2, torch.float32, 1_600_000), (3, 3, 2, torch.float32, 1_300_001), (4, 4, 2, torch.float32, 1_300_001),
    (5, 5, 2, torch.float32, 1_300_001), (3, 3, 2, torch.float64, 1 << 23), (3, 3, 2, torch.float32, 1 << 24)])
def test_bits_at_every_number_of_tiles(p, q, order, dtype, n):
    s = _surface(p, q, 20)
    prec = G.GN_FP64 if dtype == torch.float64 else G.GN_FP32
    u, v = torch.rand(2, n, dtype=dtype, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    out = torch.full((FIELDS[order], n), float("nan"), dtype=dtype, device="cuda")
    s.Evaluate(u, v, order, precision=prec, out=out)
    assert not torch.isnan(out).any()
    for a in (0, n // 3, n // 2, n - SMALL):
        one = s.Evaluate(u[a:a + SMALL].clone(), v[a:a + SMALL].clone(), order, precision=prec)
        assert torch.equal(out[:, a:a + SMALL], one), a


def test_partial_lines():
    """FP32 patches of 36 entries are bound by work, not by writes: a count that is no multiple of a line
    costs as much as one that is (a quarter more with one tile per wave)."""
    s = _surface(5, 5, 20)

    def best(n):
        u, v = torch.rand(2, n, dtype=torch.float32, device="cuda")
        out = torch.empty((18, n), device="cuda")
        t = []
        for _ in range(7):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(5):
                s.Evaluate(u, v, 2, precision=G.GN_FP32, out=out)
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t[1:])

    whole, part = best(12_000_032), best(12_000_007)
    assert part < 1.12 * whole, (part, whole)


@pytest.mark.parametrize("p,q,order,dtype,n", [
    (2, 5, 2, torch.float32, 800_000), (5, 5, 1, torch.float32, 800_003), (5, 5, 3, torch.float32, 300_003),
    (4, 4, 3, torch.float64, 300_003), (4, 4, 3, torch.float64, 458_752 - 1),
    (2, 2, 2, torch.float64, 200_003), (3, 3, 2, torch.float64, 1 << 20), (4, 4, 0, torch.float64, 600_001),
    (3, 3, 1, torch.float64, 1_500_001), (4, 4, 2, torch.float32, 1_500_007), (2, 5, 2, torch.float32, 2_000_005),
    (2, 5, 2, torch.float32, 6_000_001)])
def test_bits_in_one_round(p, q, order, dtype, n):
    test_bits_at_every_number_of_tiles(p, q, order, dtype, n)


def test_one_round():
    """FP64 patches of 25 entries run a block per CU.  Five tiles per wave take 300,003 points in one round,
    5/4 of the time of the 262,139 that four take; with four there is a second round for the rest, which
    waves of four tiles cannot share: 1.6 times and more."""
    s = _surface(4, 4, 40)

    def best(n):
        u, v = torch.rand(2, n, dtype=torch.float64, device="cuda")
        out = torch.empty((30, n), dtype=torch.float64, device="cuda")
        t = []
        for _ in range(7):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(20):
                s.Evaluate(u, v, 3, precision=G.GN_FP64, out=out)
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t[1:])

    four, five = best(262_139), best(300_003)
    assert five < 1.42 * four, (five, four)
