"""Scattered evaluation: a point gets the same bits in a call of any size, whatever number of tiles its
waves take.  Sizes at the edges of a wave and a block, on both sides of one round and of eight rounds of
resident blocks, rows that start on a line and rows that don't, and outputs beyond 800 MB."""
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

SMALL = 1000  # four blocks, one tile per wave


@pytest.mark.parametrize("p,q,order", [(3, 3, 2), (2, 2, 1), (5, 4, 3), (4, 4, 0), (2, 5, 2)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 257, 65537, 131_073, 262_145, 1_048_576, 1_300_003, 2_200_000])
def test_points_do_not_depend_on_the_calls_size(p, q, order, dtype, n):
    _check(p, q, order, dtype, n)


@pytest.mark.parametrize("p,q,order,dtype,n", [(3, 3, 2, "f64", 5_600_000), (3, 3, 2, "f32", 4_200_001),
                                               (3, 3, 3, "f32", 4_200_064), (5, 5, 3, "f64", 3_400_001)])
def test_large_calls(p, q, order, dtype, n):
    _check(p, q, order, dtype, n)


def _check(p, q, order, dtype, n):
    sd = synth.surface_G(23, 17, p, q, seed=41, jitter=0.3)
    s = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    t = torch.float64 if dtype == "f64" else torch.float32
    prec = G.GN_FP64 if dtype == "f64" else G.GN_FP32
    u, v = torch.rand(2, n, dtype=t, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    out = torch.full((3 * (1, 3, 6, 10)[order], n), float("nan"), dtype=t, device="cuda")
    s.Evaluate(u, v, order, precision=prec, out=out)
    assert not torch.isnan(out).any()
    starts = {0, max(0, n - SMALL), n // 2, n // 3}
    for a in starts:
        b = min(n, a + SMALL)
        one = s.Evaluate(u[a:b].clone(), v[a:b].clone(), order, precision=prec)
        assert torch.equal(out[:, a:b], one.reshape(out.shape[0], b - a)), (a, b)
