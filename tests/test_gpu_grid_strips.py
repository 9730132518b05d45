"""Grids of few columns (FP32): a lane per point, the bits of gn_evaluate_f32 at the edges of the spread of
rows over lanes, for ordered and unordered samples and samples on knots; and no slower than the points one
by one by more than a little."""
import time

import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu


def _surface(p, q, net):
    sd = synth.surface_G(net, net + 1, p, q, seed=41, jitter=0.3)
    return sd, G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)


@pytest.mark.parametrize("p,q,net", [(3, 3, 16), (2, 4, 9), (5, 5, 60), (1, 1, 8), (7, 3, 12)])
@pytest.mark.parametrize("cols", [1, 2, 3, 7, 8, 31, 32, 33, 64, 65])
@pytest.mark.parametrize("rows", [1, 7, 8, 255, 256, 257, 9001])
def test_strip_equals_points(p, q, net, rows, cols):
    rng = np.random.default_rng(rows * 100 + cols)
    sd, gs = _surface(p, q, net)
    us, vs = (rng.random(k).astype(np.float32) for k in (rows, cols))
    if cols % 2:
        us.sort()
    us[:: 5] = sd.ku[np.arange(us[:: 5].size) % sd.ku.size]  # on knots, as near as floats come
    vs[-1] = 1.0
    U, V = (a.ravel() for a in np.meshgrid(us, vs, indexing="ij"))
    for order in (0, 1, 2):
        got = gs.EvaluateGrid(us, vs, order).cpu().numpy()
        ref = gs.Evaluate(U, V, order, precision=G.GN_FP32).cpu().numpy()
        assert got.shape == ref.shape and np.array_equal(got, ref), order


@pytest.mark.parametrize("rows,cols", [(1 << 20, 1), (1 << 18, 4)])
def test_strip_is_not_slower_than_its_points(rows, cols):
    """Twenty times slower where a workgroup is 256 columns wide."""
    _, gs = _surface(3, 3, 16)
    us = (torch.arange(rows, device="cuda") / rows).float()
    vs = (torch.arange(cols, device="cuda") / cols).float()
    U, V = us.repeat_interleave(cols), vs.repeat(rows)
    out = torch.empty((18, rows * cols), device="cuda")

    def best(f):
        t = []
        for _ in range(6):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(5):
                f()
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t[1:])

    strip = best(lambda: gs.EvaluateGrid(us, vs, 2, out=out))
    points = best(lambda: gs.Evaluate(U, V, 2, precision=G.GN_FP32, out=out))
    assert strip < 2 * points, (strip, points)
