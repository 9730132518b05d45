"""Grid evaluation (FP32) at the edges of its tiling: 64-lane waves, 256-column workgroups and 4 to 32
rows per workgroup; one row or column; every order; exact and generic degrees; repeated and unordered
samples.  The grid kernel contracts in the per-point kernels' order (v first, then the rows, one fused
multiply-add each), so its values equal gn_evaluate_f32's at the same parameters bit for bit."""
import numpy as np
import pytest

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,q,net,rows,cols", [
    (3, 3, 8, 1, 1), (3, 3, 8, 3, 63), (2, 4, 9, 4, 64), (4, 2, 12, 5, 65), (5, 5, 10, 33, 255),
    (3, 3, 64, 31, 256), (3, 2, 20, 32, 257), (2, 2, 7, 700, 1), (1, 7, 12, 70, 513), (6, 1, 9, 65, 127),
    (3, 3, 16, 2053, 300),
])
def test_grid_equals_points(p, q, net, rows, cols):
    rng = np.random.default_rng(rows * 1000 + cols)
    sd = synth.surface_G(net, net + 1, p, q, seed=41, jitter=0.3)
    gs = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    us, vs = (rng.random(k).astype(np.float32) for k in (rows, cols))  # unordered
    us[0], vs[-1] = 0.0, 1.0
    if rows > 2:
        us[1] = us[2]
    U, V = (a.ravel() for a in np.meshgrid(us, vs, indexing="ij"))
    for order in (0, 1, 2):
        got = gs.EvaluateGrid(us, vs, order).cpu().numpy()
        ref = gs.Evaluate(U, V, order, precision=G.GN_FP32).cpu().numpy()
        assert got.shape == ref.shape and np.array_equal(got, ref), order
