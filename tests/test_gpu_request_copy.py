"""A request's results leave the server in one copy: equal to the arrays they are copied from, for
surfaces and curves, at the edges of a workgroup and of the copy's grid, and own memory."""
import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 255, 256, 257, 70_001, 8192 * 256 + 3])
def test_results_are_copies_of_the_servers_arrays(n):
    sd = synth.surface_G(9, 9, 2, 2, seed=4)
    s = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    s.BuildTree(3)
    c = G.Curve.from_def(synth.helix_curve(12, 3, seed=5))
    batch = G.Batch([s])
    srv = G.Server(batch, [c])
    try:
        P = torch.rand(3, n, dtype=torch.float64, generator=torch.Generator().manual_seed(n)).cuda()
        torch.cuda.synchronize()
        for obj in (0, 1):
            info = srv.wait(srv.submit(obj, *P))
            got = srv.results(info)
            want = [torch.as_tensor(G._DeviceView(p, n, t), device="cuda") if p else None
                    for p, t in ((info.u, "<f8"), (info.v, "<f8"), (info.status, "|u1"))]
            assert (got[1] is None) == (obj == 1 or not info.v)
            for a, b in zip(got, want):
                assert (a is None and b is None) or (torch.equal(a, b) and (n == 0 or a.data_ptr() != b.data_ptr()))
                assert a is None or (a.shape == (n,) and a.is_cuda)
    finally:
        srv.close()
