"""A batched call inside a caller's own stream capture: the graph holds its tile list and its buffers, so
every replay gives the eager call's bits, with new inputs, after other calls of the batch and beside them."""
import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

DEGREES = [(2, 2), (3, 3), (4, 4), (5, 5), (1, 6), (2, 5)]
MIXED = dict(precision=G.GN_MIXED, newton=3, fp32_iters=30, fp64_tail=40, tol_step32=3e-5, tol_step=1e-10, tol_quad=1e-10)


def _batch():
    surfs = []
    for k, (p, q) in enumerate(DEGREES):
        sd = synth.surface_G(9 + k, 12, p, q, seed=50 + k, jitter=0.2)
        s = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
        s.BuildTree(2)
        s.BuildSeedGrid(16)
        surfs.append(s)
    return surfs, G.Batch(surfs)


# one tile, a list longer than one kernel's arguments, groups above the persistent kernels' rule
@pytest.mark.parametrize("per,tile", [(1, 1024), (3000, 64), (70_001, 1024)])
@pytest.mark.parametrize("seed", [G.SEED_GRID_STEP, G.SEED_GREEDY_LEAF, G.SEED_NEAREST_LEAF])
def test_replays_give_the_eager_bits(per, tile, seed):
    surfs, b = _batch()
    b.set_shape(tile, 0)
    counts = [per + 7 * k for k in range(len(surfs))]
    n = sum(counts)
    segs = G.segments(np.arange(len(surfs)), counts)
    gen = torch.Generator().manual_seed(5)
    P = torch.rand(3, n, dtype=torch.float64, generator=gen).cuda()
    o = G.default_opts(seed_mode=seed, **MIXED)
    out = [torch.zeros(n, dtype=d, device="cuda") for d in (torch.float64, torch.float64, torch.uint8)]
    b.invert(segs, *P, o, out=out)  # (first launches load the kernels)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        b.invert(segs, *P, o, out=out)
    del segs
    other = torch.cuda.Stream()
    for rep in range(4):
        P.copy_(torch.rand(3, n, dtype=torch.float64, generator=gen))
        for t in out:
            t.zero_()
        torch.cuda.synchronize()
        g.replay()
        eager = b.invert(G.segments(np.arange(len(surfs)), counts), *P, o, stream=other)
        torch.cuda.synchronize()
        for a, e in zip(out, eager):
            assert torch.equal(a.view(torch.uint8), e.view(torch.uint8)), rep
    b.close()


def test_graphs_are_made_beside_eager_calls():
    """One thread captures batch graphs while another makes calls whose groups take the side streams: every
    call and every replay gives its bits."""
    import threading

    surfs, b = _batch()
    counts = [500 + 7 * k for k in range(len(surfs))]
    n = sum(counts)
    segs = G.segments(np.arange(len(surfs)), counts)
    P = torch.rand(3, n, dtype=torch.float64, generator=torch.Generator().manual_seed(5)).cuda()
    x, y, z = (t.contiguous() for t in P)
    o = G.default_opts(seed_mode=G.SEED_GRID_STEP, **MIXED)
    ref = [t.clone() for t in b.invert(segs, x, y, z, o)]
    new = lambda: [torch.zeros(n, dtype=t.dtype, device="cuda") for t in ref]  # noqa: E731
    eager, errors, stop = [new() for _ in range(300)], [], threading.Event()
    torch.cuda.synchronize()

    def calls():
        st = torch.cuda.Stream()
        try:
            for out in eager:
                b.invert(segs, x, y, z, o, out=out, stream=st)
        except Exception as e:  # noqa: BLE001
            errors.append(e)
        st.synchronize()
        stop.set()

    st, outs, graphs = torch.cuda.Stream(), [], []
    t = threading.Thread(target=calls)
    t.start()
    while not stop.is_set() or len(graphs) < 4:
        outs.append(new())
        st.wait_stream(torch.cuda.current_stream())
        graphs.append(b.graph(segs, x, y, z, *outs[-1], o, stream=st))
        graphs[-1].launch(stream=st)
        if len(graphs) == 60:
            break
    t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for k, out in enumerate(eager + outs):
        assert all(torch.equal(a.view(torch.uint8), r.view(torch.uint8)) for a, r in zip(out, ref)), k
    for g in graphs:
        g.close()
    b.close()
