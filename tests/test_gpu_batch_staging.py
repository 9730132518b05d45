"""The batch's staging buffers: more calls in flight than buffers, on several streams and threads, with
tile lists of different lengths (buffers grow and are reused), give every call the bits it gets alone."""
import threading

import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu


def _calls(b, nobj, n, seed, count):
    """Segment lists from one point to all points, cut at random."""
    rng = np.random.default_rng(seed)
    out = []
    for k in range(count):
        m = int(rng.integers(1, n + 1)) if k else n
        pieces = int(rng.integers(1, 9)) if k % 4 else 400
        cuts = np.sort(rng.integers(0, m + 1, pieces - 1))
        counts = np.diff(np.r_[0, cuts, m])
        out.append(G.segments(rng.integers(0, nobj, pieces), counts))
    return out


@pytest.mark.parametrize("threads", [1, 3])
def test_many_calls_in_flight(threads):
    defs = [synth.surface_G(6 + i, 9, 2 + i % 4, 2 + i // 4, seed=80 + i, jitter=0.2) for i in range(8)]
    surfs = [G.Surface(d.p, d.q, d.ku, d.kv, d.cp, d.w) for d in defs]
    for s in surfs:
        s.BuildTree(2)
    b = G.Batch(surfs)
    b.set_shape(64, 0)
    n = 20000
    gen = torch.Generator(device="cuda").manual_seed(3)
    x, y, z = (torch.rand(n, dtype=torch.float64, device="cuda", generator=gen) for _ in range(3))
    o = G.default_opts(max_iter=5)
    work = [_calls(b, len(surfs), n, 10 + t, 24) for t in range(threads)]

    def new():
        return (torch.full((n,), -1.0, dtype=torch.float64, device="cuda"),
                torch.full((n,), -1.0, dtype=torch.float64, device="cuda"),
                torch.full((n,), 99, dtype=torch.uint8, device="cuda"))

    ref = []
    for lists in work:
        r = []
        for segs in lists:
            out = new()
            b.invert(segs, x, y, z, o, out=out)
            torch.cuda.synchronize()
            r.append(out)
        ref.append(r)
    got = [[new() for _ in lists] for lists in work]
    torch.cuda.synchronize()

    def run(t):
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        for k, segs in enumerate(work[t]):
            b.invert(segs, x, y, z, o, out=got[t][k], stream=streams[k % 2])

    ts = [threading.Thread(target=run, args=(t,)) for t in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    torch.cuda.synchronize()
    for t in range(threads):
        for k in range(len(work[t])):
            for a, r in zip(got[t][k], ref[t][k]):
                assert torch.equal(a, r), (t, k)
    b.close()
