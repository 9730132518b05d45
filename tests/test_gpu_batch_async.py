"""A batched call waits for no work on another stream, however many calls are in flight there and however
long its own tile list is."""
import time

import numpy as np
import pytest
import torch

import gnurbs as G
from gnurbs import synth

pytestmark = pytest.mark.gpu

N = 200_000


@pytest.fixture(scope="module")
def work():
    sd = synth.surface_G(12, 12, 3, 3, seed=5)
    s = G.Surface(sd.p, sd.q, sd.ku, sd.kv, sd.cp, sd.w)
    s.BuildTree(2)
    P = torch.rand(3, N, dtype=torch.float64, device="cuda")
    yield s, P, G.default_opts(max_iter=4)


def _segs(pieces):
    counts = np.full(pieces, N // pieces)
    counts[0] += N - counts.sum()
    return G.segments(np.zeros(pieces, dtype=np.int64), counts)


def _outs(k):
    return [[torch.zeros(N, dtype=d, device="cuda") for d in (torch.float64, torch.float64, torch.uint8)] for _ in range(k)]


def _sleep(stream, seconds):
    """Keeps the stream busy."""
    def run(c):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        with torch.cuda.stream(stream):
            torch.cuda._sleep(c)
        torch.cuda.synchronize()
        return time.perf_counter() - t0
    run(1000)
    cycles = int(20_000_000 * seconds / run(20_000_000))
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    with torch.cuda.stream(stream):
        torch.cuda._sleep(cycles)
    return t0


def _streams():
    """Two streams that share no hardware queue: work on the second ends while the first is busy."""
    s1 = torch.cuda.Stream()
    for _ in range(12):
        s2 = torch.cuda.Stream()
        t0 = _sleep(s1, 0.05)
        with torch.cuda.stream(s2):
            torch.cuda._sleep(1000)
        s2.synchronize()
        free = time.perf_counter() - t0 < 0.025
        torch.cuda.synchronize()
        if free:
            return s1, s2
    pytest.skip("every stream shares the first one's hardware queue")


def _check(outs, ref):
    torch.cuda.synchronize()
    for k, out in enumerate(outs):
        assert all(torch.equal(a, r) for a, r in zip(out, ref)), k


def test_eight_calls_in_flight_do_not_hold_up_another_stream(work):
    s, P, o = work
    b = G.Batch([s])
    ref = [t.clone() for t in b.invert(_segs(3), *P, o)]
    outs = _outs(12)
    s1, s2 = _streams()
    t0 = _sleep(s1, 0.5)
    for out in outs[:8]:
        b.invert(_segs(3), *P, o, out=out, stream=s1)
    for out in outs[8:]:
        b.invert(_segs(3), *P, o, out=out, stream=s2)
    s2.synchronize()
    other = time.perf_counter() - t0
    torch.cuda.synchronize()
    whole = time.perf_counter() - t0
    _check(outs, ref)
    assert whole > 0.3 and other < 0.5 * whole, (other, whole)
    b.close()


def test_a_longer_list_does_not_wait_for_the_device(work):
    """All staging buffers are too small for the call's list."""
    s, P, o = work
    b = G.Batch([s])
    b.set_shape(64, 0)
    ref = [t.clone() for t in b.invert(_segs(3), *P, o)]
    outs = _outs(9)
    s1, s2 = _streams()
    _sleep(s1, 0.05)
    for out in outs[:8]:
        b.invert(_segs(3), *P, o, out=out, stream=s1)
    _check(outs[:8], ref)
    t0 = _sleep(s1, 0.5)
    b.invert(_segs(50_000), *P, o, out=outs[8], stream=s2)
    s2.synchronize()
    other = time.perf_counter() - t0
    torch.cuda.synchronize()
    whole = time.perf_counter() - t0
    _check(outs, ref)
    assert whole > 0.3 and other < 0.5 * whole, (other, whole)
    b.close()


def test_device_bytes_count_the_staging(work):
    """The memory of a batch's staging buffers, from its creation on and as they grow."""
    s, P, o = work
    free = torch.cuda.mem_get_info()[0]
    b = G.Batch([s])
    size = lambda: int(G.lib().gn_batch_device_bytes(b._h))  # noqa: E731
    first = size()
    assert abs((free - torch.cuda.mem_get_info()[0]) - first) <= 8 << 20  # (allocations are rounded up)
    b.set_shape(64, 0)
    b.invert(_segs(50_000), *P, o)
    torch.cuda.synchronize()
    assert size() - first >= 50_000 * 32
    grown = size()
    b.invert(_segs(50_000), *P, o)
    torch.cuda.synchronize()
    assert size() == grown
    b.close()
