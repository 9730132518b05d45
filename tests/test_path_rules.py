"""CPU check of the rules that send an inversion to one kernel or another (gpu-nurbs_amd/csrc/path_rules.hpp):
the sizes at which the GPU tests mean to reach the persistent kernels lie on their side of the rules, for
256 compute units."""
import os
import subprocess

import pytest

import test_gpu_batch_refill as batch_refill
import test_gpu_persistent_calls as persistent

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include "path_rules.hpp"
#include <cstdio>
#include <cstdlib>
#include <cstring>
// batch GRP POINTS SEVERAL | call P Q KNOTS POINTS, then MIXED NEWTON64 MAX_ITER FP32_ITERS FP64_TAIL: 1 if persistent
int main(int argc, char **argv) {
    auto n = [&](int k) { return (size_t)atoll(argv[k]); };
    const int at = argc - 5;
    const gn::PathOpts o{n(at) != 0, n(at + 1) != 0, (int)n(at + 2), (int)n(at + 3), (int)n(at + 4)};
    if (!strcmp(argv[1], "batch")) printf("%d", (int)gn::batch_takes_refill((int)n(2), n(3), n(4) != 0, o, 256));
    else printf("%d", (int)!gn::call_takes_tile((int)n(2), (int)n(3), n(4), n(5), o, 256));
    return 0;
}
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(DRIVER)
    inc = os.path.join(ROOT, "gpu-nurbs_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", inc, "-o", str(d / "rules"), str(d / "rules.cpp")], check=True)

    def ask(kind, *args, mixed=False, newton64=False, max_iter=20, fp32_iters=20, fp64_tail=3):
        cmd = [kind, *args, int(mixed), int(newton64), max_iter, fp32_iters, fp64_tail]
        out = subprocess.run([str(d / "rules"), *map(str, cmd)], capture_output=True, text=True, check=True)
        return out.stdout == "1"
    return ask


@pytest.mark.parametrize("grp", [0, 1, 2])
def test_batches_of_the_refill_tests_are_persistent(rule, grp):
    n = sum(c for c, (p, q) in zip(batch_refill.counts(), batch_refill.DEGREES) if batch_refill.group(p, q) == grp)
    assert rule("batch", grp, n, 1, newton64=True, max_iter=batch_refill.PLAIN["max_iter"])
    m = batch_refill.MIXED
    assert rule("batch", grp, n, 1, mixed=True, fp32_iters=m["fp32_iters"], fp64_tail=m["fp64_tail"])


def test_batch_rule(rule):
    """Up to half a round of waves every chain is short enough to wait for; long chains in many rounds are not."""
    waves = {True: (8, 4, 4), False: (4, 3, 2)}
    long = dict(newton64=True, max_iter=100, fp32_iters=30, fp64_tail=40)
    for grp in (0, 1, 2):
        for mixed in (False, True):
            half = 32 * 256 * waves[mixed][grp]
            for several in (0, 1):
                assert not rule("batch", grp, half // 2, several, mixed=mixed, **long)
                assert rule("batch", grp, 8 * half, several, mixed=mixed, **long)
    for several in (0, 1):
        assert not rule("batch", 0, 1 << 24, several, max_iter=20) and rule("batch", 0, 1 << 24, several, max_iter=21)
        assert not rule("batch", 0, 1 << 24, several, mixed=True, fp32_iters=6, fp64_tail=3)


def _call(rule, p, q, n, opts, newton64=True):
    knots = 20 + p + 1 + 23 + q + 1
    return rule("call", p, q, knots, n, mixed=True, newton64=newton64, fp32_iters=opts.get("fp32_iters", 20),
                fp64_tail=opts.get("fp64_tail", 3))


def test_calls_of_the_persistent_tests_are_persistent(rule):
    for p, q, opts, n in persistent.BITS:
        assert _call(rule, p, q, n, opts) and not _call(rule, p, q, persistent.SMALL, opts), (p, q, n)
    assert all(_call(rule, 3, 3, n, persistent.SHORT) for n in persistent.NOALLOC)
    assert _call(rule, 3, 3, persistent.STREAMS, persistent.DEFAULT)
    assert _call(rule, 2, 2, persistent.SLOW, persistent.LONG)


def test_call_rule(rule):
    """Every class reaches both sides, in both precisions; other degrees and long knot vectors never the tile."""
    for p in range(2, 6):
        for q in range(2, 6):
            for mixed in (False, True):
                assert not rule("call", p, q, 60, 4096, mixed=mixed) and rule("call", p, q, 60, 1 << 23, mixed=mixed)
                assert rule("call", p, q, 1025, 4096, mixed=mixed)
                n = [next(k for k in range(1, 24) if rule("call", p, q, 60, 1 << k, mixed=mixed, newton64=True, max_iter=m,
                                                          fp32_iters=m)) for m in (20, 200)]
                assert n[1] <= n[0]  # longer chains leave the tile kernel earlier
    assert rule("call", 1, 3, 60, 64) and rule("call", 3, 6, 60, 64)
