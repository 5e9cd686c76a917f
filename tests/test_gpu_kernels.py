"""Edges of the device paths that the workload tests reach only by chance."""
import numpy as np
import pytest

import halloc_amd as H
from halloc_amd import harness

pytestmark = pytest.mark.gpu


@pytest.fixture
def heap():
    started = []

    def start(opts):
        H.Halloc.init(opts)
        started.append(opts)
        return opts

    yield start
    if started:
        H.Halloc.shutdown()


def run(test, n, bs, size, nallocs=1, ntries=1, period=0, group=0, memory=64 << 20, probabs=((1.0, 1.0), (1.0, 1.0))):
    return H.Halloc.run_test(harness.TESTS[test], n, bs, ntries, nallocs, 1, size, size, 0, 1, period, group, probabs, 1)


@pytest.mark.parametrize("test", ["throughput", "latency", "phase-throughput", "phase-latency"])
@pytest.mark.parametrize("n,bs,nallocs,period,group", [(1, 1, 1, 0, 0), (63, 64, 3, 0, 0), (40000, 100, 2, 0, 0),
                                                       (60001, 256, 2, 1, 5), (65536, 256, 1, 0, 0)])
def test_null_check_counts_the_nulls_held(heap, test, n, bs, nallocs, period, group):
    # blocks of 3072 B on a 48 MiB slab heap: 16384 fit at most, so the larger
    # grids get NULLs.  One step from empty: every NULL returned is still held
    # when the check runs, so its count is the malloc kernel's own count, and
    # the first try is the one that fails
    print(f"[gpu] null check {test} n={n} bs={bs} nallocs={nallocs} period={period}", flush=True)
    heap(H.HallocOpts(memory=64 << 20, sb_sz_sh=21, nheads=1))
    r = run(test, n, bs, 3072, nallocs, period=period, group=group)
    active = sum(1 for i in range(n) if not (i >> group) & period)
    assert r["mallocs"] + r["nulls"] == active * nallocs
    assert (r["nulls"] > 0) == (active * nallocs > 16384)
    assert r["checks_failed"] == r["nulls"]
    assert r["failed_try"] == (0 if r["nulls"] else -1)
    assert r["mallocs"] == r["frees"]
