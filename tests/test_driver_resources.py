"""CPU checks of the drivers' host code: what they do with streams, events and device buffers on every way
out.  The built library runs on a HIP runtime of host memory (tests/native/fake_hip.cpp) in a process of its
own; no kernel runs."""
import os
import re
import subprocess
import sys

import pytest

import halloc_amd as H

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PRELUDE = """
import ctypes, sys
import numpy as np
import halloc_amd as H
from halloc_amd import harness
from halloc_amd.workloads import graph_sizes
H.lib()
fake = ctypes.CDLL("libamdhip64.so.7")
fake.fake_live.restype = ctypes.c_long
fake.fake_fail_at.argtypes = [ctypes.c_long]
fake.fake_limit.argtypes = [ctypes.c_size_t]
STREAMS, EVENTS, BUFFERS, GRAPHS, WRONG, CALLS, USED = range(7)
live = fake.fake_live
OPTS = H.HallocOpts(memory=64 << 20, sb_sz_sh=21, nheads=1)

def refused(f, match):
    try:
        f()
    except H.HallocError as e:
        assert match in str(e), e
    else:
        raise AssertionError("not refused")
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    """A directory that holds the stand-in runtime, its symbols under the versions the library asks for."""
    d = tmp_path_factory.mktemp("fake_hip")
    if not os.path.exists(H.LIB_PATH):
        from halloc_amd import build
        build.build()
    out = subprocess.run(["nm", "-D", "--undefined-only", H.LIB_PATH], capture_output=True, text=True, check=True).stdout
    vers = {}
    for name, ver in re.findall(r"\bU (\w+)@+(hip_[\d.]+)", out):
        vers.setdefault(ver, []).append(name)
    with open(d / "map", "w") as f:
        for ver, names in vers.items():
            f.write("%s { global: %s; };\n" % (ver, "; ".join(names)))
        f.write("test { global: fake_*; local: *; };\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    "-Wno-deprecated-declarations", f"-Wl,--version-script={d}/map", "-Wl,-soname,libamdhip64.so.7",
                    "-o", str(d / "libamdhip64.so.7"), os.path.join(HERE, "native", "fake_hip.cpp")], check=True)
    return d


def run(fake, script):
    env = dict(os.environ, LD_LIBRARY_PATH=str(fake), PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", PRELUDE + script], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]


def test_refused_long_order_keeps_nothing(fake):
    # 128 Ki slots and more are checked on the device, after buffers and a
    # stream were taken: a refused call leaves nothing behind
    run(fake, """
H.Halloc.init(OPTS)
base = live(BUFFERS)
n = 1 << 17
sizes = np.full((1, n), 16, np.uint32)
bad = np.zeros(n, np.uint32)
for _ in range(5):
    refused(lambda: H.Halloc.run_lists(sizes, bad), "permutation")
    assert live(STREAMS) == 0 and live(EVENTS) == 0 and live(BUFFERS) == base, [live(i) for i in range(4)]
H.Halloc.run_lists(sizes, np.arange(n, dtype=np.uint32))
H.Halloc.shutdown()
assert [live(i) for i in range(5)] == [0] * 5
""")


def test_bad_order_is_refused_as_one_when_memory_is_short(fake):
    run(fake, """
H.Halloc.init(OPTS)
n = 1 << 17
sizes = np.full((1, n), 16, np.uint32)
bad, good = np.zeros(n, np.uint32), np.arange(n, dtype=np.uint32)
full = live(USED)
for room in (0, 4 * n, 12 * n, 13 * n):
    fake.fake_limit(full + room)
    refused(lambda: H.Halloc.run_lists(sizes, bad), "permutation")
    refused(lambda: H.Halloc.run_lists(sizes, good), "memory")
    refused(lambda: H.Halloc.run_lists(sizes), "memory") if room < 12 * n else None
    assert live(USED) == full
fake.fake_limit(1 << 40)
assert H.Halloc.run_lists(sizes, good)["nulls"] == 0  # no error is left behind
""")


DRIVERS = {
    "plain": "H.Halloc.run_plain(nthreads=64, launches=3)",
    "arrays": "H.Halloc.free_ptrs(H.Halloc.malloc_sizes(np.full(9, 16, np.uint32)))",
    "lists": "H.Halloc.run_lists(np.full((2, 70000), 16, np.uint32), np.arange(140000, dtype=np.uint32))",
    "throughput": "rt('throughput')",
    "latency": "rt('latency')",
    "phase": "rt('phase-throughput')",
    "checked": "rt('checkptr')",
    "extfrag": "rt('phase-extfrag')",
    "priv": "rt('priv-throughput')",
    "graphs": "H.Halloc.run_graphs(graph_sizes(np.random.default_rng(1), 8), batch=4, waves=4, run_plain=True,"
              " run_batch=True, seed=1)",
    "serve": "H.Halloc.run_serve(np.zeros(9, np.uint64), np.full(9, 5, np.uint32), np.arange(9, dtype=np.uint32),"
             " slots=256, watermark=0)",
    "corr": "H.Halloc.run_corr_test0(128, 1, 64)",
    "copy": "H.Halloc.probe_copy(1 << 20, 2)",
    "touch": "H.Halloc.run_touch(n=256, words=2, iters=1, reps=1)",
    "stepped": "H.Halloc.run_phase(nthreads=64, bs=64, nphases=2, max_steps=3)",
    "points": "H.Halloc.run_sample('grid-points', 64, 64, ncells=4)",
    "strings": "H.Halloc.run_sample('add-strings', 64, 64)",
    "replay": "H.Halloc.replay(np.ones((2, 64, 2), np.uint32))",
    "batches": "H.Halloc.replay_batch(np.ones((2, 64, 4), np.uint32))",
}


@pytest.mark.parametrize("name", sorted(DRIVERS))
def test_failed_call_leaves_no_handles(fake, name):
    # the k-th HIP call of the driver fails, for every k: nothing of the failed
    # call is kept for later ones (it may have left work behind), and with what
    # finished calls gave back released no stream, event or buffer is left.
    # The samples' steps and the two array calls each give back their own.
    run(fake, """
def rt(test):
    o = harness.defaults_for(test)
    o.parse(["-n100", "-T64", "-s16", "-S16", "-l1", "-i1", "-t2"])
    return H.Halloc.run_test(harness.TESTS[test], o.nthreads, o.bs, o.ntries, o.nallocs, o.niters, o.alloc_sz,
                             o.max_alloc_sz, o.max_alloc_sh, harness.DISTRS[o.distr], o.period_mask, o.group_sh,
                             o.probabs, 1)
def call():
    return %s
H.Halloc.init(OPTS)
fake.fake_fail_at(0)
call()
total = live(CALLS)
assert total > 3
for pooled in (False, True):
    for k in range(1, total + 1):
        fake.fake_fail_at(0)
        H.Halloc.init(OPTS)  # gives back what was kept
        base = live(BUFFERS)
        if pooled:
            call()
        fake.fake_fail_at(k)
        try:
            call()
        except H.HallocError:
            left = [live(i) for i in (STREAMS, EVENTS, BUFFERS)]
            assert pooled or %r or left == [0, 0, base], (k, left)
        fake.hipGetLastError()  # the runtime's own record of the failure
        fake.fake_fail_at(0)
        H.Halloc.shutdown()
        left = [live(i) for i in (STREAMS, EVENTS, BUFFERS, WRONG)]
        assert left == [0] * 4, (k, left)
""" % (DRIVERS[name], name in ("points", "strings", "arrays")))


def test_kept_buffers_are_bounded_and_given_back(fake):
    # what finished calls leave for later ones stays within its bound, and one
    # call gives it back while the heap lives
    run(fake, """
H.Halloc.init(OPTS)
base, heap = live(BUFFERS), live(USED)
for n in (1 << 10, 1 << 20, 5 << 20, 1 << 20, 9 << 20, 7 << 20, 3):
    H.Halloc.run_lists(np.full((1, n), 16, np.uint32))
    assert live(USED) - heap <= 256 << 20, (n, live(USED) - heap)
    assert live(BUFFERS) - base <= 32
assert live(USED) > heap and live(STREAMS) and live(EVENTS)
H.Halloc.release_buffers()
assert [live(i) for i in (STREAMS, EVENTS, BUFFERS, WRONG)] == [0, 0, base, 0] and live(USED) == heap
assert H.Halloc.run_lists(np.full((1, 100), 16, np.uint32))["requests"] == 100
H.Halloc.release_buffers()
H.Halloc.release_buffers()
assert live(USED) == heap
""")
