"""The allocator's work, measured through its public entry points.

Every case is one workload a program on this allocator runs: it initializes
the heap once (prepare), then makes passes that allocate, use and free blocks
(run).  Every pass leaves the heap empty, so passes can follow each other on
one heap.  Lane counts, sizes, tags and orders come from the seed; lane counts
lie up to 1/64 below the case's, as a program's arrays are seldom round.
"""
from __future__ import annotations

import math

import numpy as np

import halloc_amd as H
from halloc_amd import autotune, harness
from halloc_amd.workloads import graph_sizes, pages_for, serving_requests, sweep_sizes

MIB = 1 << 20


def listed():
    return [
        # a handful of blocks kept across launches (one small array per
        # object): allocate, read back, free, three calls of one wave each
        {"name": "array_small", "kind": "array", "n": 64, "lo": 16, "hi": 256, "memory": 512 * MIB},
        # the headline: every lane of a full grid allocates, uses and frees one
        # 16 B block, launch after launch, library defaults
        {"name": "pairs_16", "kind": "pairs", "n": 1 << 20, "bs": 256, "size": 16, "iters": 1, "launches": 25,
         "memory": 512 * MIB},
        # the same with a block in the middle of the classes, an odd block
        # length (3 units), a part-filled grid and a loop inside the kernel
        {"name": "pairs_192", "kind": "pairs", "n": 300_000, "bs": 192, "size": 190, "iters": 8, "launches": 10,
         "memory": 512 * MIB},
        # temporary objects of many sizes inside one kernel (the reference's
        # priv-throughput over 8..256 B)
        {"name": "loop_8_256", "kind": "loop", "n": 1 << 20, "bs": 128, "lo": 8, "hi": 256, "nallocs": 1, "niters": 4,
         "ntries": 2, "memory": 512 * MIB},
        # one kernel builds, another frees, over every size class on the
        # drop-in heap of 512 MiB (the reference's throughput test)
        {"name": "burst_8_3072", "kind": "burst", "n": 1 << 16, "bs": 256, "lo": 8, "hi": 3072, "nallocs": 1,
         "ntries": 4, "memory": 512 * MIB},
        # 24 B list nodes, several per thread: a build kernel and a free kernel
        {"name": "burst_24", "kind": "burst", "n": 1 << 20, "bs": 256, "lo": 24, "hi": 24, "nallocs": 4, "ntries": 2,
         "memory": 512 * MIB},
        # objects that come and go over many launches with most of them live
        # (the reference's phase-throughput with its experiments' fractions)
        {"name": "chain_16_256", "kind": "chain", "n": 1 << 20, "bs": 128, "lo": 16, "hi": 256, "niters": 8,
         "ntries": 4, "memory": 512 * MIB},
        # log-uniform sizes from 16 B to 3 KiB with 1% up to 64 KiB, several
        # per lane, freed in random order
        {"name": "sweep", "kind": "sweep", "n": 1 << 16, "per": 8, "large": 0.01, "memory": 1024 * MIB},
        # buffers above 3 KiB only
        {"name": "large", "kind": "sweep", "n": 6000, "per": 2, "large": 1.0, "memory": 4096 * MIB},
        # graph building in batched calls from one persistent launch, and one
        # node per thread with plain calls
        {"name": "graphs_batched", "kind": "graphs", "njobs": 1024, "batched": True, "memory": 4096 * MIB},
        {"name": "graphs_plain", "kind": "graphs", "njobs": 512, "batched": False, "memory": 4096 * MIB},
        # paged sequences in a resident serving loop, requests queued up
        {"name": "serve", "kind": "serve", "nreq": 20_000, "slots": 65_536, "median": 256, "cap": 2048,
         "rate": 8000, "memory": 4096 * MIB},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("array", "pairs", "pairs", "loop", "burst", "burst", "chain", "sweep", "graphs", "serve"))
    if kind == "array":
        return {"kind": kind, "n": _log(rng, 1, 1 << 17), "lo": rng.choice((1, 16, 40)),
                "hi": rng.choice((64, 256, 1000)), "memory": 512 * MIB}
    if kind == "pairs":
        n = _log(rng, 20_000, 1 << 20)
        # at most 2^19 lanes are resident at once
        size = _log(rng, 16, min(1024, 100 * MIB // min(n, 1 << 19)))
        return {"kind": kind, "n": n, "bs": rng.choice((64, 128, 192, 256)), "size": size,
                "iters": rng.choice((1, 1, 2, 8)), "launches": rng.randint(5, 25), "memory": rng.choice((512, 1024)) * MIB}
    if kind == "loop":
        lo = rng.choice((8, 16, 100))
        return {"kind": kind, "n": _log(rng, 50_000, 1 << 17 if lo == 100 else 1 << 19), "bs": rng.choice((64, 128, 256)), "lo": lo,
                "hi": rng.choice((lo, 256, 512)) if lo < 100 else 1000, "nallocs": 1, "niters": rng.randint(1, 4),
                "ntries": 2, "memory": 512 * MIB}
    if kind == "burst":
        hi = _log(rng, 16, 3072)
        lo = rng.choice((8, hi))
        most = min(1 << 20, int(0.25 * 384 * MIB / (1.4 * max(16, (min(lo, hi) + hi) / 2))))
        return {"kind": kind, "n": _log(rng, max(64, most // 64), most), "bs": rng.choice((64, 128, 256)),
                "lo": min(lo, hi), "hi": hi, "nallocs": 1, "ntries": rng.randint(2, 4), "memory": 512 * MIB}
    if kind == "chain":
        hi = rng.choice((16, 64, 128, 256))
        return {"kind": kind, "n": _log(rng, 100_000, 1 << 20), "bs": rng.choice((64, 128, 256)),
                "lo": min(16, hi), "hi": hi, "niters": rng.choice((1, 4, 8)), "ntries": 4, "memory": 512 * MIB}
    if kind == "sweep":
        large = rng.choice((0.0, 0.01, 1.0))
        per = rng.randint(1, 8)
        most = 1 << 16 if large < 1.0 else 16_000 // (per + 1)  # the large region is a quarter of the pool
        return {"kind": kind, "n": _log(rng, most // 32, most), "per": per,
                "large": large, "memory": (4096 if large == 1.0 else 1024) * MIB}
    if kind == "graphs":
        return {"kind": kind, "njobs": _log(rng, 64, 512), "batched": rng.choice((True, False)),
                "memory": 4096 * MIB}
    return {"kind": kind, "nreq": _log(rng, 1000, 20_000), "slots": 256 * rng.randint(64, 256),
            "median": rng.choice((64, 200, 256)), "cap": rng.choice((512, 1500, 2048)), "rate": 8000,
            "memory": 4096 * MIB}


_heap_of = None  # the case the process's heap was initialized for


def _heap(case):
    """Initializes the heap for the case once: a process has one heap."""
    global _heap_of
    key = {k: v for k, v in case.items() if k != "name"}
    if _heap_of == key:
        return
    opts = H.HallocOpts(memory=case["memory"])
    if case["kind"] == "graphs":
        opts = autotune.opts_of(autotune.load() if case["batched"] else autotune.load_plain(), case["memory"])
    H.Halloc.init(opts)
    _heap_of = key


def _test_args(case, n, seed):
    """The option set of a reference test program, parsed as its command line."""
    test = {"loop": "priv-throughput", "burst": "throughput", "chain": "phase-throughput"}[case["kind"]]
    o = harness.defaults_for(test)
    o.parse([f"-n{n}", f"-T{case['bs']}", f"-s{case['lo']}", f"-S{case['hi']}", "-duniform",
             f"-l{case.get('nallocs', 1)}", f"-i{case.get('niters', 1)}", f"-t{case['ntries']}", f"-m{case['memory']}"]
            + (["-f0.95", "-F0.05", "-e0.91", "-g5"] if case["kind"] == "chain" else []))
    return (harness.TESTS[test], o.nthreads, o.bs, o.ntries, o.nallocs, o.niters, o.alloc_sz, o.max_alloc_sz,
            o.max_alloc_sh, harness.DISTRS[o.distr], o.period_mask, o.group_sh, o.probabs, seed & 0xFFFFFFFF)


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "array":
        s["sizes"] = rng.integers(case["lo"], case["hi"] + 1, case["n"]).astype(np.uint32)
    elif kind in ("pairs", "loop", "burst", "chain"):
        n = case["n"] - int(rng.integers(0, case["n"] // 64 + 1))
        if kind == "pairs":
            s["args"] = dict(nthreads=n, bs=case["bs"], size=case["size"], iters=case["iters"], warmup=0,
                             launches=case["launches"])
        else:
            s["args"] = _test_args(case, n, seed)
    elif kind == "sweep":
        s["sizes"] = sweep_sizes(rng, case["n"], per_max=case["per"], large_frac=case["large"])
        s["order"] = rng.permutation(s["sizes"].size).astype(np.uint32)
    elif kind == "graphs":
        s["nodes"] = graph_sizes(rng, case["njobs"])
        cfg = autotune.load()
        s["args"] = dict(batch=cfg["batch"], waves=cfg["waves"], run_plain=not case["batched"],
                         run_batch=case["batched"], seed=seed & 0xFFFFFFFF)
    else:
        arrival, length, tag = serving_requests(case["nreq"], rate_per_ms=case["rate"], median=case["median"],
                                                cap=case["cap"], seed=seed)
        s["requests"] = (arrival, length, tag)
        s["args"] = dict(slots=case["slots"], watermark=64 * MIB)
    return s


def prepare(case, seed):
    _heap(case)
    return _inputs(case, seed)


def run(state):
    kind = state["kind"]
    if kind == "array":
        ptrs = H.Halloc.malloc_sizes(state["sizes"])
        words = H.Halloc.read_words(ptrs)  # each block holds its size
        H.Halloc.free_ptrs(ptrs)
        return {"words": words}
    if kind == "pairs":
        a = state["args"]
        r = H.Halloc.run_plain(**a)
        # run_plain makes its launches twice: back to back, and each timed
        served = 2 * a["launches"] * a["iters"] * a["nthreads"] - r["nulls"]
        return {"served": served, "nulls": r["nulls"], "errors": r["errors"]}
    if kind in ("loop", "burst", "chain"):
        r = H.Halloc.run_test(*state["args"])
        return {k: r[k] for k in ("mallocs", "frees", "nulls", "checks_failed")}
    if kind == "sweep":
        r = H.Halloc.run_lists(state["sizes"], state["order"])
        return {k: r[k] for k in ("requests", "nulls", "errors")}
    if kind == "graphs":
        r = H.Halloc.run_graphs(state["nodes"], **state["args"])
        return {k: r[k] for k in ("nodes", "nulls", "errors")}
    r = H.Halloc.run_serve(*state["requests"], **state["args"])
    return {k: r[k] for k in ("checksum", "produced", "bad", "pages", "nulls", "completed")}


# A block's share of the allocator's state: its occupancy bit and its 4-bit
# length, read and written by the malloc and by the free.
STATE_BYTES = 5 * 4 / 8


def work(case):
    kind = case["kind"]
    if kind == "array":  # sizes in, pointers out and in twice, words written and read back
        return {"bytes": case["n"] * (4 + 8 + 8 + 8 + 4 + 4 + 4 + STATE_BYTES), "flops": 0}
    if kind == "pairs":  # 16 B written and read back per block
        pairs = 2 * case["launches"] * case["iters"] * case["n"]
        return {"bytes": pairs * (32 + STATE_BYTES), "flops": 0}
    if kind in ("loop", "burst"):  # a pointer stored and loaded per block
        pairs = case["n"] * case["nallocs"] * case.get("niters", 1) * case["ntries"]
        return {"bytes": pairs * (16 + STATE_BYTES), "flops": 0}
    if kind == "chain":  # every thread's state per launch; 0.95 - 0.05 of the threads change per phase pair
        pairs = 0.9 * case["n"] * max(1, case["niters"] * case["ntries"] // 2)
        return {"bytes": pairs * (16 + STATE_BYTES) + case["n"] * 8 * case["ntries"], "flops": 0}
    if kind == "sweep":  # size, pointer and order entry per slot, the stamp written and read per block
        slots = case["n"] * case["per"]
        return {"bytes": slots * (4 + 8 + 8 + 4 + 4) + (slots + case["n"]) / 2 * (8 + STATE_BYTES), "flops": 0}
    if kind == "graphs":  # per node a header, 8 targets on average and a table entry, written and read
        nodes = case["njobs"] * (65536 - 1024) / math.log(64)
        return {"bytes": nodes * (2 * (16 + 32 + 8) + 2 * STATE_BYTES), "flops": 0}
    # 16 B per token written and read, 8 B per page pointer
    tokens = case["nreq"] * min(case["cap"], case["median"] * math.exp(0.5))
    return {"bytes": tokens * 32 + tokens / 16 * (16 + STATE_BYTES), "flops": 0}


def _hash3(a, b, c):
    a, b, c = (np.asarray(x, dtype=np.uint32) for x in (a, b, c))
    with np.errstate(over="ignore"):
        x = a * np.uint32(0x9E3779B1) ^ (b + np.uint32(0x7F4A7C15)) * np.uint32(0x85EBCA77)
        x = x ^ (c + np.uint32(0x165667B1)) * np.uint32(0xC2B2AE3D)
        x ^= x >> np.uint32(16)
        x *= np.uint32(0x7FEB352D)
        x ^= x >> np.uint32(15)
        x *= np.uint32(0x846CA68B)
        x ^= x >> np.uint32(16)
    return x


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "array":
        return {"words": s["sizes"]}
    if kind == "pairs":
        a = s["args"]
        return {"served": 2 * a["launches"] * a["iters"] * a["nthreads"], "nulls": 0, "errors": 0}
    if kind in ("loop", "burst"):
        pairs = s["args"][1] * case["nallocs"] * case.get("niters", 1) * case["ntries"]
        return {"mallocs": pairs, "frees": pairs, "nulls": 0, "checks_failed": 0}
    if kind == "chain":
        return {"mallocs": None, "frees": None, "nulls": 0, "checks_failed": 0}
    if kind == "sweep":
        return {"requests": int((s["sizes"] != 0).sum()), "nulls": 0, "errors": 0}
    if kind == "graphs":
        return {"nodes": int(s["nodes"].sum()), "nulls": 0, "errors": 0}
    _, length, tag = s["requests"]
    # the checksum of a request: the sum of its tokens' hashes
    n = length.astype(np.int64)
    starts = np.concatenate(([0], np.cumsum(n)[:-1]))
    t = np.arange(int(n.sum()), dtype=np.int64) - np.repeat(starts, n)
    h = _hash3(np.repeat(tag, n), t.astype(np.uint32), np.uint32(0x5E7A11C3)).astype(np.uint64)
    checksum = (np.add.reduceat(h, starts) & 0xFFFFFFFF).astype(np.uint32)
    return {"checksum": checksum, "produced": length, "bad": np.zeros(len(n), np.uint32),
            "pages": int(pages_for(length).sum()), "nulls": 0, "completed": len(n)}
