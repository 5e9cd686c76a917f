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


@pytest.mark.parametrize("test", ["phase-throughput", "phase-latency"])
@pytest.mark.parametrize("n,bs,period,group", [(24000, 100, 0, 0), (23999, 256, 0, 0), (48000, 64, 1, 5)])
def test_null_check_names_the_first_failing_try(heap, test, n, bs, period, group):
    # half of the threads without a block allocate at each even try and nothing
    # is freed: 12 000 blocks of 3072 B fit a 48 MiB slab heap, 18 000 do not, so
    # the NULLs begin at try 2, and every later check counts all that are held
    print(f"[gpu] first failing try {test} n={n} bs={bs} period={period}", flush=True)
    opts = H.HallocOpts(memory=64 << 20, sb_sz_sh=21, nheads=1)
    for ntries in range(1, 5):
        heap(opts)  # starts an empty heap
        r = run(test, n, bs, 3072, ntries=ntries, period=period, group=group, probabs=((0.5, 0.0), (0.0, 0.0)))
        assert (r["nulls"] > 0) == (ntries > 2)
        assert r["failed_try"] == (2 if ntries > 2 else -1)
        assert r["checks_failed"] == max(ntries - 2, 0) * r["nulls"]  # try 3 changes nothing
        assert r["mallocs"] == r["frees"]


# lanes that take part in a batched call: a wave whose low lanes are inactive
# (the per-round values must not be kept in lanes 0..15), fewer lanes than
# rounds, every other lane, one lane
PARTIAL_WAVES = {"high": range(16, 64), "few": range(40, 47), "odd": range(1, 64, 2), "mixed": [2, 3, 9, 11, 14, 30, 31, 55],
                 "last": [63], "sixteen": range(48, 64)}


def partial_batch_ops(lanes, sizes=(16, 48, 128, 24, 700, 3072), cnt=16):
    """Every size: two batches of cnt blocks per lane, the first freed, then freed again (nothing happens),
    then the second freed together with a third batch's allocation by the other lanes."""
    rows = []
    for sz in sizes:
        r = len(rows)
        for kind in (1, 1, 3, 2, 2):
            row = np.zeros((64, 4), dtype=np.uint32)
            for l in lanes:
                src = {3: r, 2: r if len(rows) == r + 3 else r + 1}.get(kind, 0)
                row[l] = (1, sz, cnt - l % 3, 0) if kind == 1 else (kind, src * 64 + l, 0, 0)
            rows.append(row)
    return np.stack(rows)


@pytest.mark.parametrize("which", sorted(PARTIAL_WAVES))
def test_batched_free_of_a_partial_wave(heap, which):
    # bit-exact against the host model, and the heap empty at the end
    from oracle import model as M
    print(f"[gpu] batched free, lanes {which}", flush=True)
    opts = heap(H.HallocOpts(memory=256 << 20, sb_sz_sh=21, nheads=1))
    ops = partial_batch_ops(PARTIAL_WAVES[which])
    recs, xcc = H.Halloc.replay_batch(ops)
    m = M.ModelHeap(M.make_opts(memory=opts.memory, sb_sz_sh=opts.sb_sz_sh, nheads=1, hash_mode=1))
    want = m.replay_batch(ops, xcc % 1)
    assert (recs == want).all()
    d = H.Halloc.dump()
    assert (d == m.dump()).all()
    assert ((d[:H.Halloc.geometry()["nsbs"]] >> np.uint64(32)) == 0).all()


def refill_program(sizes, nsteps, keep, seed):
    """One wave of mixed sizes from `sizes`, freeing a share of the live blocks
    that alternates between (1 - keep) and keep of the allocations, so that
    slabs pass their busy threshold in both directions again and again."""
    rng = np.random.default_rng(seed)
    ops = np.zeros((nsteps, 64, 2), dtype=np.uint32)
    live = []
    for st in range(nsteps):
        p = keep if (st // 20) % 2 else 1 - keep
        for l in range(64):
            if live and rng.random() < p:
                ops[st, l] = (2, live.pop(int(rng.integers(len(live)))))
            else:
                ops[st, l] = (1, int(rng.choice(sizes)))
        live.extend(st * 64 + l for l in range(64) if ops[st, l, 0] == 1)
    return ops


@pytest.mark.parametrize("nheads,memory,sizes", [(1, 16 << 20, (700, 1500, 3000, 100, 200)), (1, 12 << 20, (3072,)),
                                                 (1, 12 << 20, (256, 384)), (1, 12 << 20, (16, 24)), (1, 12 << 20, (128, 192)),
                                                 (8, 40 << 20, (700, 1500, 3000, 100, 200))])
def test_heads_pass_the_busy_threshold_both_ways(heap, nheads, memory, sizes):
    # full heads, shared heads, heads filled past the threshold and exhaustion:
    # records and state equal the host model's bit for bit
    from oracle import model as M
    print(f"[gpu] busy threshold nheads={nheads} sizes={sizes}", flush=True)
    heap(H.HallocOpts(memory=memory, sb_sz_sh=21, nheads=nheads))
    nh = H.Halloc.geometry()["nheads"]
    ops = refill_program(sizes, 240, 0.3, 11)
    ih = np.arange(240, dtype=np.uint32) % nh
    recs, _ = H.Halloc.replay(ops, ih)
    m = M.ModelHeap(M.make_opts(memory=memory, sb_sz_sh=21, nheads=nheads, hash_mode=1))
    want, _ = m.replay(ops, ih)
    assert (recs == want).all()
    assert (H.Halloc.dump() == m.dump()).all()


def unmarked_full_slabs():
    """Slabs whose count is at their class's busy threshold and whose mark is not set."""
    g, d, marks = H.Halloc.geometry(), H.Halloc.dump(), H.Halloc.full_marks()
    n = g["nsbs"]
    count = (d[:n] >> np.uint64(32)).astype(np.int64)
    size_id = (d[n:3 * n:2] & np.uint64(0xFFFFFFFF)).astype(np.int64)
    busy = np.append(np.array(g["size_table"])[:, H.SIZE_TABLE_FIELDS.index("busy")].astype(np.int64), 1 << 40)
    full = count >= busy[np.minimum(size_id, H.NSIZES)]
    return int(full.sum()), np.nonzero(full & (marks == 0))[0].tolist()


# sizes of one chunk size each: 16, 24, 256 and 384 B
@pytest.mark.parametrize("nheads,sizes", [(1, (3072,)), (1, (16,)), (8, (256,)), (8, (48,)), (2, (16, 24, 256, 384)),
                                          (8, (128, 192, 2048, 3072))])
def test_marks_follow_the_counts_of_many_waves(heap, nheads, sizes):
    # the heap is filled until hamalloc returns NULL, then a share of the blocks
    # is freed again and again while other waves allocate: many slabs pass the
    # threshold in both directions, between them in one kernel (loops on a heap
    # kept near full), and every full slab is marked at the end of each step
    print(f"[gpu] full marks nheads={nheads} sizes={sizes}", flush=True)
    heap(H.HallocOpts(memory=40 << 20, sb_sz_sh=21, nheads=nheads))
    rng = np.random.default_rng(len(sizes) + nheads)
    n = int(1.3 * H.Halloc.geometry()["arena_bytes"] / np.mean(sizes))
    live = np.zeros(0, np.uint64)
    seen = 0
    for keep in (0.9, 0.8, 0.95, 0.5, 0.85, 0.0):
        p = H.Halloc.malloc_sizes(rng.choice(sizes, max(n - live.size, 64)).astype(np.uint32), 256)
        live = np.concatenate([live, p[p != 0]])
        rng.shuffle(live)
        full, bad = unmarked_full_slabs()
        assert not bad
        seen += full
        k = int(keep * live.size)
        H.Halloc.free_ptrs(live[k:])
        live = live[:k]
        assert not unmarked_full_slabs()[1]
        for sz in sizes:
            r = run("priv-throughput", 4000, 128, sz, ntries=3, memory=40 << 20)
            assert r["mallocs"] == r["frees"]
            assert not unmarked_full_slabs()[1]
    assert seen > 0 and live.size == 0
    assert H.Halloc.free_bytes() == H.Halloc.geometry()["arena_bytes"]


@pytest.mark.parametrize("length", [1, 15, 16, 17, 33, 64])
@pytest.mark.parametrize("nreq", [1, 3, 64, 256, 700])
def test_pages_drained_together(heap, nreq, length):
    # equal lengths that arrive together: up to 64 lanes of a wave drain in the
    # same step (the shared check takes four pages at a time), last pages part
    # filled; in the mixed run lengths vary by lane
    from halloc_amd.workloads import pages_for
    from tests.helpers import serve_checksums
    print(f"[gpu] drain nreq={nreq} length={length}", flush=True)
    heap(H.HallocOpts(memory=64 << 20, sb_sz_sh=21, nheads=8))
    rng = np.random.default_rng(nreq * 100 + length)
    tag = rng.integers(0, 1 << 32, nreq, dtype=np.uint64).astype(np.uint32)
    for ln in (np.full(nreq, length, np.uint32), rng.integers(1, length + 1, nreq).astype(np.uint32)):
        r = H.Halloc.run_serve(np.zeros(nreq, np.uint64), ln, tag, slots=256, watermark=0)
        assert r["completed"] == nreq and r["nulls"] == 0 and not r["bad"].any()
        assert (r["produced"] == ln).all() and (r["checksum"] == serve_checksums(tag, ln)).all()
        assert r["pages"] == int(pages_for(ln).sum())


@pytest.mark.parametrize("lanes", [1, 3, 4, 5, 7, 8, 9, 12, 16, 33, 63, 64])
def test_damaged_pages_are_charged_to_their_lanes(heap, lanes):
    # the wave's check and each lane's own, on pages with damaged tokens: up to
    # and above the number of lanes from which each checks its own page, passes
    # of four pages with one to four owners, part-filled pages (what follows
    # their tokens is never looked at), lanes that already found damage
    from tests.helpers import _hash3
    print(f"[gpu] damaged pages lanes={lanes}", flush=True)
    rng = np.random.default_rng(lanes)
    some = 0
    for rate in (0.0, 0.05, 0.5, 1.0):
        tag = rng.integers(0, 1 << 32, 64, dtype=np.uint64).astype(np.uint32)
        page = rng.integers(0, 2048, 64).astype(np.uint32)
        n = np.where(rng.random(64) < 0.5, 16, rng.integers(1, 17, 64)).astype(np.int64)
        drains = np.zeros(64, np.uint32)
        drains[rng.permutation(64)[:lanes]] = 1
        t = page[:, None] * np.uint32(16) + np.arange(16, dtype=np.uint32)
        h = _hash3(np.repeat(tag, 16), t.ravel(), np.uint32(0x5E7A11C3)).reshape(64, 16)
        pages = np.stack([np.repeat(tag[:, None], 16, 1), t, h, ~h], axis=-1)
        used = np.arange(16) < n[:, None]
        hurt = (rng.random((64, 16)) < rate) & used
        l, j = np.nonzero(hurt)
        pages[l, j, rng.integers(0, 4, l.size)] ^= np.uint32(1) << rng.integers(0, 32, l.size).astype(np.uint32)
        pages[~used] = rng.integers(0, 1 << 32, (int((~used).sum()), 4), dtype=np.uint64).astype(np.uint32)
        cs0 = rng.integers(0, 1 << 32, 64, dtype=np.uint64).astype(np.uint32)
        nb0 = rng.choice([0, 0, 3], 64).astype(np.uint32)
        bf0 = rng.integers(0, 1 << 62, 64, dtype=np.uint64)
        cs, nb, bf = H.Halloc.check_pages(pages, tag, page, page * 16 + n, drains, cs0, nb0, bf0)
        for i in range(64):
            bad = np.nonzero(hurt[i])[0] if drains[i] else np.zeros(0, int)
            good = h[i][used[i] & ~hurt[i]] if drains[i] else h[i][:0]
            assert cs[i] == (int(cs0[i]) + int(good.astype(np.uint64).sum())) & 0xFFFFFFFF
            assert nb[i] == nb0[i] + bad.size
            first = bf0[i]
            if bad.size and not nb0[i]:
                first = int(pages[i, bad[0], 0]) | int(pages[i, bad[0], 1]) << 32
            assert bf[i] == first
            some += bad.size
    assert some > 0
    with pytest.raises(H.HallocError):
        H.Halloc.check_pages(pages, tag, page, page * 16, np.ones(64), cs0, nb0, bf0)


@pytest.mark.parametrize("nthreads", [1, 4])
def test_buffers_kept_between_calls(heap, nthreads):
    # calls of changing sizes, from several threads, with a refused call between:
    # every call sees its own values, also after a shutdown and a new heap
    import threading

    print(f"[gpu] kept buffers threads={nthreads}", flush=True)
    opts = H.HallocOpts(memory=256 << 20, sb_sz_sh=21, nheads=8)
    wrong = []

    def calls(t):
        try:
            rng = np.random.default_rng(t)
            for n in (1, 1000, 70, 30000, 1, 4097, 30000, 200):
                sizes = rng.integers(1, 257, (3, n)).astype(np.uint32)
                order = rng.permutation(3 * n).astype(np.uint32)
                r = H.Halloc.run_lists(sizes, order, bs=64)
                assert r["requests"] == 3 * n and r["nulls"] == 0 and r["errors"] == 0
                with pytest.raises(H.HallocError):
                    H.Halloc.run_lists(sizes, np.zeros(3 * n, np.uint32), bs=64)
                p = H.Halloc.malloc_sizes(sizes[0])
                assert (p != 0).all() and len(np.unique(p)) == n
                H.Halloc.free_ptrs(p)
        except BaseException as e:  # reported below: a thread's own failure would be lost
            wrong.append(repr(e))

    for _ in range(2):
        heap(opts)
        ths = [threading.Thread(target=calls, args=(t,)) for t in range(nthreads)]
        for th in ths:
            th.start()
        for th in ths:
            th.join()
        assert not wrong
        assert H.Halloc.free_bytes() == H.Halloc.geometry()["arena_bytes"]
        H.Halloc.shutdown()


def test_long_lists_from_several_threads(heap):
    # lists that the device checks, in buffers that calls of other lengths and
    # threads gave back: good orders are taken, others refused
    import threading

    print("[gpu] long lists from several threads", flush=True)
    heap(H.HallocOpts(memory=1 << 30, sb_sz_sh=22))
    wrong = []

    def calls(t):
        try:
            rng = np.random.default_rng(t)
            for n in (1 << 17, 70, 150001, 1 << 17, 200003):
                sizes = (rng.integers(0, 3, (1, n)) * 16).astype(np.uint32)
                order = rng.permutation(n).astype(np.uint32)
                for _ in range(2):
                    r = H.Halloc.run_lists(sizes, order)
                    assert r["requests"] == np.count_nonzero(sizes) and r["nulls"] == 0 and r["errors"] == 0
                    bad = order.copy()
                    bad[rng.integers(0, n)] = rng.choice([n, order[0], order[n - 1]])
                    if (np.sort(bad) != np.arange(n)).any():
                        with pytest.raises(H.HallocError, match="permutation"):
                            H.Halloc.run_lists(sizes, bad)
        except BaseException as e:  # reported below: a thread's own failure would be lost
            wrong.append(repr(e))

    ths = [threading.Thread(target=calls, args=(t,)) for t in range(4)]
    for th in ths:
        th.start()
    for th in ths:
        th.join()
    assert not wrong
    assert H.Halloc.free_bytes() == H.Halloc.geometry()["arena_bytes"]


@pytest.mark.parametrize("n,per", [(1, 1), ((1 << 17) - 1, 1), (1 << 16, 2), (43691, 3), (1 << 17, 1), (100003, 7)])
def test_list_orders_checked(heap, n, per):
    # below, at and above the length from which the device checks the order and
    # counts the requests: permutations are taken, anything else is refused
    # before a block is allocated
    print(f"[gpu] list order n={n} per={per}", flush=True)
    heap(H.HallocOpts(memory=256 << 20, sb_sz_sh=22))
    total = n * per
    rng = np.random.default_rng(total)
    sizes = (rng.integers(0, 3, (per, n)) * 16).astype(np.uint32)
    good = rng.permutation(total).astype(np.uint32)
    for order in (None, good, np.arange(total, dtype=np.uint32), np.arange(total, dtype=np.uint32)[::-1]):
        r = H.Halloc.run_lists(sizes, order)
        assert r["requests"] == np.count_nonzero(sizes) and r["nulls"] == 0 and r["errors"] == 0
    arena = H.Halloc.geometry()["arena_bytes"]
    for k in (0, total // 2, total - 1):
        for v in (total, 0xFFFFFFFF, int(good[k - 1]) if total > 1 else total + 1):
            bad = good.copy()
            bad[k] = v
            with pytest.raises(H.HallocError, match="permutation"):
                H.Halloc.run_lists(sizes, bad)
    assert H.Halloc.free_bytes() == arena
