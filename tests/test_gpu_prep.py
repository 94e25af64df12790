"""GPU parity of the generator, preprocessing and core-matrix kernels at the sizes where they change path."""
import os
import subprocess
import sys

import numpy as np
import pytest

import tribit_amd
from tests.test_gpu_parity import assert_same_structure

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[case] {msg}", flush=True)


@pytest.mark.parametrize("scale", [1, 2, 7, 12, 15])
def test_rmat_generator_scales(gpu_ctx, oracle_mod, scale):
    """Even and odd scales (the last word of an odd scale gives one level): keys equal the oracle's."""
    note(f"rmat keys s{scale}")
    assert np.array_equal(gpu_ctx.gen_rmat_keys(scale, 5, seed=9), oracle_mod.gen_rmat(scale, 5, seed=9))


@pytest.mark.parametrize("core", [65536, 65537, 66001])
def test_core_wider_than_one_window(gpu_ctx, oracle_mod, core):
    """Core rows of one LDS column window, and of two."""
    note(f"core of {core} ids, er 70001")
    keys = oracle_mod.gen_er(70001, 900000, seed=4)
    with gpu_ctx.graph_from_keys(keys, 70001) as g:
        r = g.count("wedge", dense_core=core)
        assert r.dense_core == core
        assert r.triangles == oracle_mod.count_keys(keys, 70001)


@pytest.mark.parametrize("graphs", [1, 8192, 8193])
def test_batch_edge_counts(gpu_ctx, oracle_mod, graphs):
    """Per-graph edge counts at and past the largest batch summed in LDS."""
    note(f"batch of {graphs} small graphs")
    rng = np.random.default_rng(graphs)
    ns = rng.integers(2, 7, graphs)
    keys = []
    for n in ns:
        a, b = rng.integers(0, n, (2, int(rng.integers(0, 9))))
        keys.append(((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64))
    with gpu_ctx.batch_from_keys(keys, ns) as b:
        n, m = b.sizes()
        assert np.array_equal(n, ns.astype(np.uint64))
        assert [int(x) for x in m] == [len(set(k.tolist())) for k in keys]
        c, _ = b.count()
        assert [int(x) for x in c] == [oracle_mod.count_keys(k, int(v)) for k, v in zip(keys, ns)]


# (vertices, keys): one bucket, the first two buckets, the widest single pass, the first two-pass partition with
# 64-bit items, 32-bit items and items of exactly 32 bits
@pytest.mark.parametrize("n,nk", [(5, 1), (5000, 2048), (5000, 2049), (70000, 1 << 20), (1 << 26, (1 << 20) + 1),
                                  (100000, (1 << 20) + 1), (1 << 21, 1500001)])
def test_distinct_keys_partition(gpu_ctx, oracle_mod, n, nk):
    """Sentinels and repeated keys among the input; every structure equals the oracle's."""
    note(f"partition of {nk} keys over {n} ids")
    rng = np.random.default_rng(nk)
    a, b = rng.integers(0, n, (2, nk))
    k = ((np.minimum(a, b) << 32) | np.maximum(a, b)).astype(np.uint64)
    k[a == b] = oracle_mod.SENTINEL
    k[rng.integers(0, nk, nk // 5)] = k[rng.integers(0, nk, nk // 5)]
    with gpu_ctx.graph_from_keys(k, n) as g:
        assert_same_structure(g, k, n, oracle_mod)


def test_distinct_keys_repeated(gpu_ctx, oracle_mod):
    """Keys repeated thousands of times overflow their bucket: the sort takes over."""
    note("500 keys, 2M times")
    rng = np.random.default_rng(5)
    keys = oracle_mod.gen_er(3000, 500, seed=2)
    k = keys[rng.integers(0, keys.size, 2_000_000)]
    with gpu_ctx.graph_from_keys(k, 3000) as g:
        assert_same_structure(g, k, 3000, oracle_mod)


@pytest.mark.parametrize("n,nk", [(65536, 300000), (65537, 300000), (3 * 65536 + 32769, 3000000),
                                  ((1 << 27) + 70001, 300000)])
def test_degrees_by_id_range(gpu_ctx, n, nk):
    """Degrees around the ends of an id group and half group, of one group's counting tasks (a hub group), and past
    the ids of one pass."""
    note(f"degrees over {n} ids")
    rng = np.random.default_rng(n)
    a = rng.integers(0, n, nk)
    b = np.where(rng.random(nk) < 0.7, rng.integers(0, min(n, 30000), nk), n - 1 - rng.integers(0, 7, nk))
    k = np.unique(((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64))
    want = np.bincount((k >> np.uint64(32)).astype(np.int64), minlength=n)
    want += np.bincount((k & np.uint64(0xFFFFFFFF)).astype(np.int64), minlength=n)
    with gpu_ctx.graph_from_keys(k, n) as g:
        labels, _ = g.labels()
        assert np.array_equal(g.download()[2], want[labels].astype(np.uint32))


def hub_graph(rng, n, hubs, leaves, extra):
    """`hubs` top vertices joined to `leaves` random others each and to each other, plus `extra` random edges."""
    a = [np.repeat(np.arange(hubs), leaves), rng.integers(0, n, extra), np.repeat(np.arange(hubs), hubs)]
    b = [rng.integers(hubs, n, hubs * leaves), rng.integers(0, n, extra), np.tile(np.arange(hubs), hubs)]
    a, b = np.concatenate(a), np.concatenate(b)
    return np.unique(((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64))


# a wave or less, hubs that own most ranges, hubs whose own ranges are the longest (two 64K-id windows among them)
@pytest.mark.parametrize("n,hubs,leaves,extra", [(60, 1, 20, 100), (9000, 0, 0, 8192), (9000, 2, 4095, 30000),
                                                 (30000, 3, 4097, 60000), (200000, 1, 150000, 20000),
                                                 (100000, 4, 20000, 2000000), (100000, 40, 30000, 1000000),
                                                 (400000, 3, 300000, 3500000)])
def test_wedge_records(gpu_ctx, oracle_mod, n, hubs, leaves, extra):
    """Wedge ranges grouped by head: counts over them with and without a core (whose cut relies on their order) and
    from 16- and 32-bit ids (whose narrow records travel through the sort)."""
    note(f"wedges: {n} ids, {hubs} hubs of {leaves}, {extra} others")
    k = hub_graph(np.random.default_rng(n + hubs), n, hubs, leaves, extra)
    want = oracle_mod.count_keys(k, n)
    with gpu_ctx.graph_from_keys(k, n) as g:
        assert_same_structure(g, k, n, oracle_mod)
        for core in (0, 64, min(n, 5000)):
            assert g.count("wedge", dense_core=core).triangles == want, core
        assert g.count("wedge", flags=tribit_amd.WIDE_IDS).triangles == want
        assert sum(g.variant_stats("wedge")["edges"]) <= k.size


# m edges around the smallest graph whose rows are partitioned and around the second pass (2 m = 512 quanta of rows),
# and a clique: full slots (rows below 4096 arcs) and rows longer than a slot
@pytest.mark.parametrize("n,m,clique", [(300, 8192, 0), (300, 8193, 0), (70000, 8193, 0), (5000, (1 << 20) - 1, 0),
                                        (3000000, 1 << 20, 0), (200000, 1 << 21, 0), (9000, 20000, 1500),
                                        (20000, 30000, 4000), (5000, 50000, 4096), (30000, 30000, 4300)])
@pytest.mark.parametrize("relabel", [1, 2])
def test_rows_by_partition(gpu_ctx, relabel, n, m, clique):
    """The arcs of both relabelled id orders, each row's ids ascending, as a sort of the relabelled edges gives them."""
    note(f"rows: {n} ids, {m} edges, clique of {clique}, id order {relabel}")
    rng = np.random.default_rng(n + m + clique)
    k = np.zeros(0, np.uint64)
    while k.size < m:
        a, b = rng.integers(0, n, (2, m))
        x = ((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64)
        k = np.unique(np.concatenate([k, x]))
    k = rng.permutation(k)[:m]
    ids = rng.choice(n, clique, replace=False)
    i, j = np.triu_indices(clique, 1)
    k = np.unique(np.concatenate([k, ((np.minimum(ids[i], ids[j]) << 32) | np.maximum(ids[i], ids[j])).astype(np.uint64)]))
    gpu_ctx.set_relabel(relabel)
    try:
        with gpu_ctx.graph_from_keys(k, n) as g:
            order, _ = g.labels()
            row_ptr, col, deg = g.download()
    finally:
        gpu_ctx.set_relabel("auto")
    new = np.empty(n, np.int64)
    new[order] = np.arange(n)
    a, b = new[(k >> np.uint64(32)).astype(np.int64)], new[(k & np.uint64(0xFFFFFFFF)).astype(np.int64)]
    arcs = np.sort((np.minimum(a, b) << 32) | np.maximum(a, b))
    assert np.array_equal(row_ptr, np.searchsorted(arcs, np.arange(n + 1) << 32).astype(np.uint32))
    assert np.array_equal(col, (arcs & 0xFFFFFFFF).astype(np.uint32))
    assert np.array_equal(deg, np.bincount(np.concatenate([a, b]), minlength=n).astype(np.uint32))


# ids and arcs where their sorts change method: 2^16 items (keys of 16 bits), 2^18 (more bits), past 2^20
@pytest.mark.parametrize("n,m", [(30000, 65535), (30000, 65536), (1 << 16, 65536), (1 << 16, 262143),
                                 (262143, 262144), (262144, 262143), (70000, 1 << 20), (1 << 20, 300000),
                                 ((1 << 20) + 1, (1 << 20) + 1)])
def test_sort_sizes(gpu_ctx, oracle_mod, n, m):
    """Graphs of exactly m edges: structure, and the wedge ranges through a count, against the oracle."""
    note(f"sorts: {n} ids, {m} edges")
    rng = np.random.default_rng(n + m)
    k = np.zeros(0, np.uint64)
    while k.size < m:
        a, b = (rng.random((2, m)) ** 2 * n).astype(np.int64)
        x = ((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64)
        k = np.unique(np.concatenate([k, x]))
    k = np.sort(rng.permutation(k)[:m])
    with gpu_ctx.graph_from_keys(k, n) as g:
        assert_same_structure(g, k, n, oracle_mod)
        assert g.count("wedge").triangles == oracle_mod.count_keys(k, n)


# totals of small scans (2^15 ids), of the counts in LDS (2^15 ids, 2^18 edges) and of one schedule scan (2^19 ids)
@pytest.mark.parametrize("n,nk", [(32768, 100000), (32769, 100000), (32768, 262144), (32768, 270000), (8192, 60000),
                                  (524288, 600000), (524289, 600000), (600001, 400000)])
def test_scan_and_count_sizes(gpu_ctx, oracle_mod, n, nk):
    """Ids around the ends of the one-launch scans and of the degree count in LDS, counted under every schedule."""
    note(f"scans: {n} ids, {nk} keys")
    k = oracle_mod.gen_er(n, nk, seed=n % 97)
    want = oracle_mod.count_keys(k, n)
    with gpu_ctx.graph_from_keys(k, n) as g:
        assert_same_structure(g, k, n, oracle_mod)
        for sched in ("plain", "learned", "wedge"):
            assert g.count(sched).triangles == want, sched


# arcs around a wave's share (256) and its steps (64), and hubs whose ranges fill several waves
@pytest.mark.parametrize("n,hubs,leaves,extra", [(300, 0, 0, 30), (40, 0, 0, 62), (4000, 0, 0, 256), (4000, 0, 0, 257),
                                                 (60, 0, 0, 700), (3000, 3, 900, 100), (3000, 40, 2000, 9000),
                                                 (50000, 1, 40000, 300000)])
def test_wedge_work(gpu_ctx, n, hubs, leaves, extra):
    """The elements that the wedge ranges of all owners stream, summed per head while the records are unpacked."""
    note(f"wedge work: {n} ids, {hubs} hubs of {leaves}, {extra} others")
    k = hub_graph(np.random.default_rng(n + extra), n, hubs, leaves, extra)
    with gpu_ctx.graph_from_keys(k, n) as g:
        row_ptr, col, _ = g.download()
        got = sum(g.variant_stats("wedge")["wplus"])
    row_ptr = row_ptr.astype(np.int64)
    d = np.diff(row_ptr)
    after = np.repeat(row_ptr[1:], d) - np.arange(col.size) - 1
    assert got == int(after[d[col] > 0].sum())


# longest rows of exactly the arcs that one sort takes (4608) and one more, of a row with gaps among its ids (a random
# graph of average degree 6300: rows to about 6300 arcs), and of many slots
@pytest.mark.parametrize("n,m,clique,p", [(5200, 9000, 4609, 1.0), (5200, 9000, 4610, 1.0), (40000, 30000, 6000, 1.0),
                                          (9000, 0, 9000, 0.7)])
@pytest.mark.parametrize("relabel", [1, 2])
def test_rows_longer_than_a_sort(gpu_ctx, relabel, n, m, clique, p):
    """Rows past the largest sort of a slot, listed through a bitmap: the arcs as a sort of the relabelled edges gives
    them, row by row."""
    note(f"long rows: {n} ids, {m} edges, {clique} ids joined with {p}, id order {relabel}")
    rng = np.random.default_rng(n + m + clique)
    a, b = rng.integers(0, n, (2, m))
    ids = rng.choice(n, clique, replace=False)
    i, j = np.triu_indices(clique, 1)
    if p < 1:
        keep = rng.random(i.size) < p
        i, j = i[keep], j[keep]
    a, b = np.concatenate([a, ids[i]]), np.concatenate([b, ids[j]])
    k = np.unique(((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64))
    gpu_ctx.set_relabel(relabel)
    try:
        with gpu_ctx.graph_from_keys(rng.permutation(k), n) as g:
            order, _ = g.labels()
            row_ptr, col, deg = g.download()
    finally:
        gpu_ctx.set_relabel("auto")
    new = np.empty(n, np.int64)
    new[order] = np.arange(n)
    a, b = new[(k >> np.uint64(32)).astype(np.int64)], new[(k & np.uint64(0xFFFFFFFF)).astype(np.int64)]
    arcs = np.sort((np.minimum(a, b) << 32) | np.maximum(a, b))
    assert np.diff(row_ptr.astype(np.int64)).max() >= (4608 if clique == 4609 else 4609)
    assert np.array_equal(row_ptr, np.searchsorted(arcs, np.arange(n + 1) << 32).astype(np.uint32))
    assert np.array_equal(col, (arcs & 0xFFFFFFFF).astype(np.uint32))
    assert np.array_equal(deg, np.bincount(np.concatenate([a, b]), minlength=n).astype(np.uint32))


# one partition pass, the first of two, ids without edges, keys mostly repeated, and one of a workgroup's sorts
# (KiB: the least cap under which a build by sorts alone ran, by bisection; it differs by id order with the most ids)
@pytest.mark.parametrize("n,nk,kib", [(50000, 300000, (13967, 13967)), (1 << 18, (1 << 20) + 1, (51205, 51205)),
                                      (1 << 16, 2500000, (106986, 106986)), (1 << 20, 50000, (30775, 33164)),
                                      (1500, 3000000, (94168, 94168)), (900, 7000, (317, 317))])
@pytest.mark.parametrize("relabel", [1, 2])
def test_build_in_the_memory_of_the_sorts(gpu_ctx, oracle_mod, relabel, n, nk, kib):
    """A build under an allocation cap that holds what sorts need: each partition and the packed records give way to
    a sort, with the same graph and counts."""
    note(f"capped build: {nk} keys over {n} ids, id order {relabel}")
    rng = np.random.default_rng(n)
    a, b = (rng.random((2, nk)) ** 1.5 * n).astype(np.int64)
    k = ((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64)
    cap = kib[relabel - 1] << 10
    with tribit_amd.Context(0) as ctx:
        ctx.set_relabel(relabel)
        ctx.set_alloc_cap(cap)
        with ctx.graph_from_keys(k, n) as g:
            ctx.set_alloc_cap(0)
            assert ctx.pool_peak() <= cap
            row_ptr, col, deg = g.download()
            order, _ = g.labels()
            got = g.count("wedge").triangles
            work = sum(g.variant_stats("wedge")["wplus"])
        ctx.set_alloc_cap(0)
        with ctx.graph_from_keys(k, n) as g:  # with room for the partitions
            for x, y in zip((row_ptr, col, deg), g.download()):
                assert np.array_equal(x, y)
            assert np.array_equal(order, g.labels()[0])
            assert got == g.count("wedge").triangles == oracle_mod.count_keys(k, n)
            assert work == sum(g.variant_stats("wedge")["wplus"])


# edges around a block's share (2048) and the most of this way, over ids that just pass LDS and many; stars and few hubs
@pytest.mark.parametrize("n,m,hubs", [(32769, 1, 0), (40000, 2048, 0), (40000, 2049, 3), (300000, 1 << 18, 0),
                                      (300000, 1 << 18, 1), (300000, 1 << 18, 8), (1 << 24, 262143, 1)])
def test_degrees_of_few_edges(gpu_ctx, n, m, hubs):
    note(f"degrees: {m} edges over {n} ids, {hubs} hubs")
    rng = np.random.default_rng(n + m + hubs)
    k = np.zeros(0, np.uint64)
    while k.size < m:
        a = rng.integers(0, n, 2 * m) if hubs == 0 else n - 1 - rng.integers(0, hubs, 2 * m)
        b = rng.integers(0, n, 2 * m)
        x = ((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64)
        k = np.unique(np.concatenate([k, x]))
    k = rng.permutation(k)[:m]
    want = np.bincount((k >> np.uint64(32)).astype(np.int64), minlength=n)
    want += np.bincount((k & np.uint64(0xFFFFFFFF)).astype(np.int64), minlength=n)
    with gpu_ctx.graph_from_keys(k, n) as g:
        labels, _ = g.labels()
        assert np.array_equal(g.download()[2], want[labels].astype(np.uint32))


def test_star_builds_like_other_graphs(gpu_ctx):
    """Device time of a star of 2^18 edges against a random graph's: a queue of atomics on its hub made it ten times."""
    note("star and random graph of 2^18 edges")
    n, m = 300000, 1 << 18
    rng = np.random.default_rng(1)
    leaf = np.arange(1, m + 1, dtype=np.uint64)
    a, b = rng.integers(0, n, (2, m))
    other = ((np.minimum(a, b) << 32) | np.maximum(a, b))[a != b].astype(np.uint64)

    def ms(keys):
        t = []
        for _ in range(6):
            with gpu_ctx.graph_from_keys(keys, n) as g:
                t.append(g.info()["ms_preprocess"])
        return min(t)

    assert ms(leaf) < 4 * ms(other)


def test_degrees_of_more_than_2_31_edges(gpu_ctx):
    """Two spans of keys: W+ (which every degree enters) and the triangles are those that a build by sorts gave."""
    note("er of 2.3G keys over 2^24 ids")
    with gpu_ctx.gen_er(1 << 24, 2300000000, seed=1) as g:
        i = g.info()
        assert (i["m"], i["wplus"]) == (2299981280, 210131079941)
        assert g.count("wedge").triangles == 3433745


def test_records_that_need_the_largest_outdegree(gpu_ctx):
    """More than 2^28 edges over 2^26 ids: an arc's packed record fits only with the real largest outdegree, read back
    first. The wedge ranges unpacked from it against the direction-split ranges, which do not use them."""
    note("er of 272M keys over 2^26 ids")
    with gpu_ctx.gen_er(1 << 26, 272_000_000, seed=3) as g:
        assert g.info()["m"] > 1 << 28
        assert g.count("wedge").triangles == g.count("directed").triangles > 0


def test_memory_kept_by_another_context(gpu_ctx):
    """137 GB freed and kept by one context leave room for 206 GB in another."""
    note("device keys of 137 and 206 GB")
    import ctypes

    def keys(ctx, ef):
        d, n = ctypes.c_void_p(), ctypes.c_uint64()
        assert ctx.lib.tribit_gen_rmat(ctx.h, 31, ef, 0.57, 0.19, 0.19, 1, ctypes.byref(d), ctypes.byref(n)) == 0
        ctx.lib.tribit_free_device_keys(ctx.h, d)

    with tribit_amd.Context(0) as a, tribit_amd.Context(0) as b:
        keys(a, 8)
        keys(b, 12)


# edges for a sort by one workgroup and for a partition of the rows, and few and many of them for the degrees
@pytest.mark.parametrize("relabel,m,clique", [(0, 20000, 200), (1, 2000, 40), (1, 300000, 200), (2, 20000, 200)])
def test_more_than_2_31_ids(gpu_ctx, oracle_mod, relabel, m, clique):
    """Ids past 2^31, whose cleared spans have more words than a launch may have threads: counts equal those of the
    same edges over their own ids."""
    n = (1 << 31) + 1000
    note(f"{m} edges over {n} ids, id order {relabel}")
    rng = np.random.default_rng(m)
    ids = np.unique(np.concatenate([rng.integers(0, n, clique), n - 1 - rng.integers(0, 1000, 60)]))
    i, j = np.triu_indices(ids.size, 1)
    a, b = np.concatenate([ids[i], rng.integers(0, n, m)]), np.concatenate([ids[j], rng.integers(0, n, m)])
    small = np.unique(np.concatenate([a, b]), return_inverse=True)[1]
    x, y = small[:a.size], small[a.size:]
    pack = lambda u, v: ((np.minimum(u, v) << 32) | np.maximum(u, v))[u != v].astype(np.uint64)  # noqa: E731
    want = oracle_mod.count_keys(pack(x, y), int(small.max()) + 1)
    assert want >= ids.size * (ids.size - 1) * (ids.size - 2) // 6
    gpu_ctx.set_relabel(relabel)
    try:
        with gpu_ctx.graph_from_keys(pack(a, b), n) as g:
            scheds = ("plain", "directed") if relabel == 0 else ("wedge", "directed")
            assert [g.count(s).triangles for s in scheds] == [want, want]
    finally:
        gpu_ctx.set_relabel("auto")


def test_degrees_of_one_full_id_group(gpu_ctx):
    """The complete graph on 65,535 ids, whose 4,294,770,690 endpoints are one group's: W+, which every degree enters,
    is its number of triangles."""
    n = 65535
    note("complete graph on 65535 ids")
    with gpu_ctx.gen_sbm(1, n, 1.0, 0.0, 1) as g:
        i = g.info()
        assert (i["m"], i["max_outdeg"]) == (n * (n - 1) // 2, n - 1)
        assert i["wplus"] == n * (n - 1) * (n - 2) // 6


def test_keys_that_the_caller_allocated(gpu_ctx, oracle_mod):
    """tribit_graph_from_device_keys frees the keys: those of the runtime's allocator too, and another context's."""
    import ctypes

    note("caller's device keys")
    hip = ctypes.CDLL("libamdhip64.so")
    keys = oracle_mod.gen_rmat(12, 8, seed=4)
    want = oracle_mod.count_keys(keys, 1 << 12)

    def build(d):
        g = ctypes.c_void_p()
        assert gpu_ctx.lib.tribit_graph_from_device_keys(gpu_ctx.h, d, keys.size, 1 << 12, ctypes.byref(g)) == 0
        with tribit_amd.Graph(gpu_ctx, g.value) as graph:
            assert graph.count("wedge").triangles == want

    def free_bytes():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    left = []
    for _ in range(3):  # the first pass takes the pool's own memory
        d = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(d), ctypes.c_size_t(4 << 30)) == 0
        assert hip.hipMemcpy(d, keys.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(8 * keys.size), 1) == 0
        build(d)
        left.append(free_bytes())
    assert left[2] > left[0] - (1 << 30)

    with tribit_amd.Context(0) as other:
        d, n = ctypes.c_void_p(), ctypes.c_uint64()
        assert other.lib.tribit_gen_rmat(other.h, 12, 8, 0.57, 0.19, 0.19, 4, ctypes.byref(d), ctypes.byref(n)) == 0
        assert n.value == keys.size and hip.hipDeviceSynchronize() == 0
        build(d)
        again = ctypes.c_void_p()
        assert other.lib.tribit_gen_rmat(other.h, 12, 8, 0.57, 0.19, 0.19, 4, ctypes.byref(again), ctypes.byref(n)) == 0
        assert again.value == d.value  # the block was free again
        other.lib.tribit_free_device_keys(other.h, again)


def test_preprocessing_time_without_code_loading():
    """A process's first graph reports the time of its preprocessing, not of the sorts' code being loaded (5 ms a file)."""
    note("times of a process's first graph")
    code = ("import tribit_amd as tb\n"
            "ctx = tb.Context(0)\n"
            "for seed in (1, 2):\n"
            "    with ctx.gen_rmat(16, 16, seed=seed) as g:\n"
            "        g.count('directed')\n"
            "        i = g.info()\n"
            "        print(i['ms_preprocess'], i['ms_layout'][2], flush=True)\n")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100,
                         cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert out.returncode == 0, out.stderr
    first, second = (np.array(line.split(), float) for line in out.stdout.splitlines())
    assert (first < second + 4.0).all(), (first, second)
