"""BFS and components along the edge array in two launches, what is resident first: numbers of entries at the edges of rows,
segments and of a wave's share, lists that cross pages, vertices without lists, and levels found ahead of their sweep."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import SEED, Rig, _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu

KINDS = [{"by_page": True}, {"coarse": 64}, {"frontier": True}]


def _rig(bam, nb, page, cache_pages):
    pad = (-len(nb)) % (page // 8)
    r = Rig(bam, (len(nb) + pad) * 8, backing=True, n_queues=16, depth=256, stage_bytes=max(4096, min(page, 8192)))
    r.backing(len(nb) + pad)[:len(nb)] = nb
    return r, r.array(len(nb), page, cache_pages)


def _check_bfs(r, a, off, nb, sources):
    d_off = _dev(off)
    for kept in (False, True):
        if kept:
            a.set_graph(d_off)
        for src in sources:
            want, want_it = oracle.bfs_levels(off, nb, int(src))
            for kw in KINDS:
                lv, it = a.bfs(d_off, int(src), **kw)
                assert np.array_equal(lv.cpu().numpy().view(np.uint32), want) and it == want_it, (kept, src, kw, it, want_it)
    assert not r.c.aborted()


# a directed graph with lists of 0 to `most` entries: one below, at and one above a row, a segment, two, sixteen of them
@pytest.mark.parametrize("n_edges", [1, 63, 64, 65, 511, 512, 513, 1025, 8191, 8192, 8193, 33333])
@pytest.mark.parametrize("page,cache_pages", [(4096, 2), (4096, 9), (4096, 1024), (512, 40), (8192, 5), (16384, 3), (65536, 2)])
def test_levels_of_directed_graphs_of_all_lengths(bam, n_edges, page, cache_pages):
    rng = np.random.default_rng(n_edges + page + cache_pages)
    most = 1500 if n_edges > 9000 else 40
    deg = []
    while sum(deg) < n_edges:
        deg.append(0 if rng.random() < 0.3 else int(rng.integers(1, most)))
    deg = np.array([0, 0] + deg + [0])                     # the first vertices and the last have no list
    deg[np.nonzero(deg)[0][-1]] -= deg.sum() - n_edges
    n_v = len(deg)
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    # mostly to vertices nearby, so that there are several levels
    owner = np.repeat(np.arange(n_v), deg)
    nb = ((owner + rng.integers(-3, 8, n_edges)) % n_v).astype(np.uint64)
    r, a = _rig(bam, nb, page, cache_pages)
    with r:
        _check_bfs(r, a, off, nb, [0, int(np.nonzero(deg)[0][0]), int(rng.integers(0, n_v))])


@pytest.mark.parametrize("page,cache_pages", [(4096, 30), (4096, 500), (8192, 30), (65536, 4)])
def test_labels_and_levels_of_a_random_graph(bam, page, cache_pages):
    for off, nb in (oracle.rmat_csr(SEED, 13), oracle.uniform_csr(SEED, 30011, 50021)):
        r, a = _rig(bam, nb, page, cache_pages)
        with r:
            _check_bfs(r, a, off, nb, oracle.bfs_sources(SEED, off, 2))
            want, _ = oracle.cc_labels(off, nb)
            for kept in (True, True, False):
                if not kept:
                    a.set_graph(None)
                for by_page in (False, True):
                    lb, _ = a.cc(_dev(off), by_page=by_page)
                    assert np.array_equal(_u64(lb), want), (kept, by_page)
            assert not r.c.aborted()


def _two_halves(n_v, n_e):
    """two random graphs side by side, no edge between them"""
    (oa, na), (ob, nb) = oracle.uniform_csr(SEED, n_v, n_e), oracle.uniform_csr(SEED + 1, n_v, n_e)
    return np.concatenate([oa, ob[1:] + oa[-1]]), np.concatenate([na, nb + np.uint64(n_v)])


# around a row, a segment and a page of 4 KiB, and several of them; the largest graph is one that bam_cc_by_page reads in this way though all of it is cached
@pytest.mark.parametrize("before,behind,filler,n_v,n_e,share", [
    (b, a, f, 9001, 40009, s) for b, a in ((0, 1), (0, 64), (0, 512), (0, 5000), (1, 0), (64, 0), (512, 0), (1500, 0), (700, 1300))
    for f in ("zeros", "vertices") for s in (1, 2)] + [(700, 1300, "vertices", 150001, 1100003, 1)])
def test_entries_that_are_in_no_list(bam, before, behind, filler, n_v, n_e, share):
    """an array longer than the lists of its graph: what lies before the first list and behind the last is nobody's neighbour"""
    off, nb = _two_halves(n_v, n_e)
    want, _ = oracle.cc_labels(off, nb)
    assert want[n_v] == n_v
    src = int(oracle.bfs_sources(SEED, off, 1)[0])
    levels, n_levels = oracle.bfs_levels(off, nb, src)
    rng = np.random.default_rng(before + behind)

    def fill(n):
        return np.zeros(n, dtype=np.uint64) if filler == "zeros" else rng.integers(0, 2 * n_v, n).astype(np.uint64)

    nb = np.concatenate([fill(before), nb, fill(behind)])
    off = off + np.uint64(before)
    if before and filler == "zeros":
        nb[:before] = n_v                      # (entries before the first list would be the first vertex's)
    r, a = _rig(bam, nb, 4096, (len(nb) + 511) // 512 // share + 1)
    with r:
        d_off = _dev(off)
        for kept in (False, True):
            if kept:
                a.set_graph(d_off)
            for by_page in (False, True):
                lb, _ = a.cc(d_off, by_page=by_page)
                assert np.array_equal(_u64(lb), want), (kept, by_page)
            for kw in KINDS:
                lv, it = a.bfs(d_off, src, **kw)
                assert np.array_equal(lv.cpu().numpy().view(np.uint32), levels) and it == n_levels, (kept, kw)
        assert not r.c.aborted()


@pytest.mark.parametrize("beyond", [1, 64, 700, 5000])
@pytest.mark.parametrize("share", [1, 2])
def test_lists_that_go_on_behind_the_number_of_elements(bam, beyond, share):
    """an array created with fewer elements than its range holds: the entries behind them are looked up in the range"""
    # a random graph, and behind it vertices with one entry each, of a vertex before them: nobody else's list names the last ones
    n_v, n_more = 9001, 9000
    off, nb = oracle.uniform_csr(SEED, n_v, 40009)
    off = np.concatenate([off, off[-1] + np.arange(1, n_more + 1, dtype=np.uint64)])
    nb = np.concatenate([nb, (n_v - 1 + np.random.default_rng(beyond).integers(0, np.arange(1, n_more + 1))).astype(np.uint64)])
    src = n_v + n_more - 1
    want, want_it = oracle.bfs_levels(off, nb, src)
    labels, _ = oracle.cc_labels(off, nb)
    assert want_it > 2 and labels[src] != src
    pages = (len(nb) + 511) // 512
    r = Rig(bam, pages * 4096, backing=True, n_queues=16, depth=256, stage_bytes=4096)
    r.backing(len(nb))[:] = nb
    with r:
        cache = bam.PageCache(4096, pages // share + 1, 0, r.c)
        held = bam.Range(0, len(nb), 0, pages, 0, 4096, cache, 0)
        a = bam.Array(len(nb) - beyond, 0, [held], 0)
        r.objs.append((a, held, cache))
        d_off = _dev(off)
        for kept in (False, True):
            if kept:
                a.set_graph(d_off)
            for kw in KINDS[1:]:
                lv, it = a.bfs(d_off, src, **kw)
                assert np.array_equal(lv.cpu().numpy().view(np.uint32), want) and it == want_it, (kept, kw)
            lb, _ = a.cc(d_off)
            assert np.array_equal(_u64(lb), labels), kept
        assert not r.c.aborted()


# 2 x 512 workgroups' turns of four pages of 512 entries, one turn fewer, an entry and a segment more: by turns and in stretches
@pytest.mark.parametrize("n_edges", [1023 * 2048, 1023 * 2048 + 1, 1023 * 2048 + 513, 1024 * 2048, 1024 * 2048 + 1, 1535 * 2048 + 511, 3071 * 2048, 3071 * 2048 + 1, 3071 * 2048 + 513, 3584 * 2048 - 1, 3584 * 2048 + 1, 3840 * 2048 - 1, 3840 * 2048 + 1])
def test_labels_where_each_workgroup_has_a_stretch(bam, n_edges):
    """paths of 1 to 5000 vertices one after the other, all edges cached"""
    rng = np.random.default_rng(n_edges)
    n_v = n_edges // 2 + 9000
    first = np.zeros(n_v, dtype=bool)
    first[np.cumsum(rng.integers(1, 5000, n_v // 500)) % n_v] = True
    first[0] = True
    linked = ~first[1:]                                        # v and v + 1
    linked[np.cumsum(linked) * 2 > n_edges] = False
    deg = np.zeros(n_v, dtype=np.int64)
    deg[:-1] += linked
    deg[1:] += linked
    v = np.arange(n_v, dtype=np.int64)
    nb = np.stack([v - 1, v + 1], axis=1).reshape(-1)[np.stack([np.concatenate([[False], linked]), np.concatenate([linked, [False]])], axis=1).reshape(-1)]
    labels = np.maximum.accumulate(np.where(np.concatenate([[True], ~linked]), v, 0)).astype(np.uint64)
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    assert n_edges - 5000 < len(nb) <= n_edges
    nb = np.concatenate([nb, np.zeros(n_edges - len(nb), dtype=np.int64)]).astype(np.uint64)
    r, a = _rig(bam, nb, 4096, (n_edges + 511) // 512)
    with r:
        d_off = _dev(off)
        a.set_graph(d_off)
        for by_page in (False, True, False):
            lb, _ = a.cc(d_off, by_page=by_page)
            assert np.array_equal(_u64(lb), labels), by_page
        assert not r.c.aborted()


# the number of vertices over how far a neighbour is at most: neighbours side by side just so, just not, and all over the graph
@pytest.mark.parametrize("part", [70, 24, 16, 2])
@pytest.mark.parametrize("before,behind", [(0, 0), (700, 5000)])
def test_labels_of_long_arrays_by_how_far_the_neighbours_are(bam, part, before, behind):
    """all edges cached and two turns of the workgroups or more, where a look at the neighbours says how the array is shared out; the
    rest of the array, which is in no list, holds numbers of vertices too"""
    from scipy.sparse import csr_matrix
    from scipy.sparse.csgraph import connected_components
    rng = np.random.default_rng(part)
    n_v, d = 910003, 7
    deg = np.where(rng.random(n_v) < 0.2, 0, rng.integers(6, 2 * d + 2, n_v))
    off = np.concatenate([[0], np.cumsum(deg)]) + before
    owner = np.repeat(np.arange(n_v), deg)
    far = n_v // part
    nb = rng.integers(0, n_v, len(owner) + before + behind)
    # of the last vertices within the thousandth that they are in, so that there are several components
    most = n_v // 4 * 3
    nb[before:before + len(owner)] = np.where(owner < most, (owner + rng.integers(-far, far + 1, len(owner))) % most,
                                              owner // 910 * 910 + rng.integers(0, 900, len(owner)) % np.minimum(910, n_v - owner // 910 * 910))
    assert len(nb) > 1024 * 2048
    graph = csr_matrix((np.ones(len(owner), dtype=np.int8), nb[before:before + len(owner)], off - before), shape=(n_v, n_v))
    _, comp = connected_components(graph, directed=False)
    least = np.full(comp.max() + 1, n_v, dtype=np.int64)
    np.minimum.at(least, comp, np.arange(n_v))
    want = least[comp].astype(np.uint64)
    r, a = _rig(bam, nb.astype(np.uint64), 4096, (len(nb) + 511) // 512)
    with r:
        d_off = _dev(off.astype(np.uint64))
        for by_page in (False, True, False):                       # nothing cached, all cached
            lb, _ = a.cc(d_off, by_page=by_page)
            assert np.array_equal(_u64(lb), want), by_page
        assert not r.c.aborted()


# vertices without lists before, between and behind those that have some: around the spans from which owners of entries are looked up
@pytest.mark.parametrize("page,share", [(4096, 1), (4096, 4), (8192, 2), (65536, 2)])
@pytest.mark.parametrize("run,scattered", [(4094, 1), (4095, 1), (4096, 1), (32766, 1), (32767, 1), (32768, 1), (70001, 1), (540000, 1), (40, 4099), (3, 70000)])
def test_long_runs_of_vertices_without_lists(bam, page, share, run, scattered):
    """a random graph on some of the vertices: a run of `run` others after the first third of them, another before the first and
    behind the last, and every `scattered`-th vertex of the last eighth of them"""
    n = 4001
    off, nb = oracle.uniform_csr(SEED, n, 24007 if page < 65536 else 90001)
    place = np.arange(n, dtype=np.int64) + run                # where vertex v of that graph is
    place[n // 3:] += run
    place[n - n // 8:] += np.arange(n // 8) * min(scattered - 1, 4000000 // n)
    n_v = int(place[-1]) + 1 + run
    deg = np.zeros(n_v, dtype=np.uint64)
    deg[place] = off[1:] - off[:-1]
    sources = [int(x) for x in oracle.bfs_sources(SEED, off, 2)]
    want = []
    for src in sources:
        lv, it = oracle.bfs_levels(off, nb, src)
        all_levels = np.full(n_v, 0xFFFFFFFF, dtype=np.uint32)
        all_levels[place] = lv
        want.append((all_levels, it))
    comp, _ = oracle.cc_labels(off, nb)
    labels = np.arange(n_v, dtype=np.uint64)
    labels[place] = place[comp.astype(np.int64)].astype(np.uint64)      # (the order of the vertices is the same)
    off, nb = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64), place[nb.astype(np.int64)].astype(np.uint64)
    r, a = _rig(bam, nb, page, max(2, (len(nb) * 8 + page - 1) // page // share))
    with r:
        d_off = _dev(off)
        a.set_graph(d_off)
        for kw in KINDS:
            for src, (lv_want, it_want) in zip(sources, want):
                lv, it = a.bfs(d_off, int(place[src]), **kw)
                assert np.array_equal(lv.cpu().numpy().view(np.uint32), lv_want) and it == it_want, kw
        for by_page in (False, True):
            lb, _ = a.cc(d_off, by_page=by_page)
            assert np.array_equal(_u64(lb), labels), by_page
        assert not r.c.aborted()


def test_a_run_of_vertices_without_lists_is_not_gone_over(bam):
    """2^24 of them in the middle: one wave went over them on every level, 200 ms a call (and 1 ms vertex by vertex)"""
    import time
    import torch
    n, run = 4001, 1 << 24
    off, nb = oracle.uniform_csr(SEED, n, 24007)
    place = np.arange(n, dtype=np.int64)
    place[n // 2:] += run
    deg = np.zeros(n + run, dtype=np.uint64)
    deg[place] = off[1:] - off[:-1]
    r, a = _rig(bam, nb, 4096, 200)
    with r:
        d_off = _dev(np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64))
        r.backing(len(nb))[:] = place[nb.astype(np.int64)]
        a.set_graph(d_off)
        for call in (lambda: a.bfs(d_off, int(place[int(nb[0])]), frontier=True), lambda: a.bfs(d_off, int(place[int(nb[0])]), coarse=64), lambda: a.cc(d_off)):
            took = []
            for _ in range(4):
                torch.cuda.synchronize()
                t = time.perf_counter()
                call()
                torch.cuda.synchronize()
                took.append(time.perf_counter() - t)
            assert min(took) < 0.04, took


@pytest.mark.parametrize("n_v", [70001, 1048575, 1600003, (1 << 21) - 1])
@pytest.mark.parametrize("cut", [2, 1000])
def test_components_that_label_propagation_was_broken_off_in(bam, n_v, cut):
    """two paths, the shorter below or in the middle of the longer: six sweeps leave chains of a sixth of their length.  Joined as they were
    they took 0.36 s from 1.6 million vertices on, where some waves walked down what others had not come to (1.4 ms before)"""
    import time
    import torch
    v = np.arange(n_v, dtype=np.int64)
    low, high = (0, n_v // cut) if cut == 2 else (n_v // 3, n_v // 3 + n_v // cut)      # the shorter path: [low, high)
    path = (v >= low) & (v < high)
    order = np.concatenate([v[path], v[~path]])                # neighbours along it, but for the step from the one path to the other
    linked = np.ones(n_v - 1, dtype=bool)
    linked[path.sum() - 1] = False
    src, dst = order[:-1][linked], order[1:][linked]
    u, w = np.concatenate([src, dst]), np.concatenate([dst, src])
    by = np.lexsort((w, u))
    off = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n_v))]).astype(np.uint64)
    nb = w[by].astype(np.uint64)
    want = np.where(path, low, 0 if low else high).astype(np.uint64)
    r, a = _rig(bam, nb, 4096, (len(nb) + 511) // 512)
    with r:
        d_off = _dev(off)
        a.set_graph(d_off)
        took = []
        for _ in range(4):
            torch.cuda.synchronize()
            t = time.perf_counter()
            lb, it = a.cc(d_off, by_page=True)
            torch.cuda.synchronize()
            took.append(time.perf_counter() - t)
            assert np.array_equal(_u64(lb), want) and (it == 8 or len(nb) <= 1 << 17), it
        assert min(took) < 0.04, took
        assert not r.c.aborted()


@pytest.mark.parametrize("n_levels", [1, 2, 5, 6, 7, 11, 12, 13, 19])
@pytest.mark.parametrize("entries,cache_pages", [(1, 64), (700, 6)])
def test_as_many_levels_as_are_queued_at_a_time(bam, n_levels, entries, cache_pages):
    """a path, one vertex a level: around the number of sweeps between two looks of the host, all edges cached and most of them not
    (every list holds its one neighbour `entries` times)"""
    off = np.concatenate([np.arange(n_levels) * entries, [(n_levels - 1) * entries], [(n_levels - 1) * entries]]).astype(np.uint64)[: n_levels + 1]
    nb = np.repeat(np.arange(1, max(n_levels, 2)), entries).astype(np.uint64)[: max(1, (n_levels - 1) * entries)]
    if n_levels == 1:
        off, nb = np.array([0, 0, 1], dtype=np.uint64), np.zeros(1, dtype=np.uint64)      # the source has no list
    r, a = _rig(bam, nb, 4096, cache_pages)
    with r:
        _check_bfs(r, a, off, nb, [0])


@pytest.mark.parametrize("by_page", [False, True])
def test_levels_after_components_with_one_plan(bam, by_page):
    """the list of missing pages is empty again when a call ends, whichever call comes next"""
    off, nb = oracle.uniform_csr(SEED, 20011, 60007)
    src = int(oracle.bfs_sources(SEED, off, 1)[0])
    want, want_it = oracle.bfs_levels(off, nb, src)
    labels, _ = oracle.cc_labels(off, nb)
    r, a = _rig(bam, nb, 4096, 24)
    with r:
        d_off = _dev(off)
        a.set_graph(d_off)
        for _ in range(3):
            lb, _ = a.cc(d_off, by_page=by_page)
            assert np.array_equal(_u64(lb), labels)
            lv, it = a.bfs(d_off, src, by_page=by_page)
            assert np.array_equal(lv.cpu().numpy().view(np.uint32), want) and it == want_it
        assert not r.c.aborted()


def test_a_vertex_found_two_levels_ahead_and_then_nearer(bam):
    """Twelve pages behind eight, read front to back by one wave.  Page 1: vertex 1 (level 1) finds vertex 3 (level 2).  Page 2 is
    there for vertex 2 (level 1) and holds the list of vertex 3, which finds vertex 9 ahead, as of level 3.  Page 3: vertex 4
    (level 1) has it next to itself.  There is no level 3, and the sweep that looks for one must not count."""
    lists = {0: [1, 2, 4], 1: [3], 2: [5], 3: [9], 4: [9]}
    place = {0: 0, 1: 512, 2: 1024, 3: 1024 + 300, 4: 1536}
    n_edges, n_v = 12 * 512, 20
    order = [0, 10, 1, 11, 2, 12, 3, 13, 4, 14]            # 10, ... fill the pages up; nobody leads to them
    at, off_of, nb = 0, {}, np.full(n_edges, 15, dtype=np.uint64)
    for k, v in enumerate(order):
        off_of[v] = at
        if v in lists:
            assert at == place[v]
            nb[at:at + len(lists[v])] = lists[v]
            at += len(lists[v])
        else:
            at = place[order[k + 1]] if k + 1 < len(order) else n_edges
    # vertices are numbered along the array
    rank = {v: k for k, v in enumerate(order)}
    rank.update({v: len(order) + k for k, v in enumerate(x for x in range(n_v) if x not in rank)})
    off = np.full(n_v + 1, n_edges, dtype=np.uint64)
    for k, v in enumerate(order):
        off[k] = off_of[v]
    nb = np.array([rank[int(x)] for x in nb], dtype=np.uint64)
    want, want_it = oracle.bfs_levels(off, nb, rank[0])
    assert want_it == 3 and want[rank[9]] == 2 and want[rank[3]] == 2
    r, a = _rig(bam, nb, 4096, 8)
    with r:
        _check_bfs(r, a, off, nb, [rank[0]] * 3)


@pytest.mark.parametrize("page,share", [(4096, 2), (4096, 3), (4096, 60), (8192, 4)])
def test_levels_where_a_sweep_brings_in_more_than_the_cache_holds(bam, page, share):
    """slots used again for the next chunk: a cache that is empty, then full of another array's changed pages, then of the
    edges; nobody's elements suffer, and the other array's go to the store"""
    off, nb = oracle.rmat_csr(SEED, 14)
    per = page // 8
    pages = (len(nb) + per - 1) // per
    cache_pages = max(3, pages // share)
    src = int(oracle.bfs_sources(SEED, off, 1)[0])
    want, want_it = oracle.bfs_levels(off, nb, src)
    n_b = cache_pages * per - 5
    with Rig(bam, (pages + cache_pages) * page, backing=True, n_queues=16, depth=256, stage_bytes=page) as r:
        store = r.backing((pages + cache_pages) * per)
        store[:] = oracle.store(SEED, 0, len(store))
        store[:len(nb)] = nb
        pc = bam.PageCache(page, cache_pages, 0, r.c)
        rs = [bam.Range(0, len(nb), 0, pages, 0, page, pc, 0), bam.Range(0, n_b, pages, cache_pages, 0, page, pc, 0)]
        a, b = bam.Array(len(nb), 0, [rs[0]], 0), bam.Array(n_b, pages * page, [rs[1]], 0)
        d_off = _dev(off)
        a.set_graph(d_off)
        new = np.random.default_rng(page + share).integers(0, 1 << 62, n_b, dtype=np.int64).astype(np.uint64)
        for others in (False, True, False):
            if others:
                b.write(n_b, _dev(new))
            for _ in range(2):
                lv, it = a.bfs(d_off, src, by_page=True)
                assert np.array_equal(lv.cpu().numpy().view(np.uint32), want) and it == want_it, others
        assert np.array_equal(_u64(a.gather(len(nb))), nb) and np.array_equal(_u64(b.gather(n_b)), new)
        pc.flush()
        assert np.array_equal(store[pages * per:pages * per + n_b], new) and np.array_equal(store[:len(nb)], nb)
        assert not r.c.aborted()
        for x in (a, b, rs[0], rs[1], pc):
            x.close()
