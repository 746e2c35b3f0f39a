"""Arrays that the readings along whole pages do not take: pages of 512 bytes or 128 KiB, a range that starts inside a page, two ranges.
Graphs are walked vertex by vertex and over queues there, vectors added element by element; and updates of arrays that outgrow
their cache go through memref and += themselves."""
import ctypes

import numpy as np
import pytest

import oracle
from test_gpu_parity import SEED, Rig, _check_add_chains, _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu

# page size, byte offset of the first element in its page, ranges
LAYOUTS = {"inside": (4096, 808, 1), "two": (4096, 0, 2), "two_inside": (4096, 1600, 2), "small": (512, 0, 1), "large": (131072, 0, 1)}


class Laid:
    """elements behind a cache of their own, laid out as LAYOUTS says: the ranges' pages lie apart on the store"""

    def __init__(self, bam, elems, layout, cache_pages, **kw):
        page, offset, n_ranges = LAYOUTS[layout]
        per, n = page // 8, len(elems)
        cut = [n * k // n_ranges for k in range(n_ranges + 1)]
        pages = [((cut[k + 1] - cut[k]) * 8 + offset + page - 1) // page for k in range(n_ranges)]
        firsts = [3 + sum(pages[:k]) + 5 * k for k in range(n_ranges)]
        total = firsts[-1] + pages[-1] + 1
        self.r = Rig(bam, total * page, backing=True, stage_bytes=max(4096, min(page, 8192)), **kw)
        self.store = self.r.backing(total * per)
        self.parts = [self.store[f * per + offset // 8:][:cut[k + 1] - cut[k]] for k, f in enumerate(firsts)]
        self.put(elems)
        self.pc = bam.PageCache(page, cache_pages, 0, self.r.c)
        self.rs = [bam.Range(cut[k], cut[k + 1], firsts[k], pages[k], offset, page, self.pc, 0) for k in range(n_ranges)]
        self.a = bam.Array(n, 0, self.rs, 0)

    def put(self, elems):
        at = 0
        for p in self.parts:
            p[:] = elems[at:at + len(p)]
            at += len(p)

    def get(self):
        return np.concatenate(self.parts)

    def __enter__(self):
        return self.r, self.a

    def __exit__(self, *exc):
        self.a.close()
        for x in self.rs:
            x.close()
        self.pc.close()
        self.r.close()


def _check_levels(a, off, nb, sources, kinds):
    d_off = _dev(off)
    for kept in (False, True):
        if kept:
            a.set_graph(d_off)
        for src in sources:
            want, want_it = oracle.bfs_levels(off, nb, int(src))
            for kw in kinds:
                lv, it = a.bfs(d_off, int(src), **kw)
                assert np.array_equal(lv.cpu().numpy().view(np.uint32), want) and it == want_it, (kept, int(src), kw)


# vertex by vertex and over a queue, in the order of the vertices between levels and in that of discovery
@pytest.mark.parametrize("layout", list(LAYOUTS))
@pytest.mark.parametrize("scale,share", [(10, 1), (14, 1), (14, 4)])
@pytest.mark.parametrize("sort", ["1", "0"])
def test_levels_vertex_by_vertex_and_over_queues(bam, layout, scale, share, sort, monkeypatch):
    monkeypatch.setenv("BAM_FRONTIER_SORT", sort)
    off, nb = oracle.rmat_csr(SEED, scale)
    pages = len(nb) * 8 // LAYOUTS[layout][0] + 4
    with Laid(bam, nb, layout, max(160, pages // share), n_queues=16, depth=256) as (r, a):
        sources = list(oracle.bfs_sources(SEED, off, 2)) + [int(np.flatnonzero(np.diff(off) == 0)[0])]
        _check_levels(a, off, nb, sources, [{"coarse": 1}, {"coarse": 600}, {"frontier": True}] if sort == "1" else [{"frontier": True}])
        assert a.stats()["read_io_cnt"] > 0 and not r.c.aborted()


@pytest.mark.parametrize("layout", list(LAYOUTS))
@pytest.mark.parametrize("n_v,n_e,share,coarse", [(997, 700, 1, 1), (30011, 20021, 1, 64), (30011, 100003, 3, 600)])
def test_labels_vertex_by_vertex(bam, layout, n_v, n_e, share, coarse):
    off, nb = oracle.uniform_csr(SEED, n_v, n_e)
    want, _ = oracle.cc_labels(off, nb)
    d_off = _dev(off)
    with Laid(bam, nb, layout, max(160, len(nb) * 8 // LAYOUTS[layout][0] // share + 4), n_queues=16, depth=256) as (r, a):
        for kept in (False, True, True):               # calls of one plan run forwards and backwards by turns
            if kept:
                a.set_graph(d_off)
            lb, _ = a.cc(d_off, coarse=coarse)
            assert np.array_equal(_u64(lb), want), kept
        assert not r.c.aborted()


@pytest.mark.parametrize("layout", ["inside", "two", "small"])
@pytest.mark.parametrize("coarse", [1, 200])
def test_hub_lists_in_pieces(bam, layout, coarse):
    """lists of 9000 and 4096 entries on top of a sparse random graph: walked in pieces, a wave each"""
    n_v = 20000
    pu = np.empty(6000, dtype=np.uint64); pv = np.empty(6000, dtype=np.uint64)
    oracle.lib().bo_uniform_edges(SEED, n_v, 0, 6000, pu, pv)
    hubs = [np.full(9000, 7, dtype=np.uint64), np.full(4096, 15000, dtype=np.uint64)]
    leaves = [np.arange(100, 9100, dtype=np.uint64), np.arange(9100, 9100 + 4096, dtype=np.uint64)]
    off, nb = oracle.csr_from_pairs(n_v, np.concatenate([pu] + hubs), np.concatenate([pv] + leaves))
    with Laid(bam, nb, layout, 300 if layout != "small" else 2000, n_queues=8, depth=256) as (r, a):
        _check_levels(a, off, nb, (7, 15000, 100), [{"coarse": coarse}, {"frontier": True}])
        lb, _ = a.cc(_dev(off), coarse=coarse)
        assert np.array_equal(_u64(lb), oracle.cc_labels(off, nb)[0]) and not r.c.aborted()


@pytest.mark.parametrize("empty_every", [0, 4, 2])
def test_lists_that_all_cross_a_page_boundary_vertex_by_vertex(bam, empty_every):
    """lists of 600 entries behind pages of 512 that the array starts inside of"""
    n_v, d = 4096, 600
    deg = np.full(n_v, d, dtype=np.uint64)
    if empty_every:
        deg[empty_every - 1::empty_every] = 0
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    owner = np.repeat(np.arange(n_v, dtype=np.uint64), deg.astype(np.int64))
    nb = (owner + 1 + (np.arange(len(owner), dtype=np.uint64) - off[owner])) % np.uint64(n_v)
    with Laid(bam, nb, "inside", 256, n_queues=8, depth=256) as (r, a):
        _check_levels(a, off, nb, (0, 4092), [{"coarse": 1}, {"coarse": 64}, {"frontier": True}])
        assert a.stats()["read_io_cnt"] > len(nb) // 512 and not r.c.aborted()


@pytest.mark.parametrize("kernel", [dict(coarse=4), dict(frontier=True)])
def test_lost_completion_vertex_by_vertex(bam, kernel):
    """a completion that never comes: the sweep ends, and ids that never arrived stay inside the label array"""
    off, nb = oracle.rmat_csr(SEED, 13)
    laid = Laid(bam, nb, "inside", 64, n_queues=8, depth=256, drop_every=300, limit=300_000)
    with laid as (r, a):
        laid.store[:] = 0
        laid.put(nb)
        lv, it = a.bfs(_dev(off), int(oracle.bfs_sources(SEED, off, 1)[0]), **kernel)
        assert r.c.aborted() and r.t.stats()["dropped"] >= 1 and it >= 1
        lv = lv.cpu().numpy().view(np.uint32)
        assert np.all((lv == 0xFFFFFFFF) | (lv <= it))


@pytest.mark.parametrize("page,offset", [(512, 0), (4096, 808), (16384, 0)])
@pytest.mark.parametrize("n", [511, 5000, 40_003])
def test_sums_element_by_element(bam, page, offset, n):
    """vectors whose pages are not taken whole, several pages of them; every lane keeps a page of each, so the cache holds them all"""
    per = page // 8
    pages = (n * 8 + offset + page - 1) // page
    with Rig(bam, 3 * pages * page, backing=True, n_queues=8, depth=256, stage_bytes=max(4096, min(page, 8192))) as r:
        store = r.backing(3 * pages * per)
        store[:] = oracle.store(SEED, 0, len(store))
        at = [slice(k * pages * per + offset // 8, k * pages * per + offset // 8 + n) for k in range(3)]
        keep = store.copy()
        keep[at[2]] = store[at[0]] + store[at[1]]
        pc = bam.PageCache(page, max(130, 3 * pages + 4), 0, r.c)
        rs = [bam.Range(0, n, k * pages, pages, offset, page, pc, 0) for k in range(3)]
        arrs = [bam.Array(n, k * pages * page, [rs[k]], 0) for k in range(3)]
        for rep in range(2):
            bam.vectoradd(*arrs, n)
            pc.flush()
            assert np.array_equal(store, keep), rep
        assert arrs[0].stats()["access_cnt"] == 2 * n and not r.c.aborted()
        for x in arrs + rs:
            x.close()
        pc.close()


# caches that waves which hold a page of A and of B can fill, and one page more or less than those of A and B
@pytest.mark.parametrize("page,slots,n", [(8192, 97, 66001), (8192, 3, 5000), (8192, 130, 66001), (8192, 131, 66001), (512, 24, 20011), (512, 626, 20011), (512, 627, 20011), (512, 2000, 300007)])
def test_sums_where_the_waves_could_fill_the_cache(bam, page, slots, n):
    """element by element: a wave keeps its pages of A and B while it waits for one of C, so fewer waves run than the cache has slots"""
    pages = (n * 8 + page - 1) // page
    r = Rig(bam, 3 * pages * page, backing=True, n_queues=16, depth=256, stage_bytes=4096)
    store = r.backing(3 * pages * page // 8)
    store[:] = oracle.store(SEED, 0, len(store))
    with r:
        pc = bam.PageCache(page, slots, 0, r.c)
        rs = [bam.Range(0, n, k * pages, pages, 0, page, pc, 0) for k in range(3)]
        arrs = [bam.Array(n, k * pages * page, [rs[k]], 0) for k in range(3)]
        part = [store[k * pages * page // 8:][:n] for k in range(3)]
        for rep in range(3):
            bam.vectoradd(*arrs, n)
            pc.flush()
            assert not r.c.aborted(), rep
            assert np.array_equal(part[2], part[0] + part[1]), rep
        for x in arrs + rs:
            x.close()
        pc.close()


# as many requests as go to bins where the array fits its cache
@pytest.mark.parametrize("api,n", [(0, 1 << 18), (1, 1 << 17), (2, (1 << 17) + 77)])
@pytest.mark.parametrize("layout", ["two", "inside"])
def test_many_updates_element_by_element(bam, api, n, layout):
    n_elems = n + 1001
    rng = np.random.default_rng(n + api)
    x0 = oracle.store(SEED, 5, n_elems)
    # "two": two ranges, all cached; "inside": nine tenths of the pages cached
    laid = Laid(bam, x0, layout, int((n_elems // 512 + 4) * (1.0 if layout == "two" else 0.9)), n_queues=16, depth=256)
    with laid as (r, a):
        idx = rng.permutation(n_elems)[:n].astype(np.uint64)
        vals = rng.integers(1, 1 << 63, n).astype(np.uint64)
        idx[rng.integers(0, n, 2)] = np.array([n_elems, 1 << 40], dtype=np.uint64)
        inside = idx < n_elems
        if layout == "inside":
            idx[inside] = np.sort(idx[inside])             # a wave's lanes on one or two pages: what is missing comes in once
        old = _u64(a.update(api, _dev(idx), _dev(vals), block_size=64))
        assert a.stats()["access_cnt"] == inside.sum()
        assert np.array_equal(old[inside], x0[idx[inside].astype(np.int64)]) and not old[~inside].any()
        x0[idx[inside].astype(np.int64)] += vals[inside]
        laid.pc.flush()
        assert np.array_equal(laid.get(), x0) and not r.c.aborted()


@pytest.mark.parametrize("dist", [0, 1])
def test_sums_over_two_controllers(bam, dist):
    """arrays that are stored twice, and dealt out over two stores: element by element"""
    n, pages = 40_003, 80
    with Rig(bam, 3 * pages * 4096, backing=True, n_queues=8, depth=128) as r0, Rig(bam, 3 * pages * 4096, backing=True, n_queues=8, depth=128) as r1:
        for r in (r0, r1):
            r.backing(3 * pages * 512)[:] = oracle.store(SEED, 0, 3 * pages * 512)
        pc = bam.PageCache(4096, 3 * pages + 30, 0, [r0.c, r1.c])
        rs = [bam.Range(0, n, k * pages, pages, 0, 4096, pc, 0, dist) for k in range(3)]
        arrs = [bam.Array(n, k * pages * 4096, [rs[k]], 0) for k in range(3)]
        x, y = (_u64(z.gather(n, None, stride=1)).copy() for z in arrs[:2])
        for rep in range(2):
            bam.vectoradd(*arrs, n)
            assert np.array_equal(_u64(arrs[2].gather(n, None, stride=1)), x + y), rep
            pc.flush()
        assert not r0.c.aborted() and not r1.c.aborted()
        for z in arrs + rs:
            z.close()
        pc.close()
