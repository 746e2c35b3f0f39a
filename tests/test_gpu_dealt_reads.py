"""Scattered reads of arrays larger than their cache: requests put in order of their pages, and few requests spread over waves."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _dev, _u64  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


def _check(a, n, idx, words, base=0, reps=2):
    inside = idx - np.uint64(base) < len(words)
    want = np.where(inside, words[np.where(inside, idx - np.uint64(base), 0).astype(np.int64)], 0).astype(np.uint64)
    d = _dev(idx)
    for rep in range(reps):
        assert np.array_equal(_u64(a.gather(n, d)), want), rep
        st = a.stats()
        assert st["access_cnt"] == inside.sum() and st["hit_cnt"] + st["miss_cnt"] == st["access_cnt"], st
        assert a.read(n, d) == int(np.sum(want, dtype=np.uint64)), rep
        assert a.stats()["access_cnt"] == inside.sum()


# caches of two pages up, turns of 4 pages to 1024, a range's last turn and its last 1024 pages cut short; requests: one, around a wave's
# and where more are spread over each, on both sides of where they are put in order, more than one slice
@pytest.mark.parametrize("page,pages,cache_pages", [(4096, 3, 2), (4096, 11, 8), (4096, 65, 17), (4096, 1025, 256), (8192, 1030, 515), (65536, 70, 20), (512, 2049, 700),
                                                    (512, 70001, 17000), (4096, 4100, 3900)])
def test_every_element(bam, page, pages, cache_pages):
    n_elems = pages * page // 8 - 5
    words = oracle.store(SEED, 0, n_elems)
    rng = np.random.default_rng(pages)
    line = pages + 2 * cache_pages
    with Rig(bam, pages * page // 65536 * 65536 + 65536, n_queues=16, depth=256) as r:
        a = r.array(n_elems, page, cache_pages)
        for n in (1, 63, 65, 1023, line - 1, line, 4 * line + 1, (1 << 18) + 65):
            idx = rng.integers(0, n_elems, n).astype(np.uint64)
            idx[rng.integers(0, n, 3)] = np.array([n_elems, (1 << 64) - 1, 1 << 45], dtype=np.uint64)
            _check(a, n, idx, words)
        assert not r.c.aborted() and r.c.info()["error_completions"] == 0


@pytest.mark.parametrize("kind", ["one element", "one page", "skewed", "in order", "backwards"])
def test_orders_and_concentrations(bam, kind):
    """cold each time: the requests for a page are as many as there are, and each page is read from the store once while half the cache holds what is asked for together"""
    pages, cache_pages, n = 3000, 1000, 200001
    n_elems = pages * 512 - 1
    words = oracle.store(SEED, 0, n_elems)
    rng = np.random.default_rng(3)
    idx = {"one element": np.full(n, 77 * 512 + 5), "one page": 77 * 512 + rng.integers(0, 512, n), "skewed": rng.random(n) ** 6 * n_elems,
           "in order": np.arange(n) * 7, "backwards": n_elems - 1 - np.arange(n) * 7}[kind].astype(np.uint64)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(n_elems, 4096, cache_pages)
        assert np.array_equal(_u64(a.gather(n, _dev(idx))), words[idx.astype(np.int64)])
        assert a.stats()["read_io_cnt"] == len(np.unique(idx // 512))
        _check(a, n, idx, words)
        assert not r.c.aborted()


def test_more_requests_than_a_slice(bam):
    pages, cache_pages, n = 2000, 700, (1 << 22) + 12345
    words = oracle.store(SEED, 0, pages * 512)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(pages * 512, 4096, cache_pages)
        _check(a, n, np.random.default_rng(1).integers(0, pages * 512, n).astype(np.uint64), words, reps=1)
        assert not r.c.aborted()


@pytest.mark.parametrize("page,offset,first", [(512, 0, 1000), (4096, 24, 0), (8192, 504, 777)])
def test_ranges_that_begin_inside_a_page(bam, page, offset, first):
    from bam_amd import Array, PageCache, Range
    per, pages, cache_pages = page // 8, 600, 300
    n_elems = (pages * page - offset) // 8 - 3
    words = oracle.store(SEED, 3 * per + offset // 8, n_elems)
    rng = np.random.default_rng(page)
    with Rig(bam, (pages + 4) * page // 65536 * 65536 + 65536, n_queues=16, depth=256) as r:
        pc = PageCache(page, cache_pages, 0, r.c)
        rg = Range(first, first + n_elems, 3, pages, offset, page, pc, 0)
        a = Array(first + n_elems, 0, [rg], 0)
        for n in (100, 1199, 20000):
            idx = (rng.integers(0, n_elems, n) + first).astype(np.uint64)
            idx[:3] = np.array([(first - 1) % (1 << 64), first + n_elems, (1 << 64) - 1], dtype=np.uint64)
            _check(a, n, idx, words, first)
        assert not r.c.aborted()
        a.close(); rg.close(); pc.close()


@pytest.mark.parametrize("cache_pages", [64, 300])
def test_beside_a_sweep_that_holds_pages(bam, cache_pages):
    """A sweep over a graph holds up to half of the cache while it waits for more: gathers of another array, on two streams, hold none while they wait"""
    import torch
    from test_gpu_beside_evictions import OTHER, Shared
    off, nb = oracle.uniform_csr(SEED, 20011, 150007)
    src = int(oracle.bfs_sources(SEED, off, 1)[0])
    levels, n_levels = oracle.bfs_levels(off, nb, src)
    labels, _ = oracle.cc_labels(off, nb)
    n = 8001
    with Shared(bam, [len(nb)], cache_pages) as s:
        s.of(0, len(nb))[:] = nb
        d_off = _dev(off)
        s.arrs[0].set_graph(d_off)
        reqs = [np.random.default_rng(k).integers(0, OTHER * 512, n).astype(np.uint64) for k in range(2)]
        d, streams = [_dev(x) for x in reqs], [torch.cuda.Stream() for _ in reqs]
        for rep in range(4):
            torch.cuda.synchronize()
            outs = []
            for k in range(2):
                with torch.cuda.stream(streams[k]):
                    outs.append([s.arrs[-1].gather(n, d[k]) for _ in range(3)])
            if rep & 1:
                lb, _ = s.arrs[0].cc(d_off)
                assert np.array_equal(_u64(lb), labels), rep
            else:
                lv, it = s.arrs[0].bfs(d_off, src)
                assert np.array_equal(lv.cpu().numpy().view(np.uint32), levels) and it == n_levels, rep
            torch.cuda.synchronize()
            for k in range(2):
                for o in outs[k]:
                    assert np.array_equal(_u64(o), s.of(1, OTHER * 512)[reqs[k].astype(np.int64)]), (rep, k)
            assert not s.r.c.aborted()


def test_many_streams_and_arrays_of_one_cache(bam):
    """Eight streams over two arrays behind one small cache, most of whose batches come in parts."""
    import torch
    from bam_amd import Array, PageCache, Range
    pages, n = 900, 9001
    words = oracle.store(SEED, 0, 2 * pages * 512)
    rng = np.random.default_rng(5)
    with Rig(bam, 2 * pages * 4096, n_queues=16, depth=256) as r:
        pc = PageCache(4096, 256, 0, r.c)
        rgs = [Range(0, pages * 512, k * pages, pages, 0, 4096, pc, 0) for k in range(2)]
        arrays = [Array(pages * 512, 0, [rg], 0) for rg in rgs]
        reqs = [rng.integers(0, pages * 512, n).astype(np.uint64) for _ in range(8)]
        d = [_dev(x) for x in reqs]
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream() for _ in d]
        outs = [[] for _ in d]
        for rep in range(4):
            for k, s in enumerate(streams):
                with torch.cuda.stream(s):
                    outs[k].append(arrays[k % 2].gather(n, d[k]))
        torch.cuda.synchronize()
        for k, x in enumerate(reqs):
            for o in outs[k]:
                assert np.array_equal(_u64(o), words[x.astype(np.int64) + k % 2 * pages * 512]), k
        assert not r.c.aborted()
        for a in arrays: a.close()
        for rg in rgs: rg.close()
        pc.close()


# many pages for each request: the most with 2^14 and 2^18 slots and one more, and a range with more pages than counts are kept for
@pytest.mark.parametrize("page,pages,cache_pages,n,dealt", [(512, 1 << 22, 1 << 18, (1 << 20) + 1, True), (512, (1 << 22) + 4, 1 << 18, 1 << 20, False), (512, 1 << 24, 1 << 18, (1 << 18) + 1, False),
                                                            (4096, (1 << 25) - 8, 1 << 14, (1 << 18) + 1, True), (4096, (1 << 25) + 256, 1 << 14, (1 << 18) + 1, False),
                                                            (512, (1 << 26) + 8, 1 << 12, (1 << 18) + 1, False)])
def test_many_pages_to_a_request(bam, page, pages, cache_pages, n, dealt):
    """scattered reads keep a count and a beginning for every page only while there are not too many pages for each request (and slot), and
    no more of them than are worth it: seen by the memory that the first calls on a stream take"""
    import torch
    from bam_amd import gen
    n_elems = pages * page // 8
    want = oracle.lib().bo_gather_sum(SEED, SEED, 0, n, n_elems)
    with Rig(bam, pages * page, n_queues=16, depth=256) as r:
        a = r.array(n_elems, page, cache_pages)
        idx = gen.gather_indices(SEED, n, n_elems)
        out = torch.empty(n, dtype=torch.int64, device="cuda")
        assert int(out.sum()) is not None                              # what torch itself needs is there
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        got = a.read(n, idx)
        taken = free - torch.cuda.mem_get_info()[0]
        assert got == want
        assert int(a.gather(n, idx).sum()) % (1 << 64) == want
        assert a.stats()["access_cnt"] == 2 * n and not r.c.aborted()
        assert taken >= 8 * pages if dealt else taken < 8 * pages // 2, (taken, pages)


@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
def test_a_shape_that_is_named_is_the_one_that_runs(bam, lanes):
    """two launches keep a bit for each request between them, requests in order of their pages 16 bytes, and those only bam_array_read may have: seen by the memory taken"""
    import torch
    from bam_amd import gen
    pages, cache_pages, n = 8192, 2048, (1 << 20) + 37
    want = oracle.lib().bo_gather_sum(SEED, SEED, 0, n, pages * 512)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(pages * 512, 4096, cache_pages)
        idx = gen.gather_indices(SEED, n, pages * 512)
        for few in (64, 1 << 16):                                                  # what torch and the kernels' own frames take is there, and the words of the stream
            a.read_shaped(few, idx, a.TWO_LAUNCHES, lanes)
        a.stats()
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for rep in range(2):
            assert a.read_shaped(n, idx, a.TWO_LAUNCHES, lanes, block_size=64) == want
            st = a.stats()
            assert st["access_cnt"] == n and st["hit_cnt"] + st["miss_cnt"] == st["access_cnt"], st
        assert free - torch.cuda.mem_get_info()[0] < 4 * n
        assert a.read(n, idx) == want
        assert free - torch.cuda.mem_get_info()[0] >= 16 * n
        assert not r.c.aborted()
