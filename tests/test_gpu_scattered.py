"""Scattered reads in several launches (bam_array_gather, bam_array_read): what is resident first, then the rest, in order of its pages or in stretches of the range."""
import math

import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _dev, _u64  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


IN_FLIGHT = 1 << 18        # requests that are on their way together in a launch that can miss
SLICE = 1 << 22            # requests that are put in order of their pages together


def _page_by_page(pages, cache_pages, n):
    """whether a page that somebody waits for is fetched once, and all requests that wait for it count as misses, whichever launches do it (_in_order)"""
    if pages <= cache_pages or 2 * n < pages - 1 or cache_pages < 4096:
        return False
    if 2 * pages > 5 * cache_pages:
        return n >= IN_FLIGHT or n >= 4 * pages
    if pages > 2 * cache_pages:
        beyond = (n >> 17) * (pages - 2 * cache_pages)
        return n >= 3 << 17 or beyond >= cache_pages if pages - cache_pages >= 24576 else beyond > cache_pages
    return n > IN_FLIGHT and pages - cache_pages >= (16384 if pages == 2 * cache_pages else 24576)


def _in_order(pages, cache_pages, n, page=4096):
    """whether the requests that the first launch leaves are put in order of their pages"""
    if pages <= cache_pages or n <= IN_FLIGHT and n < pages + 2 * cache_pages:
        return False
    if -math.expm1(-n / pages) * pages < (1.0 if n <= IN_FLIGHT else 0.9) * cache_pages or n > SLICE and pages <= 2 * cache_pages:
        return False
    if pages > 1 << 26 or pages // max(4, (1 << (20 if page < 4096 else 21)) // cache_pages) >= min(n, SLICE):
        return False
    return not (_page_by_page(pages, cache_pages, n) and (n > SLICE or pages <= 2 * cache_pages and cache_pages >= 1 << 18))


# pages of data and of cache: everything resident; just below and at the smallest cache that is fetched for page by page, one
# stretch and several; requests around the numbers where the shape of the launch changes, and fewer than a request per two pages
@pytest.mark.parametrize("pages,cache_pages,n", [(4096, 4096, (1 << 20) + 1), (4100, 4095, 1 << 14), (4100, 4096, (1 << 14) - 1), (4100, 4096, (1 << 14) + 77),
                                                 (12289, 4096, 100003), (12289, 5000, (1 << 20) - 1), (40000, 4096, 19999), (40000, 4096, 20001),
                                                 (4100, 4095, IN_FLIGHT + 1), (4100, 4096, IN_FLIGHT), (4100, 4096, IN_FLIGHT + 1), (8192, 4096, IN_FLIGHT), (8193, 4096, 4 * 8193 - 1),
                                                 (8193, 4096, 4 * 8193), (70000, 8192, IN_FLIGHT - 1), (70000, 8192, IN_FLIGHT), (70000, 8192, IN_FLIGHT + 65),
                                                 (8193, 4096, IN_FLIGHT + 1), (10240, 4096, (1 << 17) * 3 - 1), (10240, 4096, (1 << 17) * 3), (10241, 4096, IN_FLIGHT - 1), (10241, 4096, IN_FLIGHT), (32766, 16383, IN_FLIGHT + 1), (32768, 16384, IN_FLIGHT), (32768, 16384, IN_FLIGHT + 1),
                                                 (57344, 32769, IN_FLIGHT + 1), (57344, 32768, IN_FLIGHT + 1),
                                                 (40960, 16384, IN_FLIGHT - 1), (40960, 16384, IN_FLIGHT), (40000, 15424, 3 << 17)])
def test_scattered_reads_element_by_element(bam, pages, cache_pages, n):
    """Every element of a gather and the sum of the same requests, twice (the second call finds what the first left behind),
    with a few requests outside the array (they read as 0 and are not counted) and a skewed half; every request inside is
    counted once and misses cover the reads from the store.  Page by page each page asked for is read once, cold or not.  (All sizes that are
    fetched for page by page go in order of their pages here; in stretches: below.)"""
    assert not _page_by_page(pages, cache_pages, n) or _in_order(pages, cache_pages, n)
    n_elems = pages * 512 - 37
    words = oracle.store(SEED, 0, n_elems)
    rng = np.random.default_rng(n)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(n_elems, 4096, cache_pages)
        idx = rng.integers(0, n_elems, n).astype(np.uint64)
        idx[::2] = (rng.random(len(idx[::2])) ** 4 * n_elems).astype(np.uint64)
        outside = rng.integers(0, n, 5)
        idx[outside] = np.array([n_elems, n_elems + 1, 1 << 40, (1 << 64) - 1, (1 << 63)], dtype=np.uint64)
        inside = idx < n_elems
        want = np.where(inside, words[np.where(inside, idx, 0).astype(np.int64)], 0).astype(np.uint64)
        d_idx = _dev(idx)
        asked = len(np.unique(idx[inside] // 512))
        for rep in range(2):
            assert np.array_equal(_u64(a.gather(n, d_idx)), want), rep
            st = a.stats()
            if _page_by_page(pages, cache_pages, n):
                assert st["read_io_cnt"] == asked if rep == 0 else st["read_io_cnt"] <= asked, (st, asked)
            assert st["access_cnt"] == inside.sum() and st["hit_cnt"] + st["miss_cnt"] == st["access_cnt"], st
            assert st["read_io_cnt"] <= st["miss_cnt"] or rep == 0, st
            assert a.read(n, d_idx) == int(np.sum(want, dtype=np.uint64)), rep
            assert a.stats()["access_cnt"] == inside.sum()
        if cache_pages >= pages:
            a.stats()
            a.gather(n, d_idx)
            assert a.stats()["hit_cnt"] == inside.sum()
        assert not r.c.aborted() and r.c.info()["error_completions"] == 0


# two stretches, three (the last cut short), four (of 512 pages more than a quarter); the smallest cache; one request more than goes in order
@pytest.mark.parametrize("pages,cache_pages,n", [(65536, 32768, SLICE + 13), (49157, 24576, SLICE + 64), (40000, 16384, SLICE + 1), (12289, 4096, SLICE + 77), (16384, 4096, 2 * SLICE + 5)])
@pytest.mark.parametrize("page", [512, 4096])
def test_stretches_element_by_element(bam, page, pages, cache_pages, n):
    """more requests than are put in order together: the pages that somebody waits for are fetched a stretch of the range at a time, each once, and then
    the requests for them are read; a skewed half, some outside the array, one page that most ask for"""
    assert _page_by_page(pages, cache_pages, n) and not _in_order(pages, cache_pages, n, page)
    n_elems = pages * page // 8 - 37
    words = oracle.store(SEED, 0, n_elems)
    rng = np.random.default_rng(n)
    with Rig(bam, pages * page // 65536 * 65536 + 65536, n_queues=16, depth=256) as r:
        a = r.array(n_elems, page, cache_pages)
        idx = rng.integers(0, n_elems, n).astype(np.uint64)
        idx[::2] = (rng.random(len(idx[::2])) ** 4 * n_elems).astype(np.uint64)
        idx[n // 3:n // 3 + 9999] = 5 * (page // 8) + 3
        idx[rng.integers(0, n, 5)] = np.array([n_elems, n_elems + 1, 1 << 40, (1 << 64) - 1, 1 << 63], dtype=np.uint64)
        inside = idx < n_elems
        want = np.where(inside, words[np.where(inside, idx, 0).astype(np.int64)], 0).astype(np.uint64)
        d_idx = _dev(idx)
        asked = len(np.unique(idx[inside] // (page // 8)))
        for rep in range(2):
            assert np.array_equal(_u64(a.gather(n, d_idx)), want), rep
            st = a.stats()
            assert st["read_io_cnt"] == asked if rep == 0 else st["read_io_cnt"] <= asked, (st, asked)
            assert st["access_cnt"] == inside.sum() and st["hit_cnt"] + st["miss_cnt"] == st["access_cnt"], st
            assert a.read(n, d_idx) == int(np.sum(want, dtype=np.uint64)), rep
            assert a.stats()["access_cnt"] == inside.sum()
        assert not r.c.aborted() and r.c.info()["error_completions"] == 0


@pytest.mark.parametrize("page", [512, 4096, 8192, 65536])
@pytest.mark.parametrize("first,offset", [(0, 0), (1000, 0), (0, 24), (777, 504)])
def test_scattered_reads_of_ranges_that_begin_inside_a_page(bam, page, first, offset):
    """other page sizes, ranges whose first element is not the array's first and does not start a page; resident, and larger than the
    cache, requests in front of the range and behind it among them (they read as 0)"""
    from bam_amd import Array, PageCache, Range
    per = page // 8
    pages, n = 10300, IN_FLIGHT + 77
    n_elems = (pages * page - offset) // 8 - 3
    if page == 65536:
        pages, n_elems = 4500, 4500 * per - offset // 8 - 3
    words = oracle.store(SEED, 3 * per + offset // 8, n_elems)
    rng = np.random.default_rng(page + first)
    idx = (rng.integers(0, n_elems, n) + first).astype(np.uint64)
    idx[rng.integers(0, n, 6)] = np.array([first - 1 if first else (1 << 64) - 1, 0 if first else n_elems, first + n_elems, first + n_elems + 1, 1 << 40, (1 << 64) - 1], dtype=np.uint64)
    at = idx - np.uint64(first)
    inside = at < n_elems
    want = np.where(inside, words[np.where(inside, at, 0).astype(np.int64)], 0).astype(np.uint64)
    for cache_pages in (4096, pages):
        with Rig(bam, (pages + 4) * page // 65536 * 65536 + 65536, n_queues=16, depth=256) as r:
            pc = PageCache(page, cache_pages, 0, r.c)
            rg = Range(first, first + n_elems, 3, pages, offset, page, pc, 0)
            a = Array(first + n_elems, 0, [rg], 0)
            d_idx = _dev(idx)
            for rep in range(2):
                assert np.array_equal(_u64(a.gather(n, d_idx)), want), (cache_pages, rep)
                assert a.stats()["access_cnt"] == inside.sum()
                assert a.read(n, d_idx) == int(np.sum(want, dtype=np.uint64)), (cache_pages, rep)
                assert a.stats()["access_cnt"] == inside.sum()
            assert not r.c.aborted()
            a.close(); rg.close(); pc.close()


def test_counters_of_reads_in_two_launches(bam):
    """requests that the first launch leaves count by what they find in the second: of 2^22 for one page that is on the store, those
    looked at once it is there are hits, in several times as many waves as the device holds; page by page none is"""
    n = 1 << 22
    for pages, cache_pages, by_page in ((600, 512, False), (4200, 4096, False), (10300, 4096, True)):
        with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
            a = r.array(pages * 512, 4096, cache_pages)
            assert _page_by_page(pages, cache_pages, n) == by_page
            idx = np.random.default_rng(4).integers(5 * 512, 6 * 512, n).astype(np.uint64)
            assert a.read(n, _dev(idx)) == int(np.sum(oracle.store(SEED, 0, 6 * 512)[idx.astype(np.int64)], dtype=np.uint64))
            st = a.stats()
            assert st["access_cnt"] == n and st["hit_cnt"] + st["miss_cnt"] == n and st["read_io_cnt"] == 1, st
            assert st["hit_cnt"] == 0 if by_page else st["hit_cnt"] > n // 2, st
            a.read(n, _dev(idx))
            assert a.stats()["hit_cnt"] == n and not r.c.aborted()


def test_gathers_from_a_large_resident_array(bam):
    """more than the last-level cache holds, around the number of requests from which they run in two launches; some pages missing"""
    pages = (1 << 17) + 1
    n_elems = pages * 512 - 5
    words = oracle.store(SEED, 0, n_elems)
    idx = np.random.default_rng(9).integers(0, n_elems, (1 << 21) + 1).astype(np.uint64)
    d = _dev(idx)
    want = words[idx.astype(np.int64)]
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(n_elems, 4096, pages)
        for n in ((1 << 21) + 1, (1 << 21) - 1, 1 << 21):
            assert np.array_equal(_u64(a.gather(n, d)), want[:n]), n
            assert a.stats()["access_cnt"] == n
        assert not r.c.aborted()


def test_gathers_on_several_streams_of_one_array(bam):
    """Six streams gather from one array at once, page by page, each its own requests and with notes of its own."""
    import torch
    pages, n = 10300, 60001
    n_elems = pages * 512
    words = oracle.store(SEED, 0, n_elems)
    rng = np.random.default_rng(5)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(n_elems, 4096, 4096)
        reqs = [rng.integers(0, n_elems, n).astype(np.uint64) for _ in range(6)]
        d = [_dev(x) for x in reqs]
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream() for _ in d]
        outs = [[] for _ in d]
        for rep in range(3):
            for k, s in enumerate(streams):
                with torch.cuda.stream(s):
                    outs[k].append(a.gather(n, d[k]))
        torch.cuda.synchronize()
        for k, x in enumerate(reqs):
            for o in outs[k]:
                assert np.array_equal(_u64(o), words[x.astype(np.int64)]), k
        assert a.stats()["access_cnt"] == 6 * 3 * n and not r.c.aborted()
