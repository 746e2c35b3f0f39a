"""bam_cache_stream of resident pages in rows of 4 KiB, whatever the page size, and runs shared out anew."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _dev  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu
MASK = (1 << 64) - 1


# pages of one row to sixteen groups; runs of fewer pages than a group, of no whole number of groups, of more than 64 notes; a last page
# that the array ends in, and one that it fills
@pytest.mark.parametrize("page", [512, 1024, 2048, 4096, 8192, 65536])
@pytest.mark.parametrize("short", [0, 37])
def test_sums_and_counters(bam, page, short):
    pages = 150 if page == 65536 else 1203
    per, n_elems = page // 8, pages * page // 8 - short
    words = oracle.store(SEED, 0, pages * per)
    perm = np.random.default_rng(page).permutation(pages).astype(np.uint64)
    with Rig(bam, (pages * page + 65535) // 65536 * 65536, n_queues=16, depth=256) as r:
        for cache_pages in (pages, pages * 3 // 4):
            a = r.array(n_elems, page, cache_pages)
            a.gather(cache_pages, None, stride=per)
            for ppw in (1, 3, 8, 17, 70):
                waves = pages // ppw
                whole = words[:waves * ppw * per].copy()
                beyond = words[n_elems:waves * ppw * per]
                for mode in (0, 1, 2):
                    want = int(np.sum(whole, dtype=np.uint64)) - (int(np.sum(beyond, dtype=np.uint64)) if mode < 2 else 0)
                    a.stats()
                    for rep in range(2):
                        assert a.stream(waves, ppw, mode=mode) == want & MASK, (cache_pages, ppw, mode, rep)
                    counted = a.stats()["access_cnt"]
                    if not short:
                        assert counted == 2 * waves * ppw * (per if mode == 0 else 64 if mode == 1 else 1), (ppw, mode, counted)
            # runs at page numbers of the caller's: as many pages each as the array has behind them
            starts = perm[perm < pages - 17][:40]
            for ppw in (1, 8, 13):
                want = sum(int(np.sum(words[int(p) * per:min(int(p) * per + ppw * per, n_elems)], dtype=np.uint64)) for p in starts)
                for mode in (0, 1, 2):
                    if mode == 2 and short:
                        continue
                    assert a.stream(len(starts), ppw, _dev(starts), mode=mode) == want & MASK, (cache_pages, ppw, mode)
        assert not r.c.aborted()


def test_a_run_far_outside_is_not_read(bam):
    """page numbers whose elements wrap around: modes 0 and 1 read nothing there"""
    pages, page = 256, 512
    with Rig(bam, pages * page, n_queues=4, depth=256) as r:
        a = r.array(pages * 64, page, pages)
        a.gather(pages, None, stride=64)
        starts = np.array([(1 << 58) - 1, (1 << 57) + 3, pages], dtype=np.uint64)
        for mode in (0, 1):
            assert a.stream(3, 1, _dev(starts), mode=mode) == 0
        assert not r.c.aborted()


@pytest.mark.parametrize("page,offset,first", [(512, 0, 1000), (1024, 24, 0)])
def test_ranges_that_begin_elsewhere(bam, page, offset, first):
    """page by page there; elements in front of the range read as 0 and nobody looks for their pages"""
    from bam_amd import Array, PageCache, Range
    pages = 300
    n_elems = (pages * page - offset) // 8
    with Rig(bam, (pages + 8) * page // 65536 * 65536 + 65536, n_queues=8, depth=256) as r:
        pc = PageCache(page, pages, 0, r.c)
        rg = Range(first, first + n_elems, 0, pages, offset, page, pc, 0)
        a = Array(first + n_elems, 0, [rg], 0)
        words = oracle.store(SEED, offset // 8, n_elems)
        want = int(np.sum(words[:210 * page // 8 - first], dtype=np.uint64))
        for mode in (5, 6, 0, 1, 3, 4):
            for rep in range(2):
                assert a.stream(30, 7, mode=mode) == want, (mode, rep)
        assert not r.c.aborted()
        a.close(); rg.close(); pc.close()


@pytest.mark.parametrize("page", [512, 4096])
@pytest.mark.parametrize("pages,cache_pages", [(240, 256), (1200, 64), (33, 17)])
def test_page_wise_streams_that_share_a_cache(bam, page, pages, cache_pages):
    """Three arrays behind one cache that holds one of them, or less, each streamed page by page on a stream of its own: waves hold nothing while
    they wait, so all of them end, and every page counts once however often it is asked for"""
    import torch
    from bam_amd import Array, PageCache, Range
    per, ppw = page // 8, 17 if pages > 33 else 11
    waves = pages // ppw
    words = oracle.store(SEED, 0, 3 * pages * per).reshape(3, -1)
    with Rig(bam, (3 * pages * page + 65535) // 65536 * 65536, n_queues=8, depth=256) as r:
        pc = PageCache(page, cache_pages, 0, r.c)
        rgs = [Range(0, pages * per, k * pages, pages, 0, page, pc, 0) for k in range(3)]
        arrays = [Array(pages * per, 0, [rg], 0) for rg in rgs]
        want = [int(np.sum(words[k, :waves * ppw * per], dtype=np.uint64)) for k in range(3)]
        streams = [torch.cuda.Stream() for _ in arrays]
        sums = torch.zeros((6, 3), dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        for rep in range(6):
            for k, s in enumerate(streams):
                with torch.cuda.stream(s):
                    arrays[k].stream_async(waves, ppw, sums[rep, k:], mode=2)
        torch.cuda.synchronize()
        for k, a in enumerate(arrays):
            assert [int(x) & MASK for x in sums[:, k]] == [want[k]] * 6, k
            st = a.stats()
            assert st["access_cnt"] == 6 * waves * ppw and st["read_io_cnt"] >= waves * ppw, st
        assert not r.c.aborted()
        for a in arrays: a.close()
        for rg in rgs: rg.close()
        pc.close()


@pytest.mark.parametrize("page,offset,first", [(512, 0, 0), (512, 0, 1000), (4096, 24, 0), (8192, 504, 70000)])
def test_page_wise_runs_that_leave_the_range(bam, page, offset, first):
    """pages in front of the range and behind its last one are not read and not counted; runs named and by turns, resident and not"""
    from bam_amd import Array, PageCache, Range
    pages, per, ppw = 300, page // 8, 21
    n_elems = (pages * page - offset) // 8
    words = oracle.store(SEED, 0, pages * per).reshape(pages, per)

    def model(starts):
        elem = (np.asarray(starts, dtype=np.int64)[:, None] + np.arange(ppw)).ravel() * per
        at = ((elem - first) * 8 + offset) // page
        at = at[(elem >= first) & (at < pages)]
        return int(np.sum(words[at], dtype=np.uint64)), len(at)

    with Rig(bam, (pages + 8) * page // 65536 * 65536 + 65536, n_queues=8, depth=256, stage_bytes=max(4096, page)) as r:
        for cache_pages in (pages, 40):
            pc = PageCache(page, cache_pages, 0, r.c)
            rg = Range(first, first + n_elems, 0, pages, offset, page, pc, 0)
            a = Array(first + n_elems, 0, [rg], 0)
            at = first // per
            named = np.array([0, at + 3, at + pages - 5, at + pages, at + pages + 1, 1 << 40, (1 << 58) // per], dtype=np.uint64)
            for rep in range(2):
                for starts, d in ((named, _dev(named)), (np.arange(40) * ppw, None)):
                    want, n = model(starts)
                    assert a.stream(len(starts), ppw, d, mode=2) == want, (cache_pages, rep)
                    assert a.stats()["access_cnt"] == n
            assert not r.c.aborted()
            a.close(); rg.close(); pc.close()
