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
