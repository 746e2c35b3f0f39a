"""bam_array_update dealt out to bins of pages: numbers of requests around where that begins and around a slice, numbers of pages around
a bin's and around what 512 bins hold one each, all pages resident, none and some, requests scattered, in order and on few pages."""
import ctypes

import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, _check_add_chains, _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("api,n", [(0, 1 << 18), (0, (1 << 18) + 4095), (1, 1 << 17), (2, (1 << 17) + 1), (0, (1 << 20) - 1), (2, 1 << 20), (1, (1 << 20) + 1), (0, (2 << 20) + 77)])
@pytest.mark.parametrize("page,spare,warm", [(4096, 3, 1.0), (4096, 3, 0.0), (512, 1, 0.5), (8192, 40000, 1.0)])
@pytest.mark.parametrize("kind", ["scattered", "in_order", "in_order_at_once"])
def test_updates_without_repeats(bam, api, n, page, spare, warm, kind):
    per = page // 8
    n_elems = n + spare * 7 + 5
    pages = (n_elems + per - 1) // per
    rng = np.random.default_rng(n + api)
    with Rig(bam, pages * page, backing=True, n_queues=16, depth=256, stage_bytes=max(4096, page)) as r:
        x0 = r.backing(n_elems).copy()
        a = r.array(n_elems, page, pages)
        if warm:
            a.gather(max(1, int(pages * warm)), None, stride=per)
        # the first call of an array goes element by element, unless it is a large one, and leaves the memory for the bins behind
        if kind != "in_order_at_once":
            a.update(0, _dev(np.zeros(max(n, 1 << 18), dtype=np.uint64)), _dev(np.zeros(max(n, 1 << 18), dtype=np.uint64)))
        idx = (rng.permutation(n_elems)[:n] if kind == "scattered" else np.arange(n) + 5).astype(np.uint64)
        vals = rng.integers(1, 1 << 63, n).astype(np.uint64)
        outside = rng.integers(0, n, 3)
        idx[outside] = np.array([n_elems, 1 << 40, (1 << 64) - 1], dtype=np.uint64)
        inside = idx < n_elems
        model = x0.copy()
        for rep in range(2):                                  # the second call finds everything resident, and the counts cleared
            a.stats()
            old = _u64(a.update(api, _dev(idx), _dev(vals), block_size=64))
            st = a.stats()
            assert np.array_equal(old[inside], model[idx[inside].astype(np.int64)]) and not old[~inside].any(), rep
            model[idx[inside].astype(np.int64)] += vals[inside]
            assert st["access_cnt"] == inside.sum(), st
            assert rep == 0 and warm < 1 or st["read_io_cnt"] == 0, st
        r.objs[0][2].flush()
        assert np.array_equal(r.backing(n_elems), model) and not r.c.aborted()


@pytest.mark.parametrize("span", [1, 64, 512, 3 * 4096, 40 * 512])
@pytest.mark.parametrize("pages", [1, 511, 512, 513, 1025, 1300])
def test_updates_that_meet(bam, pages, span):
    n, n_elems = (1 << 18) + 333, pages * 512 - 1
    rng = np.random.default_rng(pages + span)
    with Rig(bam, pages * 4096, backing=True, n_queues=8, depth=256) as r:
        x0 = r.backing(n_elems).copy()
        a = r.array(n_elems, 4096, pages)
        idx = (rng.integers(0, n_elems) + rng.integers(0, span, n)).astype(np.uint64) % np.uint64(n_elems)
        vals = rng.integers(1, 1 << 20, n).astype(np.uint64)
        old = _u64(a.update(0, _dev(idx), _dev(vals)))
        model = x0.copy()
        np.add.at(model, idx.astype(np.int64), vals)
        _check_add_chains(x0, idx, vals, old, model)
        # and without a place for what the elements held
        d_idx, d_vals = _dev(idx), _dev(vals)
        assert a.L.bam_array_update(a.h, 1, n, ctypes.c_void_p(d_idx.data_ptr()), ctypes.c_void_p(d_vals.data_ptr()), None, 64, None) == 0
        np.add.at(model, idx.astype(np.int64), vals)
        r.objs[0][2].flush()
        assert np.array_equal(r.backing(n_elems), model) and not r.c.aborted()


# through pointers from fewer requests on, the fewer the pages: on both sides of each line
@pytest.mark.parametrize("api,pages,n", [(1, 200, (1 << 14) - 1), (1, 74, 1 << 14), (1, 1000, 59999), (1, 1000, 60000), (1, 6000, (1 << 17) - 1), (2, 1000, 41231), (2, 1000, 41232),
                                         (2, 6000, (9 << 13) - 1), (2, 6000, 9 << 13), (2, 157, 1 << 14), (0, 100, (1 << 18) - 1)])
@pytest.mark.parametrize("kind", ["scattered", "in_order", "one_page"])
def test_updates_of_few_pages(bam, api, pages, n, kind):
    n_elems = pages * 512 - 3
    rng = np.random.default_rng(n)
    with Rig(bam, pages * 4096, backing=True, n_queues=16, depth=256) as r:
        model = r.backing(n_elems).copy()
        a = r.array(n_elems, 4096, pages)
        a.gather(pages, None, stride=512)
        a.update(0, _dev(np.zeros(1 << 18, dtype=np.uint64)), _dev(np.zeros(1 << 18, dtype=np.uint64)))      # leaves the memory for the bins behind
        idx = (rng.integers(0, n_elems, n) if kind == "scattered" else np.arange(n) % n_elems if kind == "in_order" else rng.integers(512, 1024, n)).astype(np.uint64)
        if api:                                               # no two at a time on an element
            idx = np.unique(idx) if kind != "scattered" else rng.permutation(n_elems)[:n].astype(np.uint64)
        vals = rng.integers(1, 1 << 63, len(idx)).astype(np.uint64)
        for rep in range(2):
            a.update(api, _dev(idx), _dev(vals))
            np.add.at(model, idx.astype(np.int64), vals)
        assert np.array_equal(_u64(a.gather(n_elems, None)), model) and not r.c.aborted()


# fewer than 2^17 and 73728 requests through pointers: both sides of where they meet often enough, up to 256 pages and beyond
@pytest.mark.parametrize("api,pages,n,bins", [(1, 256, 30357, False), (1, 256, 30358, True), (1, 512, 55425, False), (1, 512, 55426, True), (1, 2048, 110850, False), (1, 2048, 110852, True),
                                              (2, 256, 20861, False), (2, 256, 20862, True), (2, 257, 29560, False), (2, 512, 41722, False), (2, 512, 41723, True), (2, 1024, 59005, False), (2, 1024, 59006, True)])
def test_where_few_updates_take_bins(bam, api, pages, n, bins):
    """seen by the memory that a first call on each of 24 streams leaves for the next; below the line there is none"""
    import torch
    n_elems = pages * 512
    with Rig(bam, pages * 4096, backing=True, n_queues=8, depth=256) as r:
        model = r.backing(n_elems).copy()
        a = r.array(n_elems, 4096, pages)
        a.gather(pages, None, stride=512)
        idx = np.random.default_rng(n).permutation(n_elems)[:n].astype(np.uint64)
        d, v = _dev(idx), _dev(np.full(n, 3, dtype=np.uint64))
        streams = [torch.cuda.Stream() for _ in range(24)]
        old = torch.zeros(n, dtype=torch.int64, device="cuda")
        p = ctypes.c_void_p

        def calls(m):
            for s in streams:
                assert a.L.bam_array_update(a.h, api, m, p(d.data_ptr()), p(v.data_ptr()), p(old.data_ptr()), 64, p(s.cuda_stream)) == 0
                s.synchronize()

        calls(1000)                                           # what the kernels' own frames take is there
        free = torch.cuda.mem_get_info()[0]
        calls(n)
        taken = free - torch.cuda.mem_get_info()[0]
        assert taken >= 24 * 20 * n // 2 if bins else taken < 24 * 20 * n // 8, taken
        calls(n)
        want = model.copy()
        want[idx.astype(np.int64)] += np.uint64(2 * 24 * 3)
        want[idx[:1000].astype(np.int64)] += np.uint64(24 * 3)
        assert np.array_equal(_u64(a.gather(n_elems, None)), want) and not r.c.aborted()
