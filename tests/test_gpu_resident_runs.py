"""bam_reduce and bam_scan over elements that are resident: one pass without references, and what happens when a page is missing."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _u64  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


def _accesses(n, half, page_elems):
    """one access per thread and page it reads on: elements t and t + half of every 2 half"""
    e = np.arange(n, dtype=np.int64)
    e = e[(e // half) % 2 == 0]
    e2 = e + half
    return len(e) + int(((e2 < n) & (e // page_elems != e2 // page_elems)).sum())


# around a row (128), a wave (1024), a tile of a scan (16384), 64 of them, a page and an output; page sizes on both sides of a row
@pytest.mark.parametrize("page", [512, 4096, 8192, 65536])
@pytest.mark.parametrize("n,block", [(1, 64), (127, 64), (128, 64), (129, 192), (1023, 128), (1024, 512), (2047, 256), (2048, 256), (2049, 1024),
                                     (65537, 64), (65537, 320), (300001, 576), (300001, 960), ((1 << 22) - 1, 256), (1 << 22, 64), ((1 << 22) + 8193, 1024),
                                     (16383, 64), (16384, 64), (16385, 128), (64 * 16384 - 1, 64), (64 * 16384, 256), (65 * 16384, 256), (65 * 16384 + 1, 512)])
def test_resident_runs_element_by_element(bam, page, n, block):
    per = page // 8
    pages = (n + per - 1) // per
    vals = oracle.store(SEED, 0, n)
    with Rig(bam, (pages * page + 65535) // 65536 * 65536, n_queues=8, depth=256) as r:
        a = r.array(n, page, pages)
        want_sums, want_runs = oracle.reduce_blocks(vals, block), oracle.scan(vals)
        for rep in range(3):                    # the first scan and the first reduction after it find pages missing, the others none
            assert np.array_equal(_u64(a.scan(n, block)), want_runs), rep
            if rep:
                assert a.stats()["access_cnt"] == _accesses(n, block, per)
            assert np.array_equal(_u64(a.reduce(n, block)), want_sums), rep
            st = a.stats()
            assert rep == 0 or (st["access_cnt"] == st["hit_cnt"] == _accesses(n, block, per) and st["read_io_cnt"] == 0), st
        assert not r.c.aborted()


@pytest.mark.parametrize("first_missing", [0, 1, 77, 255])
def test_runs_with_some_pages_missing(bam, first_missing):
    """only the pages from `first_missing` on are absent when the reduction, and then the scan, begins"""
    n, pages = 257 * 512 - 3, 257
    vals = oracle.store(SEED, 0, n)
    for op in ("reduce", "scan"):
        with Rig(bam, pages * 4096, n_queues=8, depth=256) as r:
            a = r.array(n, 4096, pages)
            if first_missing:
                a.gather(first_missing, None, stride=512)
            a.stats()
            if op == "reduce":
                assert np.array_equal(_u64(a.reduce(n, 128)), oracle.reduce_blocks(vals, 128))
            else:
                assert np.array_equal(_u64(a.scan(n, 128)), oracle.scan(vals))
            st = a.stats()
            assert st["access_cnt"] == _accesses(n, 128, 512) and st["read_io_cnt"] == pages - first_missing, st
            assert not r.c.aborted()


def test_runs_on_several_streams_and_results_at_odd_addresses(bam):
    """scans and reductions of one array queued on three streams by turns, and a scan whose result starts 8 bytes past a multiple of 16"""
    import ctypes
    import torch
    n = 300001
    vals = oracle.store(SEED, 0, n)
    with Rig(bam, 600 * 4096, n_queues=8, depth=256) as r:
        a = r.array(n, 4096, 600)
        a.reduce(n, 64)
        torch.cuda.synchronize()
        outs = []
        for k, s in enumerate([torch.cuda.Stream() for _ in range(3)] * 2):
            with torch.cuda.stream(s):
                outs.append((a.scan(n - k, 64 * (k + 1)), a.reduce(n - k, 64 * (k + 1))))
        torch.cuda.synchronize()
        for k, (runs, sums) in enumerate(outs):
            assert np.array_equal(_u64(runs), oracle.scan(vals[:n - k])) and np.array_equal(_u64(sums), oracle.reduce_blocks(vals[:n - k], 64 * (k + 1)))
        out = torch.zeros(n + 2, dtype=torch.int64, device="cuda")
        assert a.L.bam_scan(a.h, n, 256, ctypes.c_void_p(out.data_ptr() + 8), None) == 0
        torch.cuda.synchronize()
        assert np.array_equal(_u64(out[1:]), oracle.scan(vals)) and not r.c.aborted()


def test_scans_while_another_array_evicts(bam):
    """pages leave before, between and during the launches of a scan: another array of the same cache is gathered from on a second
    stream, a different while after the scan is queued each time.  Every scan is right, and counts what it reads once, whichever
    kernels end up doing it"""
    import torch
    from bam_amd import Array, PageCache, Range
    pages, other = 65536, 65536
    n, n_b = pages * 512 - 3, other * 512
    n_access = _accesses(n, 64, 512)
    with Rig(bam, (pages + other) * 4096, n_queues=16, depth=256) as r:
        pc = PageCache(4096, pages + 8192, 0, r.c)
        ra, rb = Range(0, n, 0, pages, 0, 4096, pc, 0), Range(0, n_b, pages, other, 0, 4096, pc, 0)
        a, b = Array(n, 0, [ra], 0), Array(n_b, pages * 4096, [rb], 0)
        want = torch.from_numpy(oracle.scan(oracle.store(SEED, 0, n)).view(np.int64)).cuda()
        side = torch.cuda.Stream()
        ids = [torch.arange(64, dtype=torch.int64, device="cuda") * 512 + k * 32768 for k in range(other // 64)]
        for k in range(128):                        # the slots lie by turns, so that a page that comes back soon pushes out one of the other array
            a.gather(512, torch.arange(512, dtype=torch.int64, device="cuda") * 512 + k * 262144)
            b.gather(64, ids[k])
        torch.cuda.synchronize()
        began, ended = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        began.record()
        torch.cuda._sleep(1 << 20)
        ended.record()
        torch.cuda.synchronize()
        per_us = (1 << 20) / (began.elapsed_time(ended) * 1e3)
        for rep in range(80):
            for _ in range(50):                     # until all of it is resident (what comes back pushes others out, for a while)
                a.stats()
                a.reduce(n, 256)
                if not a.stats()["read_io_cnt"]:
                    break
            with torch.cuda.stream(side):
                torch.cuda._sleep(int(per_us * 5 * rep))
                b.gather(64, ids[(128 + rep) % len(ids)])
            assert torch.equal(a.scan(n, 64), want), rep
            st = a.stats()
            assert st["access_cnt"] == n_access, (rep, st)
        assert not r.c.aborted()
        a.close(); b.close(); ra.close(); rb.close(); pc.close()
