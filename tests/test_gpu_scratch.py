"""What calls in several launches keep between them (bam_array_read, bam_array_gather, bam_reduce, bam_scan): graphs, streams, threads."""
import ctypes

import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _dev, _u64  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


def _read_into(a, n, d_idx, out, shape=0):
    import torch
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    idx, dst = ctypes.c_void_p(d_idx.data_ptr()), ctypes.c_void_p(out.data_ptr())
    if shape:
        assert a.L.bam_array_read_shaped(a.h, n, idx, shape, 8, 64, dst, st) == 0
    else:
        assert a.L.bam_array_read(a.h, n, idx, 0, 1, 64, dst, st) == 0


@pytest.mark.parametrize("shape", [0, 3])
@pytest.mark.parametrize("cache_pages", [4096, 4400])
def test_captured_reads_hold_nothing_of_the_array(bam, cache_pages, shape):
    """a read recorded into a graph and replayed after, and between, larger calls on the stream it was recorded on and on seven
    others; the array larger than its cache, and resident"""
    import torch
    pages, n = 4400, (1 << 16) + 77
    words = oracle.store(SEED, 0, pages * 512)
    rng = np.random.default_rng(3)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(pages * 512, 4096, cache_pages)
        reqs = rng.integers(0, pages * 512, 4 * n).astype(np.uint64)
        d, total = _dev(reqs), torch.zeros(1, dtype=torch.int64, device="cuda")
        other = torch.zeros(1, dtype=torch.int64, device="cuda")
        want = int(np.sum(words[reqs[:n].astype(np.int64)], dtype=np.uint64))
        want_all = int(np.sum(words[reqs.astype(np.int64)], dtype=np.uint64))
        a.read(n, d)
        torch.cuda.synchronize()
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=side):
            _read_into(a, n, d, total, shape)
        streams = [torch.cuda.Stream() for _ in range(7)] + [side]
        for rep in range(3):
            total.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert int(total.item()) & (2 ** 64 - 1) == want, rep
            for s in streams:
                with torch.cuda.stream(s):
                    other.zero_()
                    _read_into(a, 4 * n, d, other)
                torch.cuda.synchronize()
                assert int(other.item()) & (2 ** 64 - 1) == want_all, rep
        assert not r.c.aborted()


def test_two_threads_on_the_stream_of_each_thread(bam):
    """hipStreamPerThread is one handle and another stream in each thread: gathers, reductions and scans of two threads on one
    array larger than its cache, and on one that fits, each thread with requests of its own"""
    import threading
    import torch
    per_thread = ctypes.c_void_p(2)
    n = (1 << 20) + 5
    for pages, cache_pages in ((9000, 4096), (4096, 4096)):
        n_elems = pages * 512
        words = oracle.store(SEED, 0, n_elems)
        with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
            a = r.array(n_elems, 4096, cache_pages)
            reqs = [np.random.default_rng(k).integers(0, n_elems, n).astype(np.uint64) for k in range(2)]
            d = [_dev(x) for x in reqs]
            outs = [[torch.zeros(n, dtype=torch.int64, device="cuda") for _ in range(3)] for _ in range(2)]
            sums = [torch.zeros(n_elems // 128, dtype=torch.int64, device="cuda") for _ in range(2)]
            runs = [torch.zeros(n_elems + 2, dtype=torch.int64, device="cuda") for _ in range(2)]
            torch.cuda.synchronize()
            rcs, start = [[], []], threading.Barrier(2)

            def work(k):
                torch.cuda.set_device(0)
                start.wait()
                for o in outs[k]:
                    rcs[k].append(a.L.bam_array_gather(a.h, n, ctypes.c_void_p(d[k].data_ptr()), 0, 64, ctypes.c_void_p(o.data_ptr()), per_thread))
                rcs[k].append(a.L.bam_reduce(a.h, n_elems - k, 64, ctypes.c_void_p(sums[k].data_ptr()), per_thread))
                rcs[k].append(a.L.bam_scan(a.h, n_elems - k, 64, ctypes.c_void_p(runs[k].data_ptr()), per_thread))

            threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
            for t in threads:
                t.start()
            for t in threads:
                t.join()
            torch.cuda.synchronize()
            assert rcs == [[0] * 5] * 2
            for k in range(2):
                for o in outs[k]:
                    assert np.array_equal(_u64(o), words[reqs[k].astype(np.int64)]), (pages, k)
                assert np.array_equal(_u64(sums[k]), oracle.reduce_blocks(words[:n_elems - k], 64)), (pages, k)
                assert np.array_equal(_u64(runs[k])[:n_elems - k + 1], oracle.scan(words[:n_elems - k])), (pages, k)
            assert not r.c.aborted()


def test_many_streams_by_turns(bam):
    """reductions on seventy streams by turns, more than sets of scratch are kept for, with gathers that need none between them: a
    second round allocates nothing, and every result is right"""
    import torch
    pages = 4400
    n_elems = pages * 512
    words = oracle.store(SEED, 0, n_elems)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(n_elems, 4096, pages)
        d = [_dev(np.random.default_rng(k).integers(0, n_elems, (1 << 20) + k).astype(np.uint64)) for k in range(8)]
        torch.cuda.synchronize()
        made = (ctypes.c_void_p * 70)()
        hip = ctypes.CDLL("libamdhip64.so.7")
        for k in range(70):
            assert hip.hipStreamCreateWithFlags(ctypes.byref(made, 8 * k), 1) == 0
        sums = torch.zeros((70, n_elems // 128), dtype=torch.int64, device="cuda")
        outs = [torch.zeros(x.numel(), dtype=torch.int64, device="cuda") for x in d]
        torch.cuda.synchronize()
        for rep in range(2):
            for k in range(70):
                st = ctypes.c_void_p(made[k])
                assert a.L.bam_array_gather(a.h, d[k % 8].numel(), ctypes.c_void_p(d[k % 8].data_ptr()), 0, 64, ctypes.c_void_p(outs[k % 8].data_ptr()), st) == 0
                assert a.L.bam_reduce(a.h, n_elems, 64, ctypes.c_void_p(sums[k].data_ptr()), st) == 0
            if rep == 0:
                torch.cuda.synchronize()
                free = torch.cuda.mem_get_info()[0]
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] == free
        want = oracle.reduce_blocks(words, 64)
        assert np.array_equal(_u64(sums), np.broadcast_to(want, (70, len(want))))
        for x, o in zip(d, outs):
            assert np.array_equal(_u64(o), words[x.cpu().numpy()])
        for k in range(70):
            assert hip.hipStreamDestroy(ctypes.c_void_p(made[k])) == 0
        assert not r.c.aborted()


@pytest.mark.parametrize("same", [False, True])
def test_scans_of_two_threads_side_by_side(bam, same):
    """two streams, many large scans each of resident elements: tiles that wait for tiles, of one array and of two"""
    import threading
    import torch
    sizes = [(1 << 24) + 5, (1 << 24) - 16384 if same else (1 << 23) + 16384]
    with Rig(bam, sum(-(-n // 512) for n in sizes) * 4096, n_queues=16, depth=256) as r:
        first = r.array(sizes[0], 4096, -(-sizes[0] // 512))
        arrs = [first, first if same else r.array(sizes[1], 4096, -(-sizes[1] // 512), -(-sizes[0] // 512) * 4096)]
        want = []
        for a, n in zip(arrs, sizes):
            x = a.gather(n, None, stride=1)
            want.append(torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), torch.cumsum(x, 0)]))
        streams = [torch.cuda.Stream() for _ in range(2)]
        outs = [torch.empty(w.numel() + 1, dtype=torch.int64, device="cuda") for w in want]
        torch.cuda.synchronize()
        bad, start = [[], []], threading.Barrier(2)

        def work(k):
            torch.cuda.set_device(0)
            with torch.cuda.stream(streams[k]):
                start.wait()
                for rep in range(25):
                    outs[k].zero_()
                    rc = arrs[k].L.bam_scan(arrs[k].h, sizes[k], 256, ctypes.c_void_p(outs[k].data_ptr()), ctypes.c_void_p(streams[k].cuda_stream))
                    if rc or not torch.equal(outs[k][:-1], want[k]):
                        bad[k].append(rep)

        threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert bad == [[], []] and not r.c.aborted()


@pytest.mark.parametrize("cold", [False, True])
def test_captured_sums_of_arrays_read_by_pages(bam, cold):
    """vectoradd and a reduction recorded into a graph after calls that take whole pages (or as the first calls at all), and replayed with other
    elements and eager work between the replays"""
    import torch
    n, pages = 200_003, 391
    with Rig(bam, 3 * pages * 4096, backing=True, n_queues=16, depth=256) as r:
        pc = bam.PageCache(4096, 3 * pages + 30, 0, r.c)
        rs = [bam.Range(0, n, k * pages, pages, 0, 4096, pc, 0) for k in range(3)]
        a, b, c = arrs = [bam.Array(n, k * pages * 4096, [rs[k]], 0) for k in range(3)]
        words = oracle.store(SEED, 0, 3 * pages * 512)
        r.backing(len(words))[:] = words
        x, y = words[:n].copy(), words[pages * 512:pages * 512 + n]
        partials = torch.zeros(n // 128 + 1, dtype=torch.int64, device="cuda")
        if not cold:
            bam.vectoradd(a, b, c, n)
            a.reduce(n, block_size=64)
            torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            bam.vectoradd(a, b, c, n)
            st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            assert a.L.bam_reduce(a.h, n, 64, ctypes.c_void_p(partials.data_ptr()), st) == 0
        for rep in range(4):
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(_u64(c.gather(n, None, stride=1)), x + y), rep
            assert np.array_equal(_u64(partials), oracle.reduce_blocks(x, 64)), rep
            idx = np.random.default_rng(rep).permutation(n)[:4096].astype(np.uint64)
            a.update(0, _dev(idx), _dev(idx + np.uint64(7)))
            x[idx.astype(np.int64)] += idx + np.uint64(7)
            if rep == 1:
                bam.vectoradd(a, b, c, n)
                assert np.array_equal(_u64(a.reduce(n, block_size=256)), oracle.reduce_blocks(x, 256))
        assert not r.c.aborted()
        for z in arrs + rs:
            z.close()
        pc.close()


def test_sums_beyond_the_sets_of_scratch(bam):
    """vectoradd on seventy streams by turns: those that get no set of scratch go element by element"""
    import torch
    n, pages = 20_003, 40
    hip = ctypes.CDLL("libamdhip64.so.7")
    with Rig(bam, 3 * pages * 4096, backing=True, n_queues=16, depth=256) as r:
        pc = bam.PageCache(4096, 3 * pages + 30, 0, r.c)
        rs = [bam.Range(0, n, k * pages, pages, 0, 4096, pc, 0) for k in range(3)]
        arrs = [bam.Array(n, k * pages * 4096, [rs[k]], 0) for k in range(3)]
        words = oracle.store(SEED, 0, 3 * pages * 512)
        r.backing(len(words))[:] = words
        want = words[:n] + words[pages * 512:pages * 512 + n]
        made = (ctypes.c_void_p * 70)()
        for k in range(70):
            assert hip.hipStreamCreateWithFlags(ctypes.byref(made, 8 * k), 1) == 0
        for k in range(70):
            arrs[2].update(0, _dev(np.arange(n, dtype=np.uint64)), _dev(np.ones(n, dtype=np.uint64)))      # not what the sums are
            torch.cuda.synchronize()
            assert arrs[0].L.bam_vectoradd(*[z.h for z in arrs], n, ctypes.c_void_p(made[k])) == 0
            torch.cuda.synchronize()
            if k in (0, 1, 63, 64, 69):
                assert np.array_equal(_u64(arrs[2].gather(n, None, stride=1)), want), k
        for k in range(70):
            assert hip.hipStreamDestroy(ctypes.c_void_p(made[k])) == 0
        assert not r.c.aborted()
        for z in arrs + rs:
            z.close()
        pc.close()
