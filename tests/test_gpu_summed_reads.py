"""Sums of scattered reads in one launch: workgroups that add to the sum themselves, and shards that are folded."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _dev  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


# a lane to several workgroups, the last workgroup that adds by itself and the first that does not, the largest in one launch and one more;
# the array in the cache, cold and resident, and (few requests, spread) twice as large
@pytest.mark.parametrize("n", [1, 65, 511, 513, 128 * 512, 128 * 512 + 1, (1 << 20), (1 << 20) + 1])
@pytest.mark.parametrize("page,pages,cache_pages", [(4096, 700, 700), (512, 4001, 4001), (8192, 300, 310), (4096, 70000, 35000)])
def test_sums_and_counters(bam, n, page, pages, cache_pages):
    n_elems = pages * page // 8 - 3
    words = oracle.store(SEED, 0, n_elems)
    idx = np.random.default_rng(n).integers(0, n_elems, n).astype(np.uint64)
    idx[n // 2] = n_elems                                  # reads as 0 and is not counted
    want = int(np.sum(words[idx[idx < n_elems].astype(np.int64)], dtype=np.uint64))
    with Rig(bam, (pages * page + 65535) // 65536 * 65536, n_queues=16, depth=256) as r:
        a = r.array(n_elems, page, cache_pages)
        d = _dev(idx)
        for rep in range(3):
            assert a.read(n, d, block_size=64 << rep) == want, rep
            st = a.stats()
            assert st["access_cnt"] == n - 1 and st["hit_cnt"] + st["miss_cnt"] == n - 1, st
        assert not r.c.aborted()


def test_sums_are_added_to(bam):
    """bam_array_read adds to what the word holds, in either way"""
    import torch
    with Rig(bam, 256 * 4096, n_queues=4, depth=256) as r:
        a = r.array(256 * 512, 4096, 256)
        words = oracle.store(SEED, 0, 256 * 512)
        s = torch.tensor([5], dtype=torch.int64, device="cuda")
        want = 5
        for n in (100, 200000):
            idx = np.random.default_rng(n).integers(0, 256 * 512, n).astype(np.uint64)
            a.read_async(n, s, _dev(idx))
            torch.cuda.synchronize()
            want = (want + int(np.sum(words[idx.astype(np.int64)], dtype=np.uint64))) & ((1 << 64) - 1)
        assert int(s.item()) & ((1 << 64) - 1) == want and not r.c.aborted()


@pytest.mark.parametrize("n,pages,cache_pages", [(200001, 900, 900), (65000, 900, 900), (65000, 70000, 35000)])
def test_sums_on_several_streams(bam, n, pages, cache_pages):
    """each stream folds its own shards"""
    import torch
    n_elems = pages * 512
    words = oracle.store(SEED, 0, n_elems)
    rng = np.random.default_rng(8)
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(n_elems, 4096, cache_pages)
        reqs = [rng.integers(0, n_elems, n).astype(np.uint64) for _ in range(6)]
        d = [_dev(x) for x in reqs]
        sums = torch.zeros(6, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream() for _ in d]
        for rep in range(8):
            for k, s in enumerate(streams):
                with torch.cuda.stream(s):
                    a.read_async(n, sums[k:k + 1], d[k])
        torch.cuda.synchronize()
        got = sums.cpu().numpy().view(np.uint64)
        for k, x in enumerate(reqs):
            want = int(np.sum(words[x.astype(np.int64)], dtype=np.uint64)) * 8 & ((1 << 64) - 1)
            assert int(got[k]) == want, k
        assert not r.c.aborted()


@pytest.mark.parametrize("n", [1000, 65000, 100001, 300000])
@pytest.mark.parametrize("pages,cache_pages", [(900, 900), (900, 300)])
def test_captured_reads(bam, n, pages, cache_pages):
    """recorded in a graph and replayed beside calls outside it"""
    import torch
    n_elems = pages * 512
    words = oracle.store(SEED, 0, n_elems)
    idx = np.random.default_rng(n).integers(0, n_elems, n).astype(np.uint64)
    want = int(np.sum(words[idx.astype(np.int64)], dtype=np.uint64))
    with Rig(bam, pages * 4096, n_queues=16, depth=256) as r:
        a = r.array(n_elems, 4096, cache_pages)
        d = _dev(idx)
        assert a.read(n, d) == want
        s = torch.zeros(1, dtype=torch.int64, device="cuda")
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            a.read_async(n, s, d)
            out = a.gather(n, d)
        for rep in range(4):
            s.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert int(s.item()) & ((1 << 64) - 1) == want, rep
            assert np.array_equal(out.cpu().numpy().view(np.uint64), words[idx.astype(np.int64)]), rep
            assert a.read(n, d) == want
        assert not r.c.aborted()
