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
