"""Scattered reads in several launches (bam_array_gather, bam_array_read): what is resident first, then the rest page by page."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _dev, _u64  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


# pages of data and of cache: everything resident; just below and at the smallest cache that is fetched for page by page, one
# stretch and several; requests around the sizes where the shape of the launch changes, and fewer than a request per two pages
@pytest.mark.parametrize("pages,cache_pages,n", [(4096, 4096, (1 << 20) + 1), (4100, 4095, 1 << 14), (4100, 4096, (1 << 14) - 1), (4100, 4096, (1 << 14) + 77),
                                                 (12289, 4096, 100003), (12289, 5000, (1 << 20) - 1), (40000, 4096, 19999), (40000, 4096, 20001)])
def test_scattered_reads_element_by_element(bam, pages, cache_pages, n):
    """Every element of a gather and the sum of the same requests, twice (the second call finds what the first left behind),
    with a few requests outside the array (they read as 0 and are not counted) and a skewed half; every request inside is
    counted once and misses cover the reads from the store."""
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
        for rep in range(2):
            assert np.array_equal(_u64(a.gather(n, d_idx)), want), rep
            st = a.stats()
            assert st["access_cnt"] == inside.sum() and st["hit_cnt"] + st["miss_cnt"] == st["access_cnt"], st
            assert st["read_io_cnt"] <= st["miss_cnt"] or rep == 0, st
            assert a.read(n, d_idx) == int(np.sum(want, dtype=np.uint64)), rep
            assert a.stats()["access_cnt"] == inside.sum()
        if cache_pages >= pages:
            a.stats()
            a.gather(n, d_idx)
            assert a.stats()["hit_cnt"] == inside.sum()
        assert not r.c.aborted() and r.c.info()["error_completions"] == 0


def test_gathers_on_several_streams_of_one_array(bam):
    """Six streams (more than the sets of notes an array keeps) gather from one array at once, each its own requests."""
    import torch
    pages, n = 9000, 60001
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
