"""vectoradd a page at a time: sizes around a page, a wave's pages and a batch; caches that hold all three arrays, half and little
of them; arrays that are the same; queues shallower than a batch; commands that fail; C cached and changed beforehand."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import SEED, Rig, _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


class Three:
    def __init__(self, bam, r, n, page, cache_pages):
        per = page // 8
        self.pages = (n + per - 1) // per
        self.store = r.backing(3 * self.pages * per)
        self.at = [slice(k * self.pages * per, k * self.pages * per + n) for k in range(3)]
        self.store[:] = oracle.store(SEED, 0, 3 * self.pages * per)
        self.pc = bam.PageCache(page, cache_pages, 0, r.c)
        self.rs = [bam.Range(0, n, k * self.pages, self.pages, 0, page, self.pc, 0) for k in range(3)]
        self.arrs = [bam.Array(n, k * self.pages * page, [self.rs[k]], 0) for k in range(3)]

    def close(self):
        for x in self.arrs + self.rs:
            x.close()
        self.pc.close()


def _rig(bam, n, page, **kw):
    pages = (n * 8 + page - 1) // page
    return Rig(bam, 3 * pages * page, backing=True, n_queues=kw.pop("n_queues", 8), depth=kw.pop("depth", 256), stage_bytes=max(4096, page), **kw)


@pytest.mark.parametrize("n", [511, 512, 513, 1024, 15 * 512, 16 * 512 + 1, 32 * 512 - 1, 32 * 512, 33 * 512, 100 * 512 + 77, 300_003])
@pytest.mark.parametrize("page,share,depth", [(4096, 1, 256), (4096, 2, 256), (4096, 5, 256), (4096, 2, 4), (8192, 2, 256)])
def test_sums_reach_the_store(bam, n, page, share, depth):
    pages = (n * 8 + page - 1) // page
    with _rig(bam, n, page, depth=depth) as r:
        t = Three(bam, r, n, page, max(40, 3 * pages // share + 4))
        a, b, c = t.arrs
        want = t.store[t.at[0]] + t.store[t.at[1]]
        keep = t.store.copy()
        for rep in range(3):                               # cold, then with what the call before left
            t.store[t.at[2]] = 0
            for x in t.arrs:
                x.stats()
            bam.host.vectoradd(a, b, c, n)
            t.pc.flush()
            assert np.array_equal(t.store[t.at[2]], want), rep
            assert all(x.stats()["access_cnt"] == n for x in t.arrs)
            assert np.array_equal(_u64(c.gather(n, None, stride=1)), want), rep
        assert np.array_equal(t.store[t.at[0]], keep[t.at[0]]) and np.array_equal(t.store[t.at[1]], keep[t.at[1]])
        assert np.array_equal(t.store[n:t.pages * page // 8], keep[n:t.pages * page // 8])         # behind the last element
        assert not r.c.aborted()
        t.close()


@pytest.mark.parametrize("share", [1, 2])
@pytest.mark.parametrize("which", ["aab", "aba", "baa", "aaa"])
def test_arrays_that_are_the_same(bam, which, share):
    n, page = 64 * 512 + 5, 4096
    with _rig(bam, n, page) as r:
        t = Three(bam, r, n, page, 200 // share)
        first = {"a": t.store[t.at[0]].copy(), "b": t.store[t.at[1]].copy()}
        x, y, z = (t.arrs["ab".index(k)] for k in which)
        want = dict(first)
        for rep in range(3):
            bam.host.vectoradd(x, y, z, n)
            want[which[2]] = want[which[0]] + want[which[1]]
            t.pc.flush()
            for k, arr in (("a", t.arrs[0]), ("b", t.arrs[1])):
                assert np.array_equal(_u64(arr.gather(n, None, stride=1)), want[k]), (rep, k)
                assert np.array_equal(t.store[t.at["ab".index(k)]], want[k]), (rep, k)
        assert not r.c.aborted()
        t.close()


def test_results_where_c_was_cached_and_changed(bam):
    """half of C's pages are in the cache, changed and not yet written back"""
    n, page = 96 * 512, 4096
    with _rig(bam, n, page) as r:
        t = Three(bam, r, n, page, 120)
        a, b, c = t.arrs
        want = t.store[t.at[0]] + t.store[t.at[1]]
        c.write(n // 2, _dev(np.full(n // 2, 7, dtype=np.uint64)))
        bam.host.vectoradd(a, b, c, n)
        assert np.array_equal(_u64(c.gather(n, None, stride=1)), want)
        t.pc.flush()
        assert np.array_equal(t.store[t.at[2]], want) and not r.c.aborted()
        t.close()


def test_results_where_commands_fail(bam):
    """every eleventh command: pages whose write failed are added up in the cache (which keeps them: A and B leave before them)"""
    n, page = 128 * 512, 4096
    with _rig(bam, n, page, fail_every=11) as r:
        t = Three(bam, r, n, page, 300)
        a, b, c = t.arrs
        want = t.store[t.at[0]] + t.store[t.at[1]]
        bam.host.vectoradd(a, b, c, n)
        assert np.array_equal(_u64(c.gather(n, None, stride=1)), want)
        assert r.t.stats()["error_cpls"] > 0 and not r.c.aborted()
        t.close()
