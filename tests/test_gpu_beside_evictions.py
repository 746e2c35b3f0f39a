"""Readings along whole pages and updates in bins while gathers on another stream, from another array of the same cache, push their pages out."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import SEED, Rig, _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu

OTHER = 4096           # pages of the other array


class Shared:
    """arrays of `sizes` elements and another one, behind one cache, one after the other on the store"""

    def __init__(self, bam, sizes, cache_pages):
        pages = [(n + 511) // 512 for n in sizes] + [OTHER]
        self.firsts = np.cumsum([0] + pages).tolist()
        self.r = Rig(bam, self.firsts[-1] * 4096, backing=True, n_queues=16, depth=256)
        self.store = self.r.backing(self.firsts[-1] * 512)
        self.store[:] = oracle.store(SEED, 0, len(self.store))
        self.pc = bam.PageCache(4096, cache_pages, 0, self.r.c)
        sizes = list(sizes) + [OTHER * 512]
        self.rs = [bam.Range(0, n, f, p, 0, 4096, self.pc, 0) for n, f, p in zip(sizes, self.firsts, pages)]
        self.arrs = [bam.Array(n, f * 4096, [x], 0) for n, f, x in zip(sizes, self.firsts, self.rs)]
        self.d_idx = _dev(np.random.default_rng(3).integers(0, OTHER * 512, 4096).astype(np.uint64))
        self.want = self.store[self.firsts[-2] * 512:][_u64(self.d_idx).astype(np.int64)].copy()

    def of(self, k, n):
        return self.store[self.firsts[k] * 512:][:n]

    def beside(self, call):
        """call() with three gathers on their way on another stream"""
        import torch
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            outs = [self.arrs[-1].gather(4096, self.d_idx) for _ in range(3)]
        got = call()
        torch.cuda.synchronize()
        for o in outs:
            assert np.array_equal(_u64(o), self.want)
        assert not self.r.c.aborted()
        return got

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for x in self.arrs + self.rs:
            x.close()
        self.pc.close()
        self.r.close()


@pytest.mark.parametrize("cache_pages", [300, 700])
def test_levels_and_labels(bam, cache_pages):
    off, nb = oracle.uniform_csr(SEED, 20011, 150007)
    src = int(oracle.bfs_sources(SEED, off, 1)[0])
    levels, n_levels = oracle.bfs_levels(off, nb, src)
    labels, _ = oracle.cc_labels(off, nb)
    with Shared(bam, [len(nb)], cache_pages) as s:
        s.of(0, len(nb))[:] = nb
        d_off = _dev(off)
        s.arrs[0].set_graph(d_off)
        for rep in range(6):
            lv, it = s.beside(lambda: s.arrs[0].bfs(d_off, src, by_page=bool(rep & 1)))
            assert np.array_equal(lv.cpu().numpy().view(np.uint32), levels) and it == n_levels, rep
            lb, _ = s.beside(lambda: s.arrs[0].cc(d_off))
            assert np.array_equal(_u64(lb), labels), rep


@pytest.mark.parametrize("cache_pages", [500, 1100])
def test_sums(bam, cache_pages):
    n = 300 * 512 + 77
    with Shared(bam, [n, n, n], cache_pages) as s:
        a, b, c = s.arrs[:3]
        want = s.of(0, n) + s.of(1, n)
        keep = s.of(0, n).copy(), s.of(1, n).copy()
        for rep in range(6):
            s.of(2, n)[:] = 0
            s.beside(lambda: bam.vectoradd(a, b, c, n))
            assert np.array_equal(_u64(c.gather(n, None, stride=1)), want), rep
            s.pc.flush()
            assert np.array_equal(s.of(2, n), want), rep
        assert np.array_equal(s.of(0, n), keep[0]) and np.array_equal(s.of(1, n), keep[1])


@pytest.mark.parametrize("api", [0, 1, 2])
def test_updates_in_bins(bam, api):
    n, n_elems = (1 << 18) + 321, 600 * 512 - 5
    rng = np.random.default_rng(api)
    with Shared(bam, [n_elems], 620) as s:
        a = s.arrs[0]
        model = s.of(0, n_elems).copy()
        missed = 0
        for rep in range(6):
            idx = rng.permutation(n_elems)[:n].astype(np.uint64)
            vals = rng.integers(1, 1 << 63, n).astype(np.uint64)
            d_idx, d_vals = _dev(idx), _dev(vals)
            a.gather(600, None, stride=512)
            a.stats()
            old = s.beside(lambda: a.update(api, d_idx, d_vals, block_size=256))
            assert np.array_equal(_u64(old), model[idx.astype(np.int64)]), rep
            model[idx.astype(np.int64)] += vals
            st = a.stats()
            missed += st["miss_cnt"]
            assert st["access_cnt"] == n, st
        s.pc.flush()
        assert missed > 0 and np.array_equal(s.of(0, n_elems), model)
