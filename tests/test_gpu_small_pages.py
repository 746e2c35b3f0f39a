"""BFS and components along pages of less than a segment of 512 entries: a page alone, pages of one segment of which some are
resident, arrays that end inside a row, a page and a segment, lists that cross all of them, caches from two pages on."""
import numpy as np
import pytest

import oracle
from test_gpu_along_pages import KINDS, _check_bfs, _rig
from test_gpu_parity import SEED, _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_edges", [1, 63, 64, 65, 127, 129, 255, 257, 511, 513, 4095, 4097, 33333])
@pytest.mark.parametrize("page,cache_pages", [(512, 2), (512, 70), (512, 600), (1024, 3), (1024, 300), (2048, 5), (2048, 200)])
def test_levels_and_labels_of_directed_lists_of_all_lengths(bam, n_edges, page, cache_pages):
    rng = np.random.default_rng(n_edges + page + cache_pages)
    deg = []
    while sum(deg) < n_edges:
        deg.append(0 if rng.random() < 0.3 else int(rng.integers(1, 700 if n_edges > 9000 else 40)))
    deg = np.array([0, 0] + deg + [0])
    deg[np.nonzero(deg)[0][-1]] -= deg.sum() - n_edges
    n_v = len(deg)
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    owner = np.repeat(np.arange(n_v), deg)
    nb = ((owner + rng.integers(-3, 8, n_edges)) % n_v).astype(np.uint64)
    r, a = _rig(bam, nb, page, cache_pages)
    with r:
        _check_bfs(r, a, off, nb, [0, int(np.nonzero(deg)[0][0]), int(rng.integers(0, n_v))])


@pytest.mark.parametrize("before,behind", [(0, 0), (3, 70), (64, 0), (700, 1300)])
@pytest.mark.parametrize("page,share", [(512, 1), (512, 2), (512, 5), (1024, 1), (1024, 3), (2048, 1), (2048, 4)])
def test_labels_and_levels_of_random_graphs(bam, page, share, before, behind):
    """(the array may be longer than the lists, which then begin inside a page)"""
    for off, nb in (oracle.rmat_csr(SEED, 13), oracle.uniform_csr(SEED, 30011, 50021)):
        want, _ = oracle.cc_labels(off, nb)
        src = int(oracle.bfs_sources(SEED, off, 1)[0])
        levels, n_levels = oracle.bfs_levels(off, nb, src)
        nb = np.concatenate([np.full(before, 1, dtype=np.uint64), nb, np.full(behind, 0, dtype=np.uint64)])
        d_off = _dev(off + np.uint64(before))
        r, a = _rig(bam, nb, page, max(2, (len(nb) * 8 // page + 1) // share))
        with r:
            for kept in (False, True, True):
                if kept:
                    a.set_graph(d_off)
                for kw in KINDS:
                    lv, it = a.bfs(d_off, src, **kw)
                    assert np.array_equal(lv.cpu().numpy().view(np.uint32), levels) and it == n_levels, (kept, kw)
                for by_page in (False, True):
                    lb, _ = a.cc(d_off, by_page=by_page)
                    assert np.array_equal(_u64(lb), want), (kept, by_page)
            assert not r.c.aborted()


@pytest.mark.parametrize("page,share", [(512, 1), (512, 3), (2048, 2)])
def test_long_runs_of_vertices_without_lists(bam, page, share):
    """owners looked up by bisection: 40000 vertices without a list between two thirds of a random graph"""
    n, run = 4001, 40000
    off, nb = oracle.uniform_csr(SEED, n, 24007)
    place = np.arange(n, dtype=np.int64)
    place[n // 3:] += run
    n_v = int(place[-1]) + 1 + run
    deg = np.zeros(n_v, dtype=np.uint64)
    deg[place] = off[1:] - off[:-1]
    src = int(oracle.bfs_sources(SEED, off, 1)[0])
    lv_some, want_it = oracle.bfs_levels(off, nb, src)
    want = np.full(n_v, 0xFFFFFFFF, dtype=np.uint32)
    want[place] = lv_some
    comp, _ = oracle.cc_labels(off, nb)
    labels = np.arange(n_v, dtype=np.uint64)
    labels[place] = place[comp.astype(np.int64)].astype(np.uint64)
    off, nb = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64), place[nb.astype(np.int64)].astype(np.uint64)
    r, a = _rig(bam, nb, page, max(2, len(nb) * 8 // page // share + 1))
    with r:
        d_off = _dev(off)
        a.set_graph(d_off)
        for kw in KINDS:
            lv, it = a.bfs(d_off, int(place[src]), **kw)
            assert np.array_equal(lv.cpu().numpy().view(np.uint32), want) and it == want_it, kw
        for by_page in (False, True):
            lb, _ = a.cc(d_off, by_page=by_page)
            assert np.array_equal(_u64(lb), labels), by_page
        assert not r.c.aborted()
