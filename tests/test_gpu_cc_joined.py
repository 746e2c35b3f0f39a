"""Components from one reading of the edges: shapes whose trees are long, wide, or not there at all."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import _dev, _graph_rig, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


def _csr(n_v, u, v):
    """both directions of every pair, ordered by vertex"""
    src, dst = np.concatenate([u, v]), np.concatenate([v, u])
    order = np.argsort(src, kind="stable")
    off = np.zeros(n_v + 1, dtype=np.uint64)
    off[1:] = np.cumsum(np.bincount(src, minlength=n_v))
    return off, dst[order].astype(np.uint64)


def _pairs(shape, n_v, rng):
    at = np.arange(n_v, dtype=np.int64)
    if shape == "path":                                   # every vertex hooks onto the one before it
        return at[:-1], at[1:]
    if shape == "scattered_path":
        p = rng.permutation(n_v)
        return p[:-1], p[1:]
    if shape == "star":                                   # one list in pieces, every join on the same root, which is the largest vertex
        return np.full(n_v - 1, n_v - 1, dtype=np.int64), at[:-1]
    if shape == "loops_and_copies":                       # each vertex to itself, and pairs of neighbours three times over
        even = at[: n_v // 2 * 2 : 2]
        return np.concatenate([at, even, even, even]), np.concatenate([at, even + 1, even + 1, even + 1])
    return at[:1], at[-1:]                                # one edge between the ends, all other vertices by themselves


@pytest.mark.parametrize("by_page", [False, True])
@pytest.mark.parametrize("shape", ["path", "scattered_path", "star", "loops_and_copies", "ends"])
@pytest.mark.parametrize("n_v", [2, 65, 512, 513, 100003])
def test_cc_labels_of_long_wide_and_empty_trees(bam, n_v, shape, by_page):
    off, nb = _csr(n_v, *_pairs(shape, n_v, np.random.default_rng(n_v)))
    ref, _ = oracle.cc_labels(off, nb)
    r, a = _graph_rig(bam, nb, 256, n_queues=16, depth=256)
    with r:
        d_off = _dev(off)
        pages = (len(nb) + 511) // 512
        a.stats()
        for kept in (False, True, True):                  # without a plan, then with one: from the front and from the back
            if kept:
                a.set_graph(d_off)
            lb, it = a.cc(d_off, by_page=by_page)
            assert np.array_equal(_u64(lb), ref), kept
            st = a.stats()
            if pages <= 256:
                assert st["read_io_cnt"] == (0 if kept else pages), (kept, st)
            else:                                         # one reading of the edges; a page that two lists share may leave in between
                assert it == 2 and st["read_io_cnt"] <= (pages if by_page else 5 * pages // 4), (kept, st, pages)
        assert not r.c.aborted()


# all edges cached, around the numbers of entries between which labels are propagated along the pages (2^17, 2^22): a wide graph,
# which a few sweeps settle, and paths, which they do not
@pytest.mark.parametrize("shape", ["wide", "path", "scattered_path", "star"])
@pytest.mark.parametrize("n_pairs", [(1 << 16) - 1, 1 << 16, (1 << 16) + 1, 300001, (1 << 21) - 1, 1 << 21])
def test_cc_labels_where_all_edges_are_cached(bam, n_pairs, shape):
    rng = np.random.default_rng(n_pairs)
    n_v = n_pairs // 4 if shape == "wide" else n_pairs + 1
    u, v = (rng.integers(0, n_v, n_pairs), rng.integers(0, n_v, n_pairs)) if shape == "wide" else _pairs(shape, n_v, rng)
    off, nb = _csr(n_v, u, v)
    ref, _ = oracle.cc_labels(off, nb)
    pages = (len(nb) + 511) // 512
    sweeps = 1 << 17 < len(nb) < 1 << 22
    r, a = _graph_rig(bam, nb, max(128, pages), n_queues=16, depth=256)
    with r:
        d_off = _dev(off)
        for kept in (False, True, True):
            if kept:
                a.set_graph(d_off)
            for by_page in (True, False):
                lb, it = a.cc(d_off, by_page=by_page)
                assert np.array_equal(_u64(lb), ref), (kept, by_page)
                # joined: a pass over the edges and one over the vertices; propagated: until a sweep changes nothing, six at most
                assert it == 2 if not (by_page and sweeps) else 2 <= it <= 6 or it == 8, (it, by_page)
                assert not (by_page and sweeps and shape == "scattered_path") or it == 8
        assert a.stats()["read_io_cnt"] == pages and not r.c.aborted()
