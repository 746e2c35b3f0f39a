"""Components from the forest of the first neighbours of lists: which of them lie in a page that is there, and graphs whose trees are long."""
import numpy as np
import pytest

import oracle
from test_gpu_along_pages import _rig
from test_gpu_cc_joined import _csr, _pairs
from test_gpu_parity import _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


def _check(bam, off, nb, page, cache_pages, calls=3):
    want, _ = oracle.cc_labels(off, nb)
    r, a = _rig(bam, nb, page, cache_pages)
    with r:
        d_off = _dev(off)
        a.set_graph(d_off)
        for k in range(calls):                            # cold, then with what each call leaves in the cache
            for by_page in (False, True):
                lb, _ = a.cc(d_off, by_page=by_page)
                assert np.array_equal(_u64(lb), want), (k, by_page)
        assert not r.c.aborted()


@pytest.mark.parametrize("shape", ["wide", "sparse", "path", "scattered_path", "star", "loops_and_copies", "one"])
@pytest.mark.parametrize("page,share", [(512, 1), (512, 3), (4096, 1), (4096, 2), (4096, 5), (65536, 1), (65536, 2)])
def test_labels(bam, shape, page, share):
    """lists whose first entries lie on both sides of a page's end, of which one page is there; fewer entries than are looked at"""
    n_v, rng = 30011, np.random.default_rng(page + share)
    if shape in ("wide", "sparse"):
        n = 4 * n_v if shape == "wide" else 3 * n_v // 5
        u, v = rng.integers(0, n_v, n), rng.integers(0, n_v, n)
    else:
        u, v = _pairs(shape, n_v, rng)
    off, nb = _csr(n_v, u, v)
    _check(bam, off, nb, page, max(2, -(-len(nb) * 8 // page) // share))


@pytest.mark.parametrize("n_v", [1, 2, 255, 256, 257, 1025])
def test_small_graphs(bam, n_v):
    rng = np.random.default_rng(n_v)
    off, nb = _csr(n_v, rng.integers(0, n_v, 2 * n_v), rng.integers(0, n_v, 2 * n_v))
    _check(bam, off, nb, 4096, 64, calls=2)


@pytest.mark.parametrize("shape", ["path", "wide"])
@pytest.mark.parametrize("n_v", [(1 << 21) - 1, 1 << 21])
def test_labels_where_a_round_is_left_out(bam, n_v, shape):
    rng = np.random.default_rng(n_v)
    u, v = _pairs(shape, n_v, rng) if shape == "path" else (rng.integers(0, n_v, n_v), rng.integers(0, n_v, n_v))
    off, nb = _csr(n_v, u, v)
    _check(bam, off, nb, 4096, -(-len(nb) // 512), calls=1)


@pytest.mark.parametrize("shape,n_v", [("wide", 30011), ("path", (1 << 20) + 3)])
@pytest.mark.parametrize("page,share", [(512, 2), (4096, 1)])
def test_without_reads_that_hold_no_reference(bam, shape, n_v, page, share, monkeypatch):
    """BAM_FAST_READS=0: every vertex begins by itself, and nothing is looked at before the pages of the edges are held"""
    monkeypatch.setenv("BAM_FAST_READS", "0")
    rng = np.random.default_rng(page)
    u, v = _pairs(shape, n_v, rng) if shape == "path" else (rng.integers(0, n_v, 4 * n_v), rng.integers(0, n_v, 4 * n_v))
    off, nb = _csr(n_v, u, v)
    _check(bam, off, nb, page, max(2, -(-len(nb) * 8 // page) // share), calls=2)
