"""Graph calls of several arrays behind one small cache at a time: a wave holds no page while it waits for another, so that whatever
their number none waits for slots that the others have."""
import threading

import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, bam, _dev, _u64  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu

CALLS = 6


@pytest.mark.parametrize("what", ["levels", "components", "pagerank"])
@pytest.mark.parametrize("page,cache_pages", [(512, 24), (512, 700), (4096, 5), (4096, 96), (131072, 4)])
def test_six_calls_at_a_time(bam, what, page, cache_pages):
    import torch
    from bam_amd import Array, PageCache, Range
    off, nb = oracle.uniform_csr(SEED, 5003, 40009) if what == "components" else oracle.rmat_csr(SEED, 12)
    per = page // 8
    pages = -(-len(nb) // per)
    srcs = [int(x) for x in oracle.bfs_sources(SEED, off, CALLS)]
    with Rig(bam, CALLS * pages * page, backing=True, n_queues=16, depth=256, stage_bytes=max(4096, min(page, 8192))) as r:
        for k in range(CALLS):
            r.backing(CALLS * pages * per)[k * pages * per:][:len(nb)] = nb
        pc = PageCache(page, cache_pages, 0, r.c)
        rgs = [Range(0, len(nb), k * pages, pages, 0, page, pc, 0) for k in range(CALLS)]
        arrays = [Array(len(nb), k * pages * page, [rg], 0) for k, rg in enumerate(rgs)]
        d_off = _dev(off)
        for a in arrays:
            a.set_graph(d_off)
        torch.cuda.synchronize()
        got, start = [[] for _ in arrays], threading.Barrier(CALLS)

        def work(k):
            torch.cuda.set_device(0)
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait(60)
                for rep in range(3):
                    if what == "levels":
                        out, it = arrays[k].bfs(d_off, srcs[k], by_page=page > 65536 or bool(rep & 1))
                    elif what == "components":
                        out, it = arrays[k].cc(d_off, by_page=page > 65536 or bool(rep & 1))
                    else:
                        out, it = arrays[k].pagerank(d_off, 0.85, 1e-3, 1000, by_page=True)
                    got[k].append((out.cpu().numpy(), it))

        threads = [threading.Thread(target=work, args=(k,)) for k in range(CALLS)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not r.c.aborted()
        if what == "pagerank":
            limit = oracle.pagerank_limit(off, nb, 0.85)
        for k in range(CALLS):
            assert len(got[k]) == 3, k
            for out, it in got[k]:
                if what == "levels":
                    want, levels = oracle.bfs_levels(off, nb, srcs[k])
                    assert np.array_equal(out.view(np.uint32), want) and it == levels, k
                elif what == "components":
                    assert np.array_equal(out.view(np.uint64), oracle.cc_labels(off, nb)[0]), k
                else:
                    tol = 1e-3 / (1 - 0.85)             # what may be left unpushed, as in test_pagerank_values
                    assert (out <= limit * (1 + 1e-5)).all() and (out >= limit * (1 - tol - 1e-5)).all(), k
        for x in arrays + rgs:
            x.close()
        pc.close()
