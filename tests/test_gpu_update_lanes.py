"""bam_array_update through AtomicAdd with several elements per lane: edges of a launch, runs of lanes on a page, missing pages."""
import numpy as np
import pytest

import oracle
from test_gpu_parity import Rig, SEED, _check_add_chains, _dev, _u64, bam  # noqa: F401  (bam is the module fixture)

pytestmark = pytest.mark.gpu


# on both sides of where four elements per thread begin, the last workgroup short by different amounts; all pages resident, none, some
@pytest.mark.parametrize("kind", ["scattered", "in_order", "one_page", "one_element"])
@pytest.mark.parametrize("n,block,warm", [(1, 64, 300), (513, 64, 0), ((1 << 17) - 1, 64, 300), (1 << 17, 64, 300), ((1 << 17) + 1, 64, 300), ((1 << 17) + 255, 256, 300),
                                          (140009, 192, 300), (133000, 1024, 300), ((1 << 17) + 1, 64, 0), (140009, 256, 77)])
def test_adds_element_by_element(bam, n, block, warm, kind):
    n_elems = 300 * 512 - 5
    rng = np.random.default_rng(n)
    with Rig(bam, 300 * 4096, backing=True, n_queues=8, depth=256) as r:
        x0 = r.backing(n_elems).copy()
        a = r.array(n_elems, 4096, 300)
        if warm:
            a.gather(warm, None, stride=512)
        idx = {"scattered": rng.permutation(n_elems)[:n], "in_order": np.arange(n) + 500, "one_page": rng.integers(512, 1024, n), "one_element": np.full(n, 77)}[kind].astype(np.uint64)
        vals = rng.integers(1, 1 << 20, n).astype(np.uint64)
        outside = rng.integers(0, n, 3) if n > 63 else np.zeros(0, dtype=np.int64)
        idx[outside] = np.array([n_elems, 1 << 40, (1 << 64) - 1], dtype=np.uint64)[: len(outside)]
        inside = idx < n_elems
        a.stats()
        old = _u64(a.update(0, _dev(idx), _dev(vals), block_size=block))
        st = a.stats()
        assert st["access_cnt"] == inside.sum() and (warm < 300 or st["hit_cnt"] == inside.sum()), st
        model = x0.copy()
        np.add.at(model, idx[inside].astype(np.int64), vals[inside])
        r.objs[0][2].flush()
        assert np.array_equal(r.backing(n_elems), model) and not old[~inside].any()
        if kind in ("scattered", "in_order"):                 # no element twice
            assert np.array_equal(old[inside], x0[idx[inside].astype(np.int64)])
        else:
            _check_add_chains(x0, idx[inside], vals[inside], old[inside], model)
        assert not r.c.aborted()


def test_adds_while_another_array_evicts(bam):
    """four elements per lane of an array that fits the cache, while gathers from another array of the same cache push its pages out:
    what is resident is added to under references, the rest the way that can miss, and nothing is lost between"""
    import torch
    from bam_amd import Array, PageCache, Range
    pages, other, n = 300, 4096, (1 << 17) + 321
    n_elems = pages * 512 - 5
    rng = np.random.default_rng(11)
    with Rig(bam, (pages + other) * 4096, backing=True, n_queues=16, depth=256) as r:
        x0 = r.backing(n_elems).copy()
        pc = PageCache(4096, 512, 0, r.c)
        ra, rb = Range(0, n_elems, 0, pages, 0, 4096, pc, 0), Range(0, other * 512, pages, other, 0, 4096, pc, 0)
        a, b = Array(n_elems, 0, [ra], 0), Array(other * 512, pages * 4096, [rb], 0)
        d_other = _dev(rng.integers(0, other * 512, 4096).astype(np.uint64))
        words = r.backing((pages + other) * 512)[pages * 512:].copy()
        want_other = words[_u64(d_other).astype(np.int64)]
        model = x0.copy()
        a.gather(pages, None, stride=512)
        side = torch.cuda.Stream()
        a.stats()
        missed = 0
        for rep in range(6):
            idx = rng.permutation(n_elems)[:n].astype(np.uint64)
            vals = rng.integers(1, 1 << 20, n).astype(np.uint64)
            d_idx, d_vals = _dev(idx), _dev(vals)
            torch.cuda.synchronize()
            outs = []
            with torch.cuda.stream(side):
                for _ in range(3):
                    outs.append(b.gather(4096, d_other))
            old = a.update(0, d_idx, d_vals, block_size=256)
            torch.cuda.synchronize()
            assert np.array_equal(_u64(old), model[idx.astype(np.int64)]), rep
            model[idx.astype(np.int64)] += vals
            for o in outs:
                assert np.array_equal(_u64(o), want_other), rep
            st = a.stats()
            missed += st["miss_cnt"]
            assert st["access_cnt"] == n, st
        pc.flush()
        assert missed > 0 and np.array_equal(r.backing(n_elems), model) and not r.c.aborted()
        a.close(); b.close(); ra.close(); rb.close(); pc.close()
