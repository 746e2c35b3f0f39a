"""Workloads of the GPU-side storage-access path, as a program that uses this package runs them.

A case is a dict of plain values.  `prepare` builds what such a program has in hand before the call (the store with its
controller, the page cache, the array over it, the index tensors, the plan of a graph), `run` makes one call or the short
sequence of calls that belongs together, and `work` says what no implementation can do without.  Sizes are those of
bench.py and of the tests, or generic; everything is 64-bit unsigned data behind pages of 512 to 8192 bytes.

Where `cache_pages` covers the array the data is resident (a working set that fits device memory, read again and again);
where it does not, every call reads from the store what earlier calls have pushed out.
"""
import ctypes
import itertools
import math
import random

import numpy as np
import torch

import bam_amd
from bam_amd import gen
from bam_amd.host import vectoradd

_serial = itertools.count()


def listed():
    return [
        # a handful of lookups in a small resident table: launch and latency are all there is
        {"name": "gather_small", "op": "gather", "n": 1021, "elems": 1 << 20, "page": 4096, "cache_pages": 1 << 11},
        # the lookups of one minibatch in a resident table of 256 MiB
        {"name": "gather_batch", "op": "gather", "n": 300007, "elems": 1 << 25, "page": 4096, "cache_pages": 1 << 16},
        # the array benchmark's access pattern with all data resident (1 GiB), values handed out
        {"name": "gather_large", "op": "gather", "n": (1 << 26) - 5, "elems": 1 << 27, "page": 4096, "cache_pages": 1 << 18},
        # lookups in an array twice as large as the cache: half of the pages come from the store
        {"name": "gather_evicting", "op": "gather", "n": (1 << 22) + 13, "elems": 1 << 28, "page": 4096, "cache_pages": 1 << 18},
        # one step of the array benchmark at full size: 2^26 reads summed, 2 GiB store behind a 1 GiB cache
        {"name": "read_step", "op": "read", "n": 1 << 26, "elems": 1 << 28, "page": 4096, "cache_pages": 1 << 18},
        # the cache benchmark: waves stream runs of pages of a resident 1 GiB through bam_ptr
        {"name": "stream_resident", "op": "stream", "mode": 1, "pages_per_wave": 16, "elems": 1 << 27, "page": 4096, "cache_pages": 1 << 18},
        # running sums over resident data, a ragged last block
        {"name": "scan", "op": "scan", "block": 256, "elems": (1 << 26) - 3, "page": 4096, "cache_pages": 1 << 17},
        # three arrays through a cache of half their size, results written back to the store
        {"name": "vectoradd", "op": "vectoradd", "elems": 10_000_003, "page": 4096, "cache_pages": 29_300},
        # scattered read-modify-write of resident data: counters, embeddings being trained
        {"name": "update", "op": "update", "api": 0, "n": 1_000_003, "elems": 1 << 25, "page": 4096, "cache_pages": 1 << 16},
        # raw random block reads into cache slots, one command per thread
        {"name": "block_read", "op": "block", "n": 200_003, "req": 4096, "page": 4096},
        # level-synchronous BFS of a power-law graph along the edge pages, a quarter of the edges cached
        {"name": "bfs", "op": "bfs", "kind": "by_page", "scale": 21, "share": 4, "page": 4096},
        # connected components of a uniform random graph, vertex by vertex through bam_ptr, half of the edges cached
        {"name": "cc", "op": "cc", "kind": "per_vertex", "scale": 22, "share": 2, "page": 4096},
    ]


def _spread(rng, low, high):
    """a whole number between low and high, spread over the logarithm, odd ones among them"""
    return max(low, min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def _pages(elems, page):
    return (elems * 8 + page - 1) // page


def draw(rng):
    op = rng.choice(["gather", "gather", "read", "stream", "scan", "reduce", "vectoradd", "update", "block", "bfs", "cc"])
    page = rng.choice([4096, 4096, 4096, 512, 8192])
    if op in ("gather", "read"):
        elems = _spread(rng, 1 << 16, 1 << 27)
        pages = _pages(elems, page)
        if rng.random() < 0.6:
            return {"op": op, "n": _spread(rng, 1000, 1 << 26), "elems": elems, "page": page, "cache_pages": pages}
        # what the store has to deliver bounds these: as many requests as keep a pass within a fraction of a second
        return {"op": op, "n": _spread(rng, 1000, 1 << 22), "elems": elems, "page": page, "cache_pages": max(256, pages // rng.choice([2, 4]))}
    if op == "stream":
        elems = _spread(rng, 1 << 18, 1 << 27)
        return {"op": op, "mode": rng.choice([0, 1, 2]), "pages_per_wave": rng.choice([1, 4, 16, 24]), "elems": elems, "page": page, "cache_pages": _pages(elems, page)}
    if op in ("scan", "reduce"):
        elems = _spread(rng, 1 << 12, 1 << 26)
        return {"op": op, "block": rng.choice([64, 128, 256, 512, 1024]), "elems": elems, "page": page, "cache_pages": _pages(elems, page)}
    if op == "vectoradd":
        elems = _spread(rng, 1 << 16, 10_000_003)
        return {"op": op, "elems": elems, "page": 4096, "cache_pages": max(256, 3 * _pages(elems, 4096) // rng.choice([1, 2]))}
    if op == "update":
        elems = _spread(rng, 1 << 18, 1 << 25)
        return {"op": op, "api": rng.choice([0, 1, 2]), "n": min(elems // 4, _spread(rng, 1000, 1 << 20)), "elems": elems, "page": page, "cache_pages": _pages(elems, page)}
    if op == "block":
        req = rng.choice([512, 2048, 4096])
        return {"op": op, "n": _spread(rng, 1000, 200_003), "req": req, "page": 4096}
    kinds = ["by_page", "per_vertex", "frontier"] if op == "bfs" else ["by_page", "per_vertex"]
    return {"op": op, "kind": rng.choice(kinds), "scale": rng.randint(12, 20 if op == "bfs" else 21), "share": rng.choice([1, 2, 4]), "page": 4096}


class _Store:
    """A store with its controller, and whatever is built on it, taken down in order."""

    def __init__(self, n_bytes, seed, backing=False, io_threads=12):
        path = "/dev/libnvm%d" % next(_serial)
        self.parts = []
        self.target = bam_amd.Target(path, (n_bytes + 8191) // 8192 * 8192, 512, backing=backing, seed=seed, n_io_threads=io_threads)
        self.ctrl = bam_amd.Controller(path, 1, 0)

    def cache(self, page, n_pages):
        pc = bam_amd.PageCache(page, n_pages, 0, self.ctrl)
        self.parts.append(pc)
        return pc

    def array(self, pc, page, elems, first_page=0):
        r = bam_amd.Range(0, elems, first_page, _pages(elems, page), 0, page, pc, 0)
        a = bam_amd.Array(elems, first_page * page, [r], 0)
        self.parts += [r, a]
        return a

    def memory(self, first_word, n_words):
        """the words of a memory-backed store, in host memory"""
        words = (ctypes.c_char * (n_words * 8)).from_address(self.target.L.bam_target_backing(self.target.h) + first_word * 8)
        words.store = self                # the memory is there for as long as somebody looks at it
        return np.frombuffer(words, dtype=np.int64)

    def __del__(self):
        torch.cuda.synchronize()
        for p in reversed(self.parts):
            p.close()
        if hasattr(self, "ctrl"):
            self.ctrl.close()
        if hasattr(self, "target"):
            self.target.close()


def _graph(case, seed):
    if case["op"] == "bfs":
        return gen.rmat_csr(seed, case["scale"])
    # eight neighbours on average: one component holds nearly everything, and some vertices stay by themselves
    return gen.uniform_csr(seed, 1 << case["scale"], 4 << case["scale"])


def prepare(case, seed):
    op, page = case["op"], case["page"]
    s = {"case": dict(case)}
    if op in ("bfs", "cc"):
        off, nb = _graph(case, seed)
        n_e = nb.numel()
        s["store"] = st = _Store(n_e * 8, seed, backing=True)
        torch.from_numpy(st.memory(0, n_e)).copy_(nb)
        s["a"] = st.array(st.cache(page, max(2048, _pages(n_e, page) // case["share"])), page, n_e)
        s["off"] = off
        s["a"].set_graph(off)
        if op == "bfs":
            # a source in the part of the graph that everything else hangs on: one of the vertices with more edges than most
            deg = off[1:] - off[:-1]
            candidates = torch.nonzero(deg >= 16).flatten()
            s["src"] = int(candidates[random.Random(seed).randrange(candidates.numel())])
        return s
    if op == "block":
        s["store"] = st = _Store(16 << 30, seed)
        s["pc"] = st.cache(page, case["n"])
        s["lbas"] = gen.block_lbas(seed, case["n"], 16 << 30, case["req"], 512)
        return s
    elems = case["elems"]
    pages = _pages(elems, page)
    if op == "vectoradd":
        s["store"] = st = _Store(3 * pages * page, seed, backing=True)
        pc = st.cache(page, case["cache_pages"])
        s["pc"] = pc
        s["a"], s["b"], s["c"] = (st.array(pc, page, elems, k * pages) for k in range(3))
        return s
    s["store"] = st = _Store(pages * page, seed, backing=op == "update", io_threads=4 if case["cache_pages"] >= pages else 12)
    s["a"] = st.array(st.cache(page, case["cache_pages"]), page, elems)
    s["a"].gather(min(pages, case["cache_pages"]), None, stride=page // 8)          # the cache is warm: one element of every page that fits
    if op in ("gather", "read"):
        s["idx"] = gen.gather_indices(seed, case["n"], elems)
    elif op == "update":
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        s["idx"] = torch.randperm(elems, generator=g, device="cuda")[: case["n"]].contiguous()      # no element twice: the order of the adds does not show
        s["values"] = gen.words(seed + 1, 0, case["n"])
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "gather":
        return s["a"].gather(case["n"], s["idx"])
    if op == "read":
        return s["a"].read(case["n"], s["idx"]) - (1 << 63)          # the sum is an unsigned 64-bit number
    if op == "stream":
        ppw = case["pages_per_wave"]
        waves = max(1, _pages(case["elems"], case["page"]) // ppw)
        return s["a"].stream(waves, min(ppw, case["cache_pages"]), mode=case["mode"]) - (1 << 63)
    if op == "scan":
        return s["a"].scan(case["elems"], block_size=case["block"])
    if op == "reduce":
        return s["a"].reduce(case["elems"], block_size=case["block"])
    if op == "vectoradd":
        vectoradd(s["a"], s["b"], s["c"], case["elems"])
        s["pc"].flush()                                               # the result is on the store
        return s["store"].memory(2 * _pages(case["elems"], case["page"]) * case["page"] // 8, case["elems"])
    if op == "update":
        return s["a"].update(case["api"], s["idx"], s["values"])
    if op == "block":
        s["pc"].block_io(case["n"], case["req"], s["lbas"])
        return s["pc"].block_checksums(case["n"], case["req"])
    if op == "bfs":
        kind = case["kind"]
        return s["a"].bfs(s["off"], s["src"], coarse=64, by_page=kind == "by_page", frontier=kind == "frontier")
    return s["a"].cc(s["off"], coarse=64, by_page=case["kind"] == "by_page")[0]          # (the number of sweeps depends on the order of the updates)


def work(case):
    """Each input read once, each output written once.  Of an array larger than its cache the pages that cannot have been
    kept are read from the store as whole pages."""
    op = case["op"]
    if op in ("bfs", "cc"):
        v = 1 << case["scale"]
        # 16 undirected edges per vertex drawn (of a power-law graph's some coincide), 4 of the uniform graph
        entries = (30 if op == "bfs" else 8) * v
        return {"bytes": entries * 8 + (v + 1) * 8 + v * (4 if op == "bfs" else 8), "flops": 0}
    if op == "block":
        return {"bytes": case["n"] * (8 + case["req"] + 8), "flops": 0}
    elems, page, n = case["elems"], case["page"], case.get("n", 0)
    pages = _pages(elems, page)
    if op in ("gather", "read"):
        touched = pages * -math.expm1(-n / pages)
        from_store = max(0.0, touched - case["cache_pages"]) * page
        return {"bytes": n * (24 if op == "gather" else 16) + from_store, "flops": 0}
    if op == "stream":
        return {"bytes": max(1, pages // case["pages_per_wave"]) * min(case["pages_per_wave"], case["cache_pages"]) * page, "flops": 0}
    if op == "scan":
        return {"bytes": elems * 16 + 8, "flops": 0}
    if op == "reduce":
        return {"bytes": elems * 8 + elems * 8 // (2 * case["block"]), "flops": 0}
    if op == "vectoradd":
        return {"bytes": elems * 24, "flops": 0}
    return {"bytes": n * 40, "flops": 0}          # update: index, value, the element in and out, what it held before


def tolerance(case):
    """Every result is whole numbers: sums modulo 2^64, elements, levels, component labels."""
    return "exact"
