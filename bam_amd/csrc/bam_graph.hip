// Graph kernels of the C-ABI library: BFS (per vertex, over queues of vertices, by edge page), connected components,
// PageRank and SSSP over CSR graphs whose neighbour ids (and weights) are read through the page cache.  Kernel shapes
// follow the reference's benchmark kernels (cited per kernel); lane arithmetic is for 64-wide waves.
#include "along_tables.h"
#include "bam_capi_internal.h"

#include <atomic>

namespace {

/* the per-vertex kernels (the group walk below) are held to the registers of this many waves per SIMD: left alone the
 * compiler takes what a workgroup of two waves may have, all 512, and one wave per SIMD is what runs */
#ifndef BAM_GRAPH_WAVES
#define BAM_GRAPH_WAVES 2
#endif
#define BAM_GRAPH_KERNEL_WAVES __attribute__((amdgpu_waves_per_eu(BAM_GRAPH_WAVES)))

// ---- BFS: wave per `coarse` vertices, edges through bam_ptr (benchmarks/bfs/main.cu:658-689) ----
#define MYINFINITY 0xFFFFFFFFu
/*
 * Read-ahead for a wave that walks one vertex's edge list through bam_ptr.  Left to itself the walk meets the
 * pages of the list one after the other and pays one full trip to the store for each; the list of a hub of a
 * power-law graph covers hundreds of pages, and the one wave that has it then decides how long the whole level
 * takes.  Whenever the walk is about to enter pages it has not asked for yet, the lanes touch the next pages of
 * the list (one each, taken and dropped again): those that are not resident are loaded as one batch of commands,
 * and the walk that follows finds them there.  Nothing is held, so a page that is evicted again before the walk
 * gets to it is simply read once more; results do not depend on it.  Arrays of one range only, and the reach
 * scales with the cache (a 64th of its pages, at most one page per lane).
 */
template <typename T>
struct list_read_ahead {
    bam::range_view<T> view;
    uint64_t asked_to = 0, last_page = 0;
    uint32_t reach = 0;
    bool long_list = false;
    __device__ __forceinline__ void init(array_d_t<T>* da)
    {
        if (da->n_ranges != 1) return;
        view.load(da->d_ranges);
        /* what is touched ahead may be placed directly up to the higher of the cache's two bounds: measured on the per-vertex
         * BFS (RMAT-24) 4.55 GTEPS with at most 1024 directly placed commands in flight, 4.7 with 4096 to 8192, 4.46 with 16384 */
        view.place = BAM_PLACE_AHEAD;
        const uint64_t r = da->d_ranges[0].cache.n_pages >> 6;
        reach = r > BAM_WAVE_SIZE ? BAM_WAVE_SIZE : (uint32_t)r;
    }
    /* every lane's elements [es, ee) (empty for lanes without any) are about to be read: touch the first and the last page
     * of each run, so that what is not resident comes in as one batch or two, not one trip to the store per run */
    __device__ __forceinline__ void group(const uint64_t es, const uint64_t ee)
    {
        if (reach < 2) return;
        const bool want = ee > es;
        if (!bam::ballot(want)) return;
        auto touch = [](uint32_t) { return true; };
        const uint64_t pf = want ? view.page_of(es) : 0, pl = want ? view.page_of(ee - 1) : 0;
        /* all lanes go in: those without a page of their own help move what the others load */
        const bool take_f = want && page_absent(view, pf), take_l = want && pl != pf && page_absent(view, pl);
        /* the last pages go along with the first ones as far as there are lanes without a first page to ask for (the k-th such
         * lane takes the last page of the k-th lane that has one): one batch of commands instead of two, of which the second
         * would be small (few lists cross a page boundary) */
        const uint64_t need_l = bam::ballot(take_l), idle = ~bam::ballot(take_f);
        const uint32_t k = bam::popc(idle & bam::lanes_below(bam::lane()));
        const bool adopt = !take_f && k < bam::popc(need_l);
        uint64_t m = need_l;
        if (adopt) for (uint32_t i = 0; i < k; i++) m &= m - 1;
        const uint64_t adopted = bam::shfl(pl, adopt ? bam::first_lane(m) : 0u);
        const bool take_1 = take_f || adopt;
        if (bam::ballot(take_1)) view.template acquire_helped<true>(take_f ? pf : adopted, take_1, false, touch, touch);
        /* last pages nobody had a lane for */
        const bool take_2 = take_l && bam::popc(need_l & bam::lanes_below(bam::lane())) >= bam::popc(idle);
        if (bam::ballot(take_2)) view.template acquire_helped<true>(pl, take_2, false, touch, touch);
        view.n_access = view.n_hit = 0;
    }
    /*
     * The lists of the items [first, last) lie in the array in the order of the items (consecutive vertices, or a sorted
     * queue of them): touch every page that holds
     * entries of a list that is about to be walked (item(v, v) says which; lists that go to the queue of long ones are
     * left out), `reach` pages at a time with one page per lane, so that what is not resident comes in as few, large
     * batches of commands.  The store path moves several times more pages per second in batches of sixteen than in
     * batches of two or three, which is what touching the lists of 64 vertices at a time gives on a graph with a few
     * dozen edges per vertex.  False if the span is too wide for that (the caller then touches list by list).
     */
    template <typename Item>
    __device__ __forceinline__ bool span(const uint64_t* vertexList, const uint64_t first, const uint64_t last, const uint64_t heavy_from, Item item,
                                         bool& nothing)
    {
        nothing = false;
        if (reach < 2) return false;
        uint64_t v_first = 0, v_last = 0;
        item(first, v_first); item(last - 1, v_last);
        const uint64_t e0 = vertexList[v_first], e1 = vertexList[v_last + 1];
        if (e1 <= e0) { nothing = true; return true; }
        const uint64_t p0 = view.page_of(e0), p1 = view.page_of(e1 - 1);
        if (p1 - p0 >= 4ull * reach) return false;
        auto touch = [](uint32_t) { return true; };
        const uint32_t lane = bam::lane();
        uint64_t seen = 0;
        for (uint64_t c = p0; c <= p1; c += reach) {
            uint64_t m = 0;
            for (uint64_t b = first; b < last; b += BAM_WAVE_SIZE) {
                uint64_t v = 0;
                if (b + lane < last && item(b + lane, v)) {
                    const uint64_t es = vertexList[v], ee = vertexList[v + 1];
                    if (ee > es && ee - es < heavy_from) {
                        const uint64_t pf = view.page_of(es), pl = view.page_of(ee - 1);
                        const uint64_t f = pf > c ? pf - c : 0, l = pl < c + reach - 1 ? pl - c : reach - 1;
                        if (pl >= c && f <= l) m |= (~0ull >> (63 - l)) & (~0ull << f);
                    }
                }
            }
#pragma unroll
            for (uint32_t o = BAM_WAVE_SIZE / 2; o; o >>= 1) m |= bam::shfl(m, lane ^ o);
            const bool take = ((m >> lane) & 1) != 0 && page_absent(view, c + lane);
            if (bam::ballot(take)) view.template acquire_helped<true>(c + lane, take, false, touch, touch);
            seen |= m;
        }
        view.n_access = view.n_hit = 0;
        nothing = seen == 0;            /* no list to walk in [first, last): the caller need not look again */
        return true;
    }
    /* wave-uniform: the list is elements [start, end); its first `asked` pages have been touched already */
    __device__ __forceinline__ void begin(const uint64_t start, const uint64_t end, const uint32_t asked = 0)
    {
        long_list = false;
        if (reach < 2 || end <= start) return;
        last_page = view.page_of(end - 1);
        long_list = last_page > view.page_of(start);
        asked_to = asked ? view.page_of(start) + asked : 0;
    }
    /* lane l brings page (l mod 16) of a run of elements [start, end) of its own (four runs per wave, `want` says whether
     * the lane's run is to be read at all): one batch of commands for what is not resident of the first sixteen pages of
     * each.  False if the cache is too small for a wave to ask for that much at a time. */
    __device__ __forceinline__ bool quads(const uint64_t start, const uint64_t end, const bool want)
    {
        if (reach < BAM_WAVE_SIZE) return false;
        auto touch = [](uint32_t) { return true; };
        const uint64_t page = want ? view.page_of(start) + (bam::lane() & 15u) : 0;
        const bool take = want && end > start && page <= view.page_of(end - 1) && page_absent(view, page);
        if (bam::ballot(take)) view.template acquire_helped<true>(page, take, false, touch, touch);
        view.n_access = view.n_hit = 0;
        return true;
    }
    /* wave-uniform: the walk is about to read from element `at` on */
    __device__ __forceinline__ void step(const uint64_t at)
    {
        if (!long_list) return;
        const uint64_t pg = view.page_of(at);
        if (pg < asked_to) return;
        const uint64_t p = pg + bam::lane();
        auto touch = [](uint32_t) { return true; };
        const bool take = bam::lane() < reach && p <= last_page && page_absent(view, p);
        if (bam::ballot(take)) view.template acquire_helped<true>(p, take, false, touch, touch);
        asked_to = pg + reach;
        view.n_access = view.n_hit = 0;         /* not accesses of the kernel's own: kept out of the counters */
    }
};

/*
 * Every lane brings a run of elements [es, ee) (possibly empty, each shorter than 2^20) and the vertex `src` the run
 * belongs to; the wave visits all elements of all runs, 64 per step, consecutive lanes taking consecutive elements
 * across the ends of the runs.  With lists of a dozen edges, walking one list per step leaves most lanes idle and
 * pays the whole chain of dependent loads (offsets, payload, label) once per vertex; packed, it is paid once per 64
 * edges.  A lane finds the run its element belongs to by binary search in the running sums of the run lengths
 * (six shuffles).  `read(i)` fetches element i, `visit(src, value, i)` consumes it.
 */
template <typename Read, typename Visit>
__device__ __forceinline__ void walk_packed(const uint64_t es, const uint64_t ee, const uint64_t src, Read read, Visit visit)
{
    const uint32_t lane = bam::lane();
    const uint32_t len = (uint32_t)(ee - es);
    uint32_t incl = len;
#pragma unroll
    for (uint32_t o = 1; o < BAM_WAVE_SIZE; o <<= 1) {
        const uint32_t u = bam::shfl(incl, lane >= o ? lane - o : lane);
        if (lane >= o) incl += u;
    }
    const uint32_t total = bam::shfl(incl, BAM_WAVE_SIZE - 1), excl = incl - len;
    for (uint32_t base = 0; base < total; base += BAM_WAVE_SIZE) {
        const uint32_t k = base + lane;
        uint32_t j = 0;                                          /* number of runs that end at or before k */
#pragma unroll
        for (uint32_t step = BAM_WAVE_SIZE / 2; step; step >>= 1)
            if (bam::shfl(incl, j + step - 1) <= k) j += step;
        j &= BAM_WAVE_SIZE - 1;                                  /* lanes past the end: any valid lane, they do not visit */
        const uint64_t i = bam::shfl(es, j) + (k - bam::shfl(excl, j));
        const uint64_t s = bam::shfl(src, j);
        if (k < total) visit(s, read(i), i);
    }
}

/*
 * The traversal of the reference's coarsened per-vertex kernels (bfs/main.cu:658-689, cc/main.cu:123-144): the
 * vertices are handed out in groups of `coarse`, and the edge list of every active vertex is read through bam_ptr.
 * What differs, for the store's and the memory system's sake:
 *  - the launch has as many waves as the device holds at a time, and a wave takes the next piece of work when it is
 *    done with its last one (one atomic each).  One group per wave of a large grid leaves most of the device idle
 *    here: groups differ in length by orders of magnitude, and workgroups are started in order;
 *  - the flags and offsets of 64 vertices are read at a time, one vertex per lane, and the lists of those vertices
 *    are walked packed (walk_packed): 64 edges per step whichever vertices they belong to;
 *  - before the walk the pages that hold the lists of the group's active vertices are touched (list_read_ahead::span),
 *    so that what is not resident comes in as one batch of commands, not one trip to the store per vertex;
 *  - lists of BAM_HEAVY_EDGES entries and more are walked in pieces, by a wave each (below).
 */
/*
 * A list of BAM_HEAVY_EDGES entries or more is not walked with its group: it is cut into pieces of BAM_PIECE_EDGES
 * entries, each walked by a wave of its own.  The hubs of a power-law graph have lists of hundreds of pages; walked
 * by one wave, a single hub takes longer than all other vertices of its level together.  Which lists are long does
 * not change from sweep to sweep, so the pieces are listed once per call (k_heavy_pieces) and every sweep hands them
 * out before the groups, longest work first: a piece whose vertex is not active costs its wave one look at the flag.
 */
#define BAM_HEAVY_EDGES 1024u
/* entries per piece: 16 pages of 4 KiB, which the wave that walks the piece asks for as one batch of commands.  Pieces
 * of the threshold's size reach the store as batches of two or three commands, and the store path moves far fewer
 * pages per second in such batches than in batches of sixteen */
#define BAM_PIECE_EDGES 8192u
#define BAM_PIECE_BUNDLE 4u             /* pieces handed to a wave at a time: sixteen lanes look after the sixteen pages of each */
static_assert(BAM_PIECE_BUNDLE * 16u == BAM_WAVE_SIZE && BAM_PIECE_EDGES * 8u == 16u * 4096u, "a bundle's pages are shared out one per lane");
struct heavy_piece_t { uint64_t v, first, last; };      /* entries [first, last) of the list of vertex v */

/* *lists_end: where the last list ends, for the host */
__global__ void k_heavy_pieces(const uint64_t* vertexList, const uint64_t vertex_count, heavy_piece_t* pieces, unsigned long long* count, unsigned long long* lists_end)
{
    const uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= vertex_count) return;
    const uint64_t start = vertexList[v], end = vertexList[v + 1];
    if (v == vertex_count - 1) *lists_end = end;
    if (end - start < BAM_HEAVY_EDGES) return;
    const uint64_t n = (end - start + BAM_PIECE_EDGES - 1) / BAM_PIECE_EDGES;
    const unsigned long long at = atomicAdd(count, (unsigned long long)n);
    for (uint64_t k = 0; k < n; k++) {
        const uint64_t f = start + k * BAM_PIECE_EDGES;
        pieces[at + k] = heavy_piece_t{v, f, f + BAM_PIECE_EDGES < end ? f + BAM_PIECE_EDGES : end};
    }
}

/*
 * Reads with the page referenced for the one read only.  bam_ptr keeps every lane's page referenced until the lane
 * moves on: fine where the lanes of a wave read side by side, but 64 lanes that walk lists scattered over the edge
 * array would pin up to 64 pages per wave, and a cache with fewer free slots than that stops for good (lanes that
 * have their page wait for those that cannot get one).  Lanes on the same page still share one pair of atomics.
 */
template <typename T>
struct touch_reader {
    array_d_t<T>* da = nullptr;
    bam::range_view<T> view;
    bool one_range = false, fast = false;
    __device__ __forceinline__ void init(array_d_t<T>* a)
    {
        da = a;
        one_range = a->n_ranges == 1;
        if (one_range) { view.load(a->d_ranges); fast = a->d_ranges[0].cache.fast_reads != 0; }
    }
    __device__ __forceinline__ T read(const uint64_t i)
    {
        if (!one_range) return da->seq_read(i);
        T ret = T();                                    /* stays T() if the wait is given up */
        const uint64_t byte = view.byte_of(i);
        /* resident pages without a reference at all, as array_d_t::seq_read does */
        if (fast && bam_read_unpinned(view.pages + (byte >> view.page_size_log), view.base_addr, view.page_size_log, byte & (view.page_size - 1), ret)) {
            view.account(true);
            return ret;
        }
        auto use = [&](uint32_t slot) { ret = bam::ld_payload((T*)(view.slot_addr(slot) + (byte & (view.page_size - 1)))); return true; };
        view.template acquire<true>(byte >> view.page_size_log, false, use, use);
        return ret;
    }
    __device__ __forceinline__ void fini() { if (one_range) view.flush_stats(); }
};

/*
 * One sweep: the pieces of the long lists whose vertex is active(v), then `n_items` work items in groups of `coarse`,
 * each of which names a vertex and says whether it is to be walked: item(i, v).  visit(src, value, i) for every entry.
 * HOLD: the items are the vertices themselves (item i is vertex i, lists side by side), read through bam_ptr;
 * otherwise the items' lists lie anywhere, and they are read page by page without holding any.
 */
#define BAM_WORK_RUN 8
template <bool HOLD, typename Item, typename Active, typename Visit>
__device__ __forceinline__ void walk_item_groups(array_d_t<uint64_t>* da, const uint64_t* vertexList, const uint64_t n_items, const uint64_t coarse,
                                                 const heavy_piece_t* heavy, const uint64_t n_heavy, unsigned long long* next_work,
                                                 const bool backwards, Item item, Active active, Visit visit,
                                                 list_read_ahead<uint32_t>* with = nullptr, const bool in_order = HOLD)
{
    const uint64_t laneIdx = threadIdx.x % BAM_WAVE_SIZE;
    const uint64_t n_groups = (n_items + coarse - 1) / coarse;
    const uint64_t n_bundles = (n_heavy + BAM_PIECE_BUNDLE - 1) / BAM_PIECE_BUNDLE;
    bam_ptr<uint64_t> ptr(da);
    touch_reader<uint64_t> touch;
    if (!HOLD) touch.init(da);
    list_read_ahead<uint64_t> ahead;
    bool ready = false;
    /* A wave whose last group had nothing to walk takes BAM_WORK_RUN turns at the counter in one: every wave of the device
     * adds to the same word, which takes the device about 12 ns a time, and a sweep with nothing to walk is made of little
     * else (0.6 ms for 2^24 vertices one group per turn, 0.35 ms this way, 0.2 ms with runs of four for everybody).  A wave that
     * found work goes back to single turns: on a dense level, runs of neighbouring groups per wave cost 7 % (fewer waves
     * share a page at a time). */
    bool idle = false;
    for (unsigned long long w0 = 0, left = 0;;) {
        if (!left) {
            left = idle ? BAM_WORK_RUN : 1;
            if (laneIdx == 0) w0 = atomicAdd(next_work, left);
            w0 = bam::bcast((uint64_t)w0, 0);
        }
        const unsigned long long w = w0++;
        left--;
        /* every other sweep runs from the far end of both lists of work: what the last sweep left in the cache is what
         * this one asks for first */
        const uint64_t wb = backwards ? n_bundles - 1 - w : w;
        if (w < n_bundles) {
            /* pieces of long lists, BAM_PIECE_BUNDLE per turn at the counter (every turn costs one atomic on one word, and on
             * a sweep with little to do those atomics are what the sweep takes): all lanes side by side through bam_ptr,
             * read ahead over the piece */
            /* what the active pieces of the bundle need comes in as one batch: a piece by itself asks for six pages on
             * average on a power-law graph, where most long lists are just over the threshold */
            bool asked = false;
            {
                const uint64_t k = wb * BAM_PIECE_BUNDLE + laneIdx / 16;
                heavy_piece_t mine = {0, 0, 0};
                bool want = false;
                if (k < n_heavy) { mine = heavy[k]; want = active(mine.v); }
                if (bam::ballot(want)) {
                    if (!ready) { ahead.init(da); ready = true; }
                    asked = ahead.quads(mine.first, mine.last, want);
                    if (with) with->quads(mine.first, mine.last, want);
                }
            }
            for (uint64_t k = wb * BAM_PIECE_BUNDLE; k < (wb + 1) * BAM_PIECE_BUNDLE && k < n_heavy; k++) {
                const heavy_piece_t pc = heavy[k];
                if (!active(pc.v)) continue;
                if (!ready) { ahead.init(da); ready = true; }
                ahead.begin(pc.first, pc.last, asked ? 16u : 0u);
                if (with) with->begin(pc.first, pc.last, asked ? 16u : 0u);
                for (uint64_t i = (pc.first & 0xFFFFFFFFFFFFFFF0ull) + laneIdx; i < pc.last; i += BAM_WAVE_SIZE) {
                    ahead.step(i - laneIdx > pc.first ? i - laneIdx : pc.first);
                    if (with) with->step(i - laneIdx > pc.first ? i - laneIdx : pc.first);
                    if (i >= pc.first) visit(pc.v, ptr.read(i), i);
                }
            }
            continue;
        }
        if (w - n_bundles >= n_groups) break;
        const uint64_t g = backwards ? n_groups - 1 - (w - n_bundles) : w - n_bundles;
        const uint64_t first = g * coarse;
        bool touched = false, nothing = false;
        if (in_order) {
            if (!ready) { ahead.init(da); ready = true; }
            touched = ahead.span(vertexList, first, first + coarse < n_items ? first + coarse : n_items, BAM_HEAVY_EDGES, item, nothing);
            if (with && touched && !nothing) { bool none; with->span(vertexList, first, first + coarse < n_items ? first + coarse : n_items, BAM_HEAVY_EDGES, item, none); }
            idle = nothing;
            if (nothing) continue;
        }
        for (uint64_t b = 0; b < coarse; b += BAM_WAVE_SIZE) {
            const uint64_t at_item = first + b + laneIdx;
            uint64_t mine = 0;
            const bool act = b + laneIdx < coarse && at_item < n_items && item(at_item, mine);
            if (!bam::ballot(act)) continue;
            if (!ready) { ahead.init(da); ready = true; }
            uint64_t es = 0, ee = 0;
            if (act) { es = vertexList[mine]; ee = vertexList[mine + 1]; }
            if (ee - es >= BAM_HEAVY_EDGES) ee = es;            /* walked in pieces */
            if (!touched) {
                /* a group whose lists cover too many pages for one look: the same for the 64 vertices at hand */
                bool block_touched = false;
                if (in_order) {
                    const uint64_t last = first + coarse < n_items ? first + coarse : n_items;
                    bool none;
                    block_touched = ahead.span(vertexList, first + b, first + b + BAM_WAVE_SIZE < last ? first + b + BAM_WAVE_SIZE : last, BAM_HEAVY_EDGES, item, none);
                    if (with && block_touched) with->span(vertexList, first + b, first + b + BAM_WAVE_SIZE < last ? first + b + BAM_WAVE_SIZE : last, BAM_HEAVY_EDGES, item, none);
                }
                if (!block_touched) { ahead.group(es, ee); if (with) with->group(es, ee); }
            }
            walk_packed(es, ee, mine, [&](uint64_t i) { if constexpr (HOLD) return ptr.read(i); else return touch.read(i); }, visit);
        }
    }
    if (!HOLD) touch.fini();
}

/* the items are the vertices themselves, walked where active(v) */
template <typename Active, typename Visit>
__device__ __forceinline__ void walk_vertex_groups(array_d_t<uint64_t>* da, const uint64_t* vertexList, const uint64_t vertex_count, const uint64_t coarse,
                                                   const heavy_piece_t* heavy, const uint64_t n_heavy, unsigned long long* next_work, const bool backwards,
                                                   Active active, Visit visit, list_read_ahead<uint32_t>* with = nullptr)
{
    walk_item_groups<true>(da, vertexList, vertex_count, coarse, heavy, n_heavy, next_work, backwards,
                           [&](uint64_t i, uint64_t& v) { v = i; return active(i); }, active, visit, with);
}

__global__ __launch_bounds__(128) BAM_GRAPH_KERNEL_WAVES void k_bfs_coalesce_coarse_ptr_pc(array_d_t<uint64_t>* da, uint32_t* label, const uint32_t level, const uint64_t vertex_count,
                                                                   const uint64_t* vertexList, uint64_t* changed, uint64_t coarse,
                                                                   const heavy_piece_t* heavy, uint64_t n_heavy, unsigned long long* next_work)
{
    bool any = false;
    walk_vertex_groups(da, vertexList, vertex_count, coarse, heavy, n_heavy, next_work, (level & 1u) != 0,
                       [&](uint64_t v) { return label[v] == level; },
                       [&](uint64_t, uint64_t next, uint64_t) { if (label[next] == MYINFINITY) { label[next] = level + 1; any = true; } });
    if (any) *changed = 1;
}

// ---- the reference's other ways of sharing the vertices out (benchmarks/bfs/main.cu:733-760 hash, :810-850 hash + coarse,
// :852-905 sixteen lanes per vertex, :961-1000 chunks; benchmarks/cc has the same set) ----
/*
 * The same relaxation as the kernels above, the vertices shared out as these variants of the reference do, with none of
 * the machinery around the group walk (no touching ahead, no pieces of long lists): a unit of lanes walks a vertex's
 * list through bam_ptr, and which vertex unit u takes is
 *   SHAPE 0  unit = wave:       v = u / nep + (u % nep) * stride, nep = (V + stride) / stride          (hash)
 *   SHAPE 1  unit = wave:       the `coarse` vertices c * coarse + j of c = u / nep + (u % nep) * stride,
 *                               nep = (V + stride * coarse) / (stride * coarse)                          (hash, coarse)
 *   SHAPE 2  unit = 16 lanes:   v as for SHAPE 0 (four vertices per wave side by side; the reference's page-cache
 *                               version of this kernel has an empty loop body, its in-memory twin has the relaxation)
 *   SHAPE 3  unit = wave:       the eight vertices 8 u .. 8 u + 7 one after the other                   (chunk)
 * The units of a launch are walked by a bounded number of waves (`n_units` are shared out round robin), so that the
 * pages the waves hold fit the cache.
 */
#define BAM_SHAPE_CHUNK 8
template <int SHAPE, typename Active, typename Visit>
__device__ __forceinline__ void walk_shaped(array_d_t<uint64_t>* da, const uint64_t* vertexList, const uint64_t n, const uint64_t coarse, const uint64_t stride,
                                            const uint64_t n_units, Active active, Visit visit)
{
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, n_threads = (uint64_t)gridDim.x * blockDim.x;
    bam_ptr<uint64_t> ptr(da);
    const uint64_t width = SHAPE == 2 ? 16 : BAM_WAVE_SIZE;
    const uint64_t l = tid % width;
    auto walk = [&](const uint64_t v) {
        const uint64_t start = vertexList[v], end = vertexList[v + 1];
        for (uint64_t i = (start & 0xFFFFFFFFFFFFFFF0ull) + l; i < end; i += width)
            if (i >= start) visit(v, ptr.read(i), i);
    };
    for (uint64_t u = tid / width; u < n_units; u += n_threads / width) {
        if (SHAPE == 3) {
            for (uint64_t v = u * BAM_SHAPE_CHUNK; v < (u + 1) * BAM_SHAPE_CHUNK && v < n; v++)
                if (active(v)) walk(v);
        } else if (SHAPE == 1) {
            const uint64_t nep = (n + stride * coarse) / (stride * coarse);
            const uint64_t c = u / nep + (u % nep) * stride;
            for (uint64_t j = 0; j < coarse; j++) {
                const uint64_t v = c * coarse + j;
                if (v < n && active(v)) walk(v);
            }
        } else {
            const uint64_t nep = (n + stride) / stride;
            const uint64_t v = u / nep + (u % nep) * stride;
            if (v < n && active(v)) walk(v);
        }
    }
}

template <int SHAPE>
__global__ __launch_bounds__(128) void k_bfs_shaped(array_d_t<uint64_t>* da, uint32_t* label, const uint32_t level, const uint64_t vertex_count, const uint64_t* vertexList,
                                                    uint64_t* changed, uint64_t coarse, uint64_t stride, uint64_t n_units)
{
    bool any = false;
    walk_shaped<SHAPE>(da, vertexList, vertex_count, coarse, stride, n_units,
                       [&](uint64_t v) { return label[v] == level; },
                       [&](uint64_t, uint64_t next, uint64_t) { if (label[next] == MYINFINITY) { label[next] = level + 1; any = true; } });
    if (any) *changed = 1;
}

// ---- BFS over a queue of the level's vertices (benchmarks/bfs/main.cu:409-451 kernel_frontier_coalesce_ptr_pc) ----
/* a vertex found for the first time (the exchange on its label decides who found it) goes to the next level's queue;
 * the lanes of a wave that found one at the same step take their places in it with one atomic */
__device__ __forceinline__ void bfs_frontier_visit(uint32_t* label, const uint32_t level, uint32_t* next_frontier, unsigned long long* next_size, const uint64_t next)
{
    if (label[next] != MYINFINITY) return;
    if (atomicExch(label + next, level + 1) != MYINFINITY) return;
    const uint64_t mask = bam::active_mask();
    const uint32_t leader = bam::first_lane(mask);
    unsigned long long pos = 0;
    if (bam::lane() == leader) pos = atomicAdd(next_size, (unsigned long long)bam::popc(mask));
    pos = bam::bcast((uint64_t)pos, leader);
    next_frontier[pos + bam::rank_in(mask)] = (uint32_t)next;
}

__global__ __launch_bounds__(128) BAM_GRAPH_KERNEL_WAVES void k_bfs_frontier_coalesce_ptr_pc(array_d_t<uint64_t>* da, uint32_t* label, const uint32_t level, const uint64_t* vertexList,
                                                                     const uint32_t* curr_frontier, const uint64_t curr_size, uint32_t* next_frontier,
                                                                     unsigned long long* next_size, uint64_t group,
                                                                     const heavy_piece_t* heavy, uint64_t n_heavy, unsigned long long* next_work, bool sorted)
{
    walk_item_groups<false>(da, vertexList, curr_size, group, heavy, n_heavy, next_work, false,
                            [&](uint64_t i, uint64_t& v) { v = curr_frontier[i]; return true; },
                            [&](uint64_t v) { return label[v] == level; },
                            [&](uint64_t, uint64_t next, uint64_t) { bfs_frontier_visit(label, level, next_frontier, next_size, next); },
                            nullptr, sorted);
}

/*
 * The queue of a level put in the order of its vertices.  A vertex enters a queue once, so the entries are distinct, and
 * sorting distinct numbers below V is marking them in a map of V bits and reading the map front to back: four small
 * kernels (mark; count the marks of every 4096 vertices, a wave each; running sums of those counts by one workgroup;
 * write the vertices out, a wave per 4096 again, and clear the map), a few microseconds a level for 2^24 vertices,
 * and no library.
 */
__global__ void k_queue_mark(const uint32_t* __restrict__ queue, const uint64_t n, unsigned long long* bits)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { const uint32_t v = queue[i]; atomicOr(&bits[v >> 6], 1ull << (v & 63u)); }
}
__global__ void k_bits_count(const unsigned long long* __restrict__ bits, const uint64_t n_words, uint32_t* totals)
{
    const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / BAM_WAVE_SIZE, at = wave * BAM_WAVE_SIZE + bam::lane();
    const uint64_t c = wave_sum((uint64_t)bam::popc(at < n_words ? bits[at] : 0ull));
    if (bam::lane() == 0 && wave * BAM_WAVE_SIZE < n_words) totals[wave] = (uint32_t)c;
}
/* totals[k] <- totals[0] + ... + totals[k - 1]; one workgroup of 1024 threads, a run of entries per thread */
__global__ void k_totals_scan(uint32_t* totals, const uint64_t n)
{
    __shared__ uint32_t sums[1024];
    const uint64_t per = (n + blockDim.x - 1) / blockDim.x, a = threadIdx.x * per, b = a + per < n ? a + per : n;
    uint32_t mine = 0;
    for (uint64_t k = a; k < b; k++) mine += totals[k];
    sums[threadIdx.x] = mine;
    __syncthreads();
    for (uint32_t o = 1; o < blockDim.x; o <<= 1) {
        const uint32_t add = threadIdx.x >= o ? sums[threadIdx.x - o] : 0;
        __syncthreads();
        sums[threadIdx.x] += add;
        __syncthreads();
    }
    uint32_t run = sums[threadIdx.x] - mine;
    for (uint64_t k = a; k < b; k++) { const uint32_t t = totals[k]; totals[k] = run; run += t; }
}
__global__ void k_bits_emit(unsigned long long* bits, const uint64_t n_words, const uint32_t* __restrict__ first_of_wave, uint32_t* out)
{
    const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / BAM_WAVE_SIZE, at = wave * BAM_WAVE_SIZE + bam::lane();
    if (wave * BAM_WAVE_SIZE >= n_words) return;
    unsigned long long w = at < n_words ? bits[at] : 0ull;
    if (w) bits[at] = 0;
    const uint32_t c = bam::popc(w);
    uint32_t incl = c;
#pragma unroll
    for (uint32_t o = 1; o < BAM_WAVE_SIZE; o <<= 1) {
        const uint32_t u = bam::shfl(incl, bam::lane() >= o ? bam::lane() - o : bam::lane());
        if (bam::lane() >= o) incl += u;
    }
    uint32_t pos = first_of_wave[wave] + incl - c;
    for (; w; w &= w - 1) out[pos++] = (uint32_t)(at * 64 + (uint64_t)__builtin_ctzll(w));
}

// ---- CC: min-label propagation (benchmarks/cc/main.cu:123-144, 595-617) ----
__device__ __forceinline__ void cc_compute(uint64_t cid, unsigned long long* comp, uint64_t next, bool* next_visit, bool* changed)
{
    const unsigned long long comp_src = comp[cid], comp_next = comp[next];
    if (comp_next == comp_src) return;
    uint64_t next_target;
    unsigned long long comp_target;
    if (comp_src < comp_next) { next_target = next; comp_target = comp_src; }
    else { next_target = cid; comp_target = comp_next; }
    atomicMin(&comp[next_target], comp_target);
    next_visit[next_target] = true;
    *changed = true;
}

/*
 * The same labels from one reading of the edges: comp[] as a forest in which every vertex points at a smaller one of its
 * component or at itself, the trees of the two ends of every edge joined by an exchange on the larger root, chains halved
 * on the way up (the hooking of J. Jaiganesh and M. Burtscher, "A High-Performance Connected Components Implementation for
 * GPUs", 2018), and a pass over the vertices that points each at its root, which is the smallest vertex of the component.
 * Propagating labels reads every list again whenever its vertex's label drops: bound by the store, as all of this is, it
 * took three readings of most of the edges and a short one (2^22 vertices, 8 entries each, half of the edges cached:
 * 16.6 ms and 133 000 pages from the store then, 6.6 ms and 34 500 now; all edges cached: 2.2 ms, along the pages 1.6).
 * A vertex that is not a root never becomes one again and what it points at only moves towards the root, so a word read a
 * while ago still names an ancestor, and the exchange, which goes by the word as it is, tells when it does not name a root.
 */
__device__ __forceinline__ unsigned long long cc_root(unsigned long long* comp, unsigned long long v)
{
    unsigned long long up = bam::ld_relaxed(comp + v);
    while (up != v) {
        const unsigned long long upper = bam::ld_relaxed(comp + up);
        if (upper == up) return up;
        bam::st_relaxed(comp + v, upper);
        v = upper;
        up = bam::ld_relaxed(comp + v);
    }
    return v;
}
/* the trees that u and v are in */
__device__ __forceinline__ void cc_join_trees(unsigned long long* comp, unsigned long long u, unsigned long long v)
{
    u = cc_root(comp, u); v = cc_root(comp, v);
    while (u != v) {
        if (u < v) { const unsigned long long t = u; u = v; v = t; }
        /* one lane of those that would exchange the same root's word as the first: exchanges on one address are performed one after the other */
        if (u == bam::first((uint64_t)u) && bam::lane() != bam::first_lane(bam::active_mask())) { u = cc_root(comp, u); continue; }
        const unsigned long long was = atomicCAS(comp + u, u, v);
        if (was == u) break;
        u = cc_root(comp, was);
    }
}
__device__ __forceinline__ void cc_join(unsigned long long* comp, const uint64_t a, const uint64_t b)
{
    /* most edges join what is joined already, and once the chains are short both ends name the same vertex: two loads side by side */
    const unsigned long long u = bam::ld_relaxed(comp + a), v = bam::ld_relaxed(comp + b);
    if (u != v) cc_join_trees(comp, u, v);
}
/*
 * Every vertex to the root of its tree, where trees are long: label propagation that was broken off leaves chains of as many steps as
 * the component is long, over how many it made.  A lane moves its own vertex alone, and always down; those with smaller numbers, which
 * it comes to, began earlier or at the same time, so that chains halve together.  Joined as they were, a path of 2^21 vertices took
 * 360 ms, since some waves walked down chains of vertices whose own waves had not begun; with this launch, 168 us there, 1.05.
 */
__global__ void k_cc_shorten(unsigned long long* comp, uint64_t vertex_count)
{
    const uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= vertex_count) return;
    unsigned long long up = bam::ld_relaxed(comp + v);
    for (;;) {
        const unsigned long long upper = bam::ld_relaxed(comp + up);
        if (upper == up) return;
        bam::st_relaxed(comp + v, upper);
        up = upper;
    }
}
/*
 * The forest that the joins begin with, from the first BAM_CC_FIRST neighbours of lists, as far as those lie in one page that is resident.  First
 * (ROUND false, all vertices) each vertex is put under the smallest of its own, if that is smaller than itself: no exchange, and no
 * tree that another wave is joining meanwhile.  Then, with trees shortened (k_cc_shorten), rounds over every `each`-th vertex point the
 * larger root of an entry's two ends at the smaller one, by a minimum that nobody waits for: of several for one root the smallest stays, and
 * what the others would have joined is joined when the edges are read, as all are.  What makes a reading of the edges slow is
 * that most of them meet on a few roots which are being joined, each exchange waiting for the others on its word; with nearly all of a component
 * under one root before it begins, both ends of most name that.
 *   Uniform random graphs, 8 entries a vertex, all cached, medians in us of two graphs before, with one launch of the first kind and with three rounds: 2^14 vertices 99 149, 158, 76
 * 74; 2^16 237 269, 378, 92 93; 2^17 670 406, 890, 121 111; 2^18 378 605, 638, 154 161; 2^19 362 885, 635, 254 258; 2^20 399 560, 606, 369 371; half
 * cached 2^19 819 1349, 901, 653 655, 2^22 3950 3788, 4042, 3806 3806, within 1 % from call to call instead of 20.  From 2^21 vertices on, all cached, two
 * rounds: 620 840 -> 577 575 (three 630 628), 2^22 1198 1124 -> 1116 1146.  Power-law 2^16, 2^18, 2^20 126, 217, 559 -> 73, 137, 381; grids of
 * 64 x 4096, 1024 x 1024, 2048 x 2048 454, 825, 902 -> 77, 184, 525; a path of 2^21 723 -> 281.  Rounds over all vertices: 2^17 229, 2^22 1535.
 */
#define BAM_CC_FIRST 4
template <bool ROUND>
__global__ __launch_bounds__(256) void k_cc_begin(array_d_t<uint64_t>* da, const uint64_t* offsets, const uint64_t n_vertices, unsigned long long* comp, const uint32_t each)
{
    const uint64_t v = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * (ROUND ? each : 1u);
    bam::range_view<uint64_t> view;
    view.load(da->d_ranges);
    if (v >= n_vertices) return;
    const uint64_t e = offsets[v], end = offsets[v + 1];
    unsigned long long up = ROUND ? bam::ld_relaxed(comp + v) : v;
    if (e < end && end <= view.index_end) {
        const uint64_t byte = view.byte_of(e);
        const uint32_t in_page = (uint32_t)byte & (view.page_size - 1), here = (view.page_size - in_page) / (uint32_t)sizeof(uint64_t);
        const uint32_t n = end - e < here ? (uint32_t)(end - e) : here;
        const data_page_t* const dp = view.pages + (byte >> view.page_size_log);
        const uint64_t was = __hip_atomic_load((const uint64_t*)dp, __ATOMIC_RELAXED, BAM_AGENT);
        if (((uint32_t)was >> (CNT_SHIFT + 1)) == V_NB) {
            const uint64_t* at[BAM_CC_FIRST];
            uint64_t x[BAM_CC_FIRST];
            /* (the first entry again where there are fewer) */
#pragma unroll
            for (uint32_t j = 0; j < BAM_CC_FIRST; j++) at[j] = (const uint64_t*)(view.slot_addr((uint32_t)(was >> 32) & BAM_SLOT_MASK) + in_page) + (j < n ? j : 0);
            bam::ld_payload_nt(at, x);
            if (((__hip_atomic_load((const uint64_t*)dp, __ATOMIC_RELAXED, BAM_AGENT) ^ was) & 0xFFFFFFFFC0000000ull) == 0) {
                if constexpr (!ROUND) {
#pragma unroll
                    for (uint32_t j = 0; j < BAM_CC_FIRST; j++) up = x[j] < up ? x[j] : up;
                } else {
                    unsigned long long high[BAM_CC_FIRST], low[BAM_CC_FIRST];
#pragma unroll
                    for (uint32_t j = 0; j < BAM_CC_FIRST; j++) high[j] = bam::ld_relaxed(comp + x[j]);
#pragma unroll
                    for (uint32_t j = 0; j < BAM_CC_FIRST; j++) { low[j] = high[j] < up ? high[j] : up; high[j] = high[j] < up ? up : high[j]; }
#pragma unroll
                    for (uint32_t j = 0; j < BAM_CC_FIRST; j++)
                        if (low[j] != high[j] && bam::ld_relaxed(comp + high[j]) > low[j]) __hip_atomic_fetch_min(comp + high[j], low[j], __ATOMIC_RELAXED, BAM_AGENT);
                }
            }
        }
    }
    if constexpr (!ROUND) bam::st_relaxed(comp + v, up);
}
/* n_missing, next_chunk: along_t's, of the reading before, which are zero between sweeps (NULL: it had none) */
__global__ void k_cc_settle(unsigned long long* comp, uint64_t vertex_count, unsigned long long* n_missing, unsigned long long* next_chunk)
{
    const uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v == 0 && n_missing) *n_missing = *next_chunk = 0;
    if (v >= vertex_count) return;
    unsigned long long r = v;
    for (unsigned long long up = bam::ld_relaxed(comp + r); up != r; up = bam::ld_relaxed(comp + r)) r = up;
    bam::st_relaxed(comp + v, r);
}

__global__ __launch_bounds__(128) BAM_GRAPH_KERNEL_WAVES void k_cc_coalesce_coarse_ptr_pc(array_d_t<uint64_t>* da, uint64_t vertex_count, const uint64_t* vertexList, unsigned long long* comp,
                                                                  uint64_t coarse, const heavy_piece_t* heavy, uint64_t n_heavy, unsigned long long* next_work, bool backwards)
{
    walk_vertex_groups(da, vertexList, vertex_count, coarse, heavy, n_heavy, next_work, backwards,
                       [&](uint64_t) { return true; },
                       [&](uint64_t v, uint64_t next, uint64_t) { cc_join(comp, v, next); });
}

template <int SHAPE>
__global__ __launch_bounds__(128) void k_cc_shaped(array_d_t<uint64_t>* da, bool* curr_visit, bool* next_visit, uint64_t vertex_count, const uint64_t* vertexList,
                                                   unsigned long long* comp, bool* changed, uint64_t coarse, uint64_t stride, uint64_t n_units)
{
    walk_shaped<SHAPE>(da, vertexList, vertex_count, coarse, stride, n_units,
                       [&](uint64_t v) { return curr_visit[v]; },
                       [&](uint64_t v, uint64_t next, uint64_t) { cc_compute(v, comp, next, next_visit, changed); });
}

// ---- BFS / CC by edge page (benchmarks/bfs/main.cu:1074-1140 kernel_optimized_ptr_pc, first-vertex table :122-181) ----
/*
 * first[p], p = 0 .. n_pages: the vertex whose edge list holds edge p * epp (the last vertex with
 * offsets[v] <= p * epp); first[n_pages] = V - 1.  The vertices with edges on page p are first[p] .. first[p + 1].
 */
__global__ void k_page_first_vertex(const uint64_t* offsets, uint64_t n_vertices, uint64_t epp, uint64_t n_pages, uint64_t* first)
{
    const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p > n_pages) return;
    const uint64_t e = p * epp;
    uint64_t lo = 0, hi = n_vertices + 1;            /* first index with offsets[idx] > e */
    while (lo < hi) {
        const uint64_t mid = (lo + hi) >> 1;
        if (offsets[mid] > e) hi = mid; else lo = mid + 1;
    }
    uint64_t v = lo ? lo - 1 : 0;
    if (v >= n_vertices) v = n_vertices - 1;
    first[p] = v;
}

/*
 * For PageRank, and for BFS and components where a page is larger than 64 KiB (else k_along_resident; components also as cc_read_edges has it):
 * one wave, `ppw` consecutive pages of the edge array per trip (lane l looks after page l of the trip), trips
 * handed out wave by wave along the array.  A page is wanted when one of its vertices is active; the wanted pages
 * of a trip are taken with one acquire, so their misses go to the store as one batch of commands, and the whole
 * wave then walks the active vertices of each page, 64 edges at a time, before the references are dropped.
 * A wave holds at most `ppw` pages at a time; the launch keeps waves x ppw under half the cache.
 */
template <typename Active, typename Visit>
__device__ __forceinline__ void graph_by_page(array_d_t<uint64_t>* da, const uint64_t* offsets, const uint64_t* first, const uint64_t n_edges,
                                              const uint32_t ppw, const bool backwards, Active active, Visit visit)
{
    const uint32_t lane = bam::lane();
    const uint64_t wave = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / BAM_WAVE_SIZE;
    const uint64_t n_waves = (uint64_t)gridDim.x * blockDim.x / BAM_WAVE_SIZE;
    bam::range_view<uint64_t> view;
    view.load(da->d_ranges);
    const uint32_t epp = view.page_size / 8;
    const uint64_t n_pages = (n_edges + epp - 1) / epp;
    const uint64_t pso_pages = view.pso >> view.page_size_log;
    const uint64_t n_trips = (n_pages + ppw - 1) / ppw;
    for (uint64_t t = wave; t < n_trips; t += n_waves) {
        /* every other sweep runs from the far end: what the last sweep left in the cache is what this one asks for first */
        const uint64_t p0 = (backwards ? n_trips - 1 - t : t) * ppw;
        const uint64_t p = p0 + lane;
        /* which pages of the trip hold entries of an active vertex: the lanes go over the trip's vertices side by side
         * (their flags and offsets are consecutive in memory) and mark the pages each active list covers */
        const uint64_t p_end = p0 + ppw < n_pages ? p0 + ppw : n_pages;
        const uint64_t trip_start = p0 * epp, trip_end = p_end * epp < n_edges ? p_end * epp : n_edges;
        uint64_t marks = 0;
        for (uint64_t vbase = first[p0], v_last = first[p_end]; vbase <= v_last; vbase += BAM_WAVE_SIZE) {
            const uint64_t v = vbase + lane;
            if (v <= v_last && active(v)) {
                uint64_t es = offsets[v], ee = offsets[v + 1];
                if (es < trip_start) es = trip_start;
                if (ee > trip_end) ee = trip_end;
                if (ee > es) marks |= (~0ull >> (63 - (ee - 1 - trip_start) / epp)) & (~0ull << ((es - trip_start) / epp));
            }
        }
#pragma unroll
        for (uint32_t o = BAM_WAVE_SIZE / 2; o; o >>= 1) marks |= bam::shfl(marks, lane ^ o);
        const bool want = ((marks >> lane) & 1) != 0;
        uint64_t va = 0, vb = 0;
        if (want) { va = first[p]; vb = first[p + 1]; }
        /* those that can be had without waiting are walked and given back before the others are waited for; a page whose wait was given up (the
         * controller is marked aborted) is not walked */
        for (bool left = want; bam::ballot(left);) {
            uint32_t slot;
            /* the lanes without a page of their own come along and help move what the others load */
            const bool in = view.acquire_some(p + pso_pages, left, slot);
            if (!bam::ballot(in)) break;
            left = left && !in;
            for (uint64_t m = bam::ballot(in); m; m &= m - 1) {
                const uint32_t j = bam::first_lane(m);
                const uint64_t va_j = bam::bcast(va, j), vb_j = bam::bcast(vb, j);
                const uint64_t ps = (p0 + j) * epp, pe = ps + epp < n_edges ? ps + epp : n_edges;
                const uint64_t* payload = (const uint64_t*)view.slot_addr(bam::bcast(slot, j));
                for (uint64_t vbase = va_j; vbase <= vb_j; vbase += BAM_WAVE_SIZE) {
                    const uint64_t v = vbase + lane;
                    uint64_t es = 0, ee = 0;
                    if (v <= vb_j && active(v)) {
                        es = offsets[v]; ee = offsets[v + 1];
                        if (es < ps) es = ps;
                        if (ee > pe) ee = pe;
                    }
                    if (ee < es) ee = es;
                    walk_packed(es, ee, v, [&](uint64_t i) { return bam::ld_payload(payload + (i - ps)); }, visit);
                }
            }
            if (in) bam_release_refs(view.pages + p + pso_pages, 1, false);
        }
    }
    view.flush_stats();
}

__global__ __launch_bounds__(64) void k_bfs_by_page(array_d_t<uint64_t>* da, uint32_t* label, const uint32_t level, const uint64_t* offsets,
                                                     const uint64_t* first, uint64_t n_edges, uint32_t ppw, uint64_t* changed)
{
    bool any = false;
    graph_by_page(da, offsets, first, n_edges, ppw, (level & 1u) != 0,
                  [&](uint64_t v) { return label[v] == level; },
                  [&](uint64_t, uint64_t next, uint64_t) { if (label[next] == MYINFINITY) { label[next] = level + 1; any = true; } });
    if (any) *changed = 1;
}

__global__ __launch_bounds__(64) void k_cc_sweep_by_page(array_d_t<uint64_t>* da, bool* curr_visit, bool* next_visit, const uint64_t* offsets,
                                                          const uint64_t* first, uint64_t n_edges, uint32_t ppw, unsigned long long* comp, bool* changed)
{
    graph_by_page(da, offsets, first, n_edges, ppw, false,
                  [&](uint64_t v) { return curr_visit[v]; },
                  [&](uint64_t src, uint64_t next, uint64_t) { cc_compute(src, comp, next, next_visit, changed); });
}

__global__ __launch_bounds__(64) void k_cc_by_page(array_d_t<uint64_t>* da, const uint64_t* offsets, const uint64_t* first, uint64_t n_edges, uint32_t ppw, bool backwards,
                                                    unsigned long long* comp)
{
    graph_by_page(da, offsets, first, n_edges, ppw, backwards,
                  [&](uint64_t) { return true; },
                  [&](uint64_t src, uint64_t next, uint64_t) { cc_join(comp, src, next); });
}

// ---- BFS / CC along the edge array, what is resident first ----
/*
 * A reading of the edge array in two launches.  The first visits the pages that are wanted and resident, and lists the
 * wanted ones that are not; the second fetches those in batches of up to 64 commands and visits them.  Front to back,
 * whatever is resident, a sweep over an array larger than its cache pushes out what it has not reached yet: of 27 800
 * cached and wanted pages of 118 000 (2^21 vertices, a power-law graph) it found 1 000.  The list also makes every batch
 * but the last a whole one whichever pages are wanted, where a wave that looks after a run of neighbouring pages sends as many
 * commands as the cache has pages for each wave (seven there, 9 M pages/s; batches of 64 reach 13).
 *
 * Both launches take a segment at a time: 512 entries, eight rows of 64, one per lane and row, all loaded before any is
 * used; which entries are to be visited, and for which vertex, is worked out in LDS while they are on their way.  The
 * pages are referenced meanwhile (a take and a drop per page and wave; a page is 512 entries).
 * Bound by the store where edges are missing: BFS of that graph 19.2 -> 10.9 ms (175 000 -> 124 000 page reads, 11.6 M a second), and 9.0
 * (98 000) with the slots used again; with 2^18 vertices 4.8 -> 1.6; components of 2^22 vertices, 8 entries each, half cached, 4.7 -> 3.8.  All cached, by the
 * trips to memory a wave makes one after the other: BFS of 2^20 vertices 1.65 -> 0.47 ms, components of 2^22 1.55 -> 1.2.
 */
#define BAM_SEG_ROWS 8u
#define BAM_SEG_EDGES (BAM_SEG_ROWS * BAM_WAVE_SIZE)
#define BAM_ALL_ROWS ((1u << BAM_SEG_ROWS) - 1u)
#define BAM_TRIP_SEGS 16u
#define BAM_TRIP_WAVES 4u                       /* waves to a workgroup of the first launch: they share an add to the list */
struct along_t {
    const uint64_t* offsets;                    /* [n_vertices + 1] */
    uint64_t n_vertices;
    const uint64_t* first;                      /* [n_segs + 1] the vertex whose list holds the segment's first entry */
    uint64_t n_edges, n_pages, n_segs;          /* of the array, which may hold more than the lists */
    uint32_t seg_log;                           /* log2 of the segments in a page, at most that of BAM_TRIP_SEGS (0 where a page is less than one) */
    uint32_t part_log;                          /* log2 of the pages in a segment (0 where a page is one or more) */
    uint32_t trip_segs;                         /* segments a wave of the first launch looks after: whole pages, BAM_TRIP_SEGS at most */
    uint32_t* missing;                          /* [n_pages] the pages the first launch leaves to the second */
    unsigned long long* n_missing;              /* zero between sweeps, like the next one */
    unsigned long long* next_chunk;             /* of the list, for the waves of the second launch */
    uint64_t* ahead;                            /* [n_segs * BAM_SEG_ROWS] a bit per entry (bfs_along) */
    unsigned long long* flags;                  /* [2] what the sweep tells the host, and the sweeps queued behind it */
    const unsigned long long* stretches;        /* not 0: a stretch of the array to each workgroup (k_cc_look); NULL: by turns */
    /* the sweep is made if it is sure to be wanted, or if one of these words, NULL or an earlier sweep's, says so */
    uint32_t sure;
    const unsigned long long* gate[2];
};
__device__ __forceinline__ void raise_flag(unsigned long long* flag, const bool mine)
{
    const uint64_t m = bam::ballot(mine);
    if (m && bam::lane() == bam::first_lane(m) && bam::ld_relaxed(flag) == 0) bam::st_relaxed(flag, 1ull);
}

/*
 * Whose lists the entries of a segment are in, found from the entries, where the vertices between its first and its last list are too
 * many to be gone over: a run of vertices without lists lies in one segment whatever its length, and one wave has it.  (2^17 entries,
 * half of them among the first vertices of 2^26 and half among the last: BFS, 8 levels, 867 ms gone over, 0.28 looked up, 1.06 over
 * queues of vertices.)  The owner of entry e0 + 64 r + lane, r = r0 and r0 + 1, is v0 + at[r - r0]: the last of the vertices
 * v0 .. v0 + span whose list begins there or before; only of use for entries of [offsets[0], offsets[V]).  Two searches side by side:
 * four took 20 registers more, which every other sweep would pay for.
 *   From how many vertices to a segment on: entries scattered over 2^13, 2^14, 2^15, 2^16 vertices a segment, levels (gone over 256 at a
 * time) 95, 140, 236, 571 us and looked up 135, 213, 314, 428; joins (64 at a time) 223, 408, 715, 1273 and 198, 329, 527, 838, with 2^12
 * the same.
 */
#define BAM_SEG_SPAN_LEVELS 32768u
#define BAM_SEG_SPAN_JOINS 4096u
__device__ __forceinline__ void segment_owners(const uint64_t* offsets, const uint64_t v0, const uint64_t span, const uint64_t e0, const uint32_t r0, uint64_t (&at)[2])
{
    const uint64_t* const from = offsets + v0;
    const uint64_t e = e0 + r0 * BAM_WAVE_SIZE + bam::lane();
#pragma unroll
    for (uint32_t r = 0; r < 2; r++) at[r] = 0;
#pragma unroll 1
    for (uint64_t len = span + 1; len > 1; len -= len / 2)
#pragma unroll
        for (uint32_t r = 0; r < 2; r++)
            if (from[at[r] + len / 2] <= e + r * BAM_WAVE_SIZE) at[r] += len / 2;
}

/*
 * One level of BFS.  AHEAD: the entries of vertices found on this very level are visited along with those of the level
 * itself where their page is at hand anyway; the neighbours they find are two levels on, as far as is known (somebody nearer
 * may still be looking at them, hence the minimum), and are not visited from before the next level, when their labels are
 * settled.  A bit per entry says that it has been visited ahead of its level, so that the next one does not bring the page in for
 * it: 43 300 page reads instead of 34 200 without it on a 2^19-vertex power-law graph, a quarter of the edges cached.  The bits of
 * a segment are those of the last sweep that visited it: of older levels' entries nobody asks.
 */
template <bool AHEAD>
struct bfs_along {
    uint32_t* label;
    uint32_t level;
    static constexpr bool joins = false;
    static constexpr bool again = AHEAD;       /* a page that is visited on one level is likely to be wanted on the next */
    struct lds_t { unsigned long long now[BAM_TRIP_SEGS * BAM_SEG_ROWS], next[AHEAD ? BAM_TRIP_SEGS * BAM_SEG_ROWS : 1]; };

    static __device__ __forceinline__ void mark(unsigned long long* bits, const uint32_t a, const uint32_t b, const bool mine)      /* entries [a, b), b > a where mine */
    {
        const uint32_t lane = bam::lane(), wa = a / BAM_WAVE_SIZE, wb = mine ? (b - 1) / BAM_WAVE_SIZE : wa;
        const bool wide = mine && wb - wa >= 4;
        if (mine && !wide)
            for (uint32_t w = wa; w <= wb; w++)
                atomicOr(bits + w, (w == wa ? ~0ull << (a % BAM_WAVE_SIZE) : ~0ull) & (w == wb ? ~0ull >> (63 - (b - 1) % BAM_WAVE_SIZE) : ~0ull));
        for (uint64_t m = bam::ballot(wide); m; m &= m - 1) {
            const uint32_t j = bam::first_lane(m), ja = bam::bcast(a, j), jb = bam::bcast(b, j) - 1;
            for (uint32_t w = ja / BAM_WAVE_SIZE + lane; w <= jb / BAM_WAVE_SIZE; w += BAM_WAVE_SIZE)
                atomicOr(bits + w, (w == ja / BAM_WAVE_SIZE ? ~0ull << (ja % BAM_WAVE_SIZE) : ~0ull) & (w == jb / BAM_WAVE_SIZE ? ~0ull >> (63 - jb % BAM_WAVE_SIZE) : ~0ull));
        }
    }
    /* which of the n_segs segments from seg0 on are wanted; s is ready for visit() of any of them */
    __device__ __forceinline__ uint32_t prepare(const along_t& g, lds_t& s, const uint64_t seg0, const uint32_t n_segs) const
    {
        const uint32_t lane = bam::lane(), n_words = n_segs * BAM_SEG_ROWS;
        wave_lds_fence();                       /* what was read there before has been read */
        for (uint32_t w = lane; w < n_words; w += BAM_WAVE_SIZE) { s.now[w] = 0; if (AHEAD) s.next[w] = 0; }
        wave_lds_fence();
        const uint64_t e0 = seg0 * BAM_SEG_EDGES, e1 = e0 + n_segs * BAM_SEG_EDGES < g.n_edges ? e0 + n_segs * BAM_SEG_EDGES : g.n_edges;
        const uint64_t v_last = g.first[seg0 + n_segs];
        const uint64_t v_first = g.first[seg0];
        const bool few_lists = v_last - v_first > (uint64_t)n_segs * BAM_SEG_SPAN_LEVELS;
        if (few_lists) {
#pragma unroll 1
            for (uint32_t r0 = 0; r0 < n_words; r0 += 2) {
                const uint64_t seg = seg0 + r0 / BAM_SEG_ROWS, v0 = g.first[seg];
                uint64_t at[2];
                segment_owners(g.offsets, v0, g.first[seg + 1] - v0, e0, r0, at);
#pragma unroll
                for (uint32_t r = 0; r < 2; r++) {
                    const uint64_t e = e0 + (r0 + r) * BAM_WAVE_SIZE + lane;
                    const uint32_t l = e >= g.offsets[0] && e < g.offsets[g.n_vertices] ? bam::ld_relaxed(label + v0 + at[r]) : MYINFINITY;
                    const uint64_t now = bam::ballot(l == level), next = AHEAD ? bam::ballot(l == level + 1) : 0ull;
                    if (lane == 0) { s.now[r0 + r] = now; if (AHEAD) s.next[r0 + r] = next; }
                }
            }
        }
        for (uint64_t vbase = few_lists ? v_last + 1 : v_first; vbase <= v_last; vbase += 4 * BAM_WAVE_SIZE) {
            /* four vertices to a lane at a time: most sweeps find few or none of their level, and are the trips of these loads */
            uint32_t l[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; q++) { const uint64_t v = vbase + q * BAM_WAVE_SIZE + lane; l[q] = v <= v_last ? bam::ld_relaxed(label + v) : MYINFINITY; }
#pragma unroll
            for (uint32_t q = 0; q < 4; q++) {
                const uint64_t v = vbase + q * BAM_WAVE_SIZE + lane;
                bool mine = l[q] == level || (AHEAD && l[q] == level + 1);
                if (!bam::ballot(mine)) continue;
                uint64_t es = 0, ee = 0;
                if (mine) { es = g.offsets[v]; ee = g.offsets[v + 1]; }
                if (es < e0) es = e0;
                if (ee > e1) ee = e1;
                mine = mine && ee > es;
                const uint32_t a = (uint32_t)(es - e0), b = (uint32_t)(ee - e0);
                mark(s.now, a, b, mine && l[q] == level);
                if (AHEAD) mark(s.next, a, b, mine && l[q] != level);
            }
        }
        wave_lds_fence();
        uint64_t any = 0;                       /* bit k: word 64 q + k of turn q is not empty; a segment is a byte of it */
        uint32_t wanted = 0;
        for (uint32_t w0 = 0; w0 < n_words; w0 += BAM_WAVE_SIZE) {
            const uint32_t w = w0 + lane;
            unsigned long long now = w < n_words ? s.now[w] : 0ull;
            if constexpr (AHEAD) {
                const unsigned long long next = w < n_words ? s.next[w] : 0ull;
                if (now | next) {
                    const unsigned long long seen = g.ahead[seg0 * BAM_SEG_ROWS + w];
                    now &= ~seen;
                    s.now[w] = now;
                    s.next[w] = next & ~seen;
                }
            }
            any = bam::ballot(now != 0);
            for (uint32_t k = 0; k < BAM_WAVE_SIZE / BAM_SEG_ROWS; k++)
                if ((any >> (k * BAM_SEG_ROWS)) & ((1u << BAM_SEG_ROWS) - 1u)) wanted |= 1u << (w0 / BAM_SEG_ROWS + k);
        }
        wave_lds_fence();
        return wanted;
    }
    /* whether entries of rows [row, row + n) of those prepared are wanted */
    __device__ __forceinline__ bool wants(const along_t&, lds_t& s, const uint64_t, const uint32_t row, const uint32_t n) const
    {
        unsigned long long any = 0;
        for (uint32_t r = 0; r < n; r++) any |= s.now[row + r];
        return any != 0;
    }
    /* the entries of the segment, the k-th of those prepared: lane l holds entry 64 r + l in id[r]; of the rows that `rows` has a bit for */
    __device__ __forceinline__ void visit(const along_t& g, lds_t& s, const uint64_t seg, const uint32_t k, const uint64_t (&id)[BAM_SEG_ROWS], bool& found, bool& found_ahead,
                                          const uint32_t rows = BAM_ALL_ROWS) const
    {
        const uint32_t lane = bam::lane();
        uint32_t have[BAM_SEG_ROWS];
        unsigned long long all[BAM_SEG_ROWS], next[BAM_SEG_ROWS];
#pragma unroll
        for (uint32_t r = 0; r < BAM_SEG_ROWS; r++) {
            next[r] = AHEAD ? bam::first((uint64_t)s.next[k * BAM_SEG_ROWS + r]) : 0ull;
            all[r] = bam::first((uint64_t)s.now[k * BAM_SEG_ROWS + r]) | next[r];
            if (!((rows >> r) & 1)) all[r] = 0;
            have[r] = 0;
            if ((all[r] >> lane) & 1) have[r] = bam::ld_relaxed(label + id[r]);
        }
#pragma unroll
        for (uint32_t r = 0; r < BAM_SEG_ROWS; r++) {
            const bool on = AHEAD && ((next[r] >> lane) & 1);
            const uint32_t to = level + 1u + (on ? 1u : 0u);
            if (have[r] > to) {                 /* (zero where the lane has nothing to visit) */
                if (AHEAD) __hip_atomic_fetch_min(label + id[r], to, __ATOMIC_RELAXED, BAM_AGENT);
                else bam::st_relaxed(label + id[r], to);
                found |= !on; found_ahead |= on;
            }
        }
        if (AHEAD && lane < BAM_SEG_ROWS && ((rows >> lane) & 1)) g.ahead[seg * BAM_SEG_ROWS + lane] = s.next[k * BAM_SEG_ROWS + lane];
    }
};

/* connected components: every entry of a list is visited once, with the vertex whose list it is in.  What the array holds before
 * the first list and behind the last is nobody's neighbour, and need not be the number of a vertex. */
struct cc_along {
    unsigned long long* comp;
    static constexpr bool joins = true;
    static constexpr bool again = false;       /* every page once */
    struct lds_t { unsigned long long starts[BAM_SEG_ROWS]; uint32_t vertex[BAM_SEG_EDGES]; };      /* where lists begin; whose, from the segment's first vertex on */
    __device__ __forceinline__ uint32_t prepare(const along_t& g, lds_t&, const uint64_t seg0, const uint32_t n_segs) const
    {
        const uint64_t begin = g.offsets[0], end = g.offsets[g.n_vertices];
        uint32_t wanted = 0;
        for (uint32_t k = 0; k < n_segs; k++)
            if ((seg0 + k) * BAM_SEG_EDGES < end && (seg0 + k + 1) * BAM_SEG_EDGES > begin) wanted |= 1u << k;
        return wanted;
    }
    __device__ __forceinline__ bool wants(const along_t& g, lds_t&, const uint64_t seg0, const uint32_t row, const uint32_t n) const
    {
        const uint64_t e = seg0 * BAM_SEG_EDGES + row * BAM_WAVE_SIZE;
        return e < g.offsets[g.n_vertices] && e + n * BAM_WAVE_SIZE > g.offsets[0];
    }
    __device__ __forceinline__ void visit(const along_t& g, lds_t& s, const uint64_t seg, const uint32_t, const uint64_t (&id)[BAM_SEG_ROWS], bool&, bool&,
                                          const uint32_t rows = BAM_ALL_ROWS) const
    {
        const uint32_t lane = bam::lane();
        const uint64_t e0 = seg * BAM_SEG_EDGES, begin_all = g.offsets[0], end_all = g.offsets[g.n_vertices];
        const uint64_t e1 = e0 + BAM_SEG_EDGES < end_all ? e0 + BAM_SEG_EDGES : end_all;
        const uint64_t v0 = g.first[seg], v_last = g.first[seg + 1];
        wave_lds_fence();
        const bool few_lists = v_last - v0 > BAM_SEG_SPAN_JOINS;      /* every entry is taken for the beginning of its list */
        if (lane < BAM_SEG_ROWS) s.starts[lane] = few_lists ? ~0ull : lane ? 0ull : 1ull;
        if (lane == 0) s.vertex[0] = 0;
        wave_lds_fence();
        if (few_lists)
#pragma unroll 1
            for (uint32_t r0 = 0; r0 < BAM_SEG_ROWS; r0 += 2) {
                uint64_t at[2];
                segment_owners(g.offsets, v0, v_last - v0, e0, r0, at);
#pragma unroll
                for (uint32_t r = 0; r < 2; r++) s.vertex[(r0 + r) * BAM_WAVE_SIZE + lane] = (uint32_t)at[r];
            }
        for (uint64_t vbase = few_lists ? v_last + 1 : v0 + 1; vbase <= v_last; vbase += BAM_WAVE_SIZE) {
            const uint64_t v = vbase + lane;
            uint64_t es = 0, ee = 0;
            if (v <= v_last) { es = g.offsets[v]; ee = g.offsets[v + 1]; }
            if (ee > es && es >= e0 && es < e1) {
                const uint32_t a = (uint32_t)(es - e0);
                s.vertex[a] = (uint32_t)(v - v0);
                atomicOr(s.starts + a / BAM_WAVE_SIZE, 1ull << (a % BAM_WAVE_SIZE));
            }
        }
        wave_lds_fence();
        uint32_t begin = 0;                     /* the last list that begins before the row */
        unsigned long long u[BAM_SEG_ROWS], w[BAM_SEG_ROWS];
        /* most entries join what is joined already, and once the chains are short both ends name the same vertex: the loads
         * of all rows side by side.  A word read a while ago still names an ancestor. */
#pragma unroll
        for (uint32_t r = 0; r < BAM_SEG_ROWS; r++) {
            const uint64_t m = bam::first((uint64_t)s.starts[r]), below = m & (~0ull >> (63 - lane));
            const uint64_t src = v0 + s.vertex[below ? r * BAM_WAVE_SIZE + 63u - (uint32_t)__builtin_clzll(below) : begin];
            if (m) begin = r * BAM_WAVE_SIZE + 63u - (uint32_t)__builtin_clzll(m);
            u[r] = w[r] = 0;
            const uint64_t e = e0 + r * BAM_WAVE_SIZE + lane;
            if (((rows >> r) & 1) && e >= begin_all && e < e1) { u[r] = bam::ld_relaxed(comp + src); w[r] = bam::ld_relaxed(comp + id[r]); }
        }
#pragma unroll
        for (uint32_t r = 0; r < BAM_SEG_ROWS; r++) {
            /* the rows before may have joined these two (or given what they name a parent): all cached, 1.56 -> 1.45 ms */
            if (r && u[r] != w[r]) { u[r] = bam::ld_relaxed(comp + u[r]); w[r] = bam::ld_relaxed(comp + w[r]); }
            if (u[r] != w[r]) cc_join_trees(comp, u[r], w[r]);
        }
    }
};

/* Whether the graph's neighbours lie side by side, as far as its array is resident: 256 entries are looked at, and of most the two ends
 * are less than a 64th of the vertices apart.  (A path, a grid of any but the widest rows; by chance, one entry in 32.) */
__global__ __launch_bounds__(256) void k_cc_look(array_d_t<uint64_t>* da, const along_t g, unsigned long long* stretches)
{
    bam::range_view<uint64_t> view;
    view.load(da->d_ranges);
    const uint64_t begin = g.offsets[0], end = g.offsets[g.n_vertices];
    if (begin >= end) { if (threadIdx.x == 0) *stretches = 0; return; }
    const uint64_t e = begin + (end - begin) / 512 * (2 * threadIdx.x + 1), seg = e / BAM_SEG_EDGES;
    uint64_t id = 0;
    const bool there = bam_read_unpinned(view.pages + (view.pso >> view.page_size_log) + ((e << 3) >> view.page_size_log), view.slot_addr(0), view.page_size_log, (e << 3) & (view.page_size - 1), id);
    const uint64_t low = g.first[seg], high = g.first[seg + 1];
    const bool near = there && (id < low ? low - id : id > high ? id - high : 0ull) < (g.n_vertices + 63) / 64;
    const int n_there = __syncthreads_count(there), n_near = __syncthreads_count(near);
    if (threadIdx.x == 0) *stretches = 2 * n_near > n_there;
}

/*
 * Pages of less than a segment: those of one segment that a wave holds (bit q of `held`: its q-th, in slot `slot` of lane lane0 + q; one at least)
 * are visited together, since where the lists begin is worked out for all of it.  The rows of the others are loaded
 * from a page that is held, and not looked at.  Pages of 512 bytes, 2^20 vertices of a power-law graph, all, a half and a quarter of the edges
 * cached, by page and by vertex, ms: levels 1.63, 9.5, 11.8 and 4.6, 48.7, 61.0 -> 0.42, 3.9, 6.1; components of 2^21 vertices of a uniform one,
 * a half and a quarter, 3.7, 4.6 and 20.2, 9.7 -> 2.4, 4.2.
 */
template <typename A>
__device__ __forceinline__ void visit_parts(const A& algo, const along_t& g, typename A::lds_t& s, const bam::range_view<uint64_t>& view, const uint64_t seg, const uint32_t k,
                                            const uint64_t held, const uint32_t lane0, const uint32_t slot, bool& found, bool& found_ahead)
{
    const uint32_t row_log = 3u - g.part_log, lane = bam::lane();          /* log2 of the rows in a page */
    static_assert(BAM_SEG_ROWS == 8u, "eight rows to a segment");
    uint64_t id[BAM_SEG_ROWS];
    uint32_t rows = 0;
#pragma unroll
    for (uint32_t r = 0; r < BAM_SEG_ROWS; r++) {
        const uint32_t q = r >> row_log;
        const bool in = ((held >> q) & 1) != 0;
        rows |= in ? 1u << r : 0u;
        id[r] = bam::ld_payload((const uint64_t*)view.slot_addr(bam::bcast(slot, lane0 + (in ? q : bam::first_lane(held)))) + (r & ((1u << row_log) - 1u)) * BAM_WAVE_SIZE + lane);
    }
    algo.visit(g, s, seg, k, id, found, found_ahead, rows);
}

/* a workgroup takes trips of 16 segments at most, a wave each, until there are none left */
template <typename A, bool PARTS>
__global__ __launch_bounds__(BAM_TRIP_WAVES * BAM_WAVE_SIZE) void k_along_resident(array_d_t<uint64_t>* da, const along_t g, const A algo)
{
    if (!g.sure && !(g.gate[0] && *g.gate[0]) && !(g.gate[1] && *g.gate[1])) return;
    __shared__ typename A::lds_t lds[BAM_TRIP_WAVES];
    __shared__ uint32_t left[BAM_TRIP_WAVES];
    __shared__ unsigned long long base;
    const uint32_t lane = bam::lane(), w_in_block = bam::first(threadIdx.x / BAM_WAVE_SIZE);
    typename A::lds_t& s = lds[w_in_block];
    bam::range_view<uint64_t> view;
    view.load(da->d_ranges);
    bool found = false, found_ahead = false;
    /* trips by turns, or, of joins, a stretch of them each (along_sweep) */
    const uint64_t n_blk = (g.n_segs + BAM_TRIP_WAVES * g.trip_segs - 1) / (BAM_TRIP_WAVES * g.trip_segs);
    const bool stretch = A::joins && g.stretches && *g.stretches;
    const uint64_t per = stretch ? (n_blk + gridDim.x - 1) / gridDim.x : 1, step = stretch ? 1 : gridDim.x;
    const uint64_t blk_end = stretch && (blockIdx.x + 1) * per < n_blk ? (blockIdx.x + 1) * per : n_blk;
    for (uint64_t blk = blockIdx.x * per; blk < blk_end; blk += step) {
        const uint64_t trip = blk * BAM_TRIP_WAVES + w_in_block, seg0 = trip * g.trip_segs;
        const uint64_t p0 = PARTS ? seg0 << g.part_log : seg0 >> g.seg_log;
        bool miss = false;
        if (seg0 < g.n_segs) {
            const uint32_t n_segs = (uint32_t)(g.n_segs - seg0 < g.trip_segs ? g.n_segs - seg0 : g.trip_segs);
            const uint32_t wanted = algo.prepare(g, s, seg0, n_segs);
            /* lane j: the trip's j-th page */
            const uint32_t per = 1u << (PARTS ? g.part_log : g.seg_log);
            bool want;
            if constexpr (PARTS) {
                const uint32_t rows = BAM_SEG_ROWS >> g.part_log;
                want = lane < (n_segs << g.part_log) && p0 + lane < g.n_pages && algo.wants(g, s, seg0, lane * rows, rows);
            } else want = lane < (g.trip_segs >> g.seg_log) && ((wanted >> (lane << g.seg_log)) & ((1u << per) - 1u)) != 0;
            data_page_t* const dp = view.pages + (view.pso >> view.page_size_log) + p0 + (want ? lane : 0);
            uint64_t sv = 0;
            uint32_t slot = 0;
            bool have = false;
            if (want && ((bam::ld_relaxed(&dp->state)) >> (CNT_SHIFT + 1)) == V_NB) {
                have = bam_try_hit(dp, 1, false, sv, slot);
                if (!have) __hip_atomic_fetch_add(&dp->state, 0u - 1u, __ATOMIC_RELAXED, BAM_AGENT);      /* it went in between: not waited for here */
            }
            miss = want && !have;
            view.n_access += have ? 1u : 0u;
            view.n_hit = view.n_access;
            if constexpr (PARTS) {
                const uint64_t here = bam::ballot(have);
                for (uint32_t k = 0; k < n_segs; k++) {
                    const uint64_t m = (here >> (k << g.part_log)) & ((1ull << per) - 1ull);
                    if (m) visit_parts(algo, g, s, view, seg0 + k, k, m, k << g.part_log, slot, found, found_ahead);
                }
            } else for (uint64_t m = bam::ballot(have); m; m &= m - 1) {
                const uint32_t j = bam::first_lane(m);
                const uint64_t* payload = (const uint64_t*)view.slot_addr(bam::bcast(slot, j)) + lane;
                for (uint32_t k = j << g.seg_log; k < (j + 1) << g.seg_log; k++) {
                    if (!((wanted >> k) & 1)) continue;
                    const uint64_t* const at = payload + (k & (per - 1u)) * BAM_SEG_EDGES;
                    uint64_t id[BAM_SEG_ROWS];
#pragma unroll
                    for (uint32_t r = 0; r < BAM_SEG_ROWS; r++) id[r] = bam::ld_payload(at + r * BAM_WAVE_SIZE);
                    algo.visit(g, s, seg0 + k, k, id, found, found_ahead);
                }
            }
            if (have) bam_release_refs(dp, 1, false);
        }
        const uint64_t mm = bam::ballot(miss);
        if (lane == 0) left[w_in_block] = bam::popc(mm);
        __syncthreads();
        uint32_t before = 0, total = 0;
#pragma unroll
        for (uint32_t k = 0; k < BAM_TRIP_WAVES; k++) { if (k < w_in_block) before += left[k]; total += left[k]; }
        if (threadIdx.x == 0 && total) base = __hip_atomic_fetch_add(g.n_missing, (unsigned long long)total, __ATOMIC_RELAXED, BAM_AGENT);
        __syncthreads();
        if (miss) g.missing[base + before + bam::popc(mm & bam::lanes_below(lane))] = (uint32_t)(p0 + lane);
    }
    view.flush_stats();
    raise_flag(g.flags, found);
    raise_flag(g.flags + 1, found_ahead);
}

/*
 * A wave holds at most `chunk` pages at a time; the launch keeps waves x chunk under half the cache.
 * Where more pages are missing than the cache holds, the round-robin hand would have pushed out every page of it by the end of the sweep,
 * those that the first launch found and visited before most vertices of the next level were known among them, and on the next
 * level they would come in again.  So a wave puts its next chunk where its last one is (BAM_PLACE_AGAIN), and fewer waves than keep
 * the store busiest do it, with as many slots: of 31 000 pages cached (BFS of 2^21 vertices) 27 000 stay.  Reads per call and ms,
 * before, with 512, 256 and 128 waves of 32 pages: 124 100 11.36, 108 100 9.83, 102 000 9.14, 98 000 8.88; 2^20 vertices, half cached,
 * 46 700 4.78, 32 900 3.32, 30 900 3.19, 30 700 3.20; 2^19, half, 28 500 3.17, 21 700 2.38, 18 400 2.07, 16 100 1.96.
 */
template <typename A, bool PARTS>
__global__ __launch_bounds__(BAM_WAVE_SIZE) void k_along_missing(array_d_t<uint64_t>* da, const along_t g, const A algo, const uint32_t chunk, const uint32_t again_waves)
{
    __shared__ typename A::lds_t s;
    const uint64_t n = *g.n_missing;
    if (!n) return;
    const uint32_t lane = bam::lane();
    bam::range_view<uint64_t> view;
    view.load(da->d_ranges);
    view.place = BAM_PLACE_PULLED;
    const uint64_t pso_pages = view.pso >> view.page_size_log;
    bool found = false, found_ahead = false;
    const bool again = A::again && n >= da->d_ranges->cache.n_pages;
    if (again && blockIdx.x >= again_waves) return;
    if (A::again) view.again = BAM_NO_SLOT;
    for (;;) {
        uint64_t c = 0;
        if (lane == 0) c = __hip_atomic_fetch_add(g.next_chunk, 1ull, __ATOMIC_RELAXED, BAM_AGENT) * chunk;
        c = bam::bcast(c, 0);
        if (c >= n) break;
        const bool want = lane < chunk && c + lane < n;
        const uint64_t p = g.missing[want ? c + lane : c];
        uint32_t last = BAM_NO_SLOT;
        /* as graph_by_page has it: no page is held while another is waited for */
        for (bool left = want; bam::ballot(left);) {
            uint32_t slot;
            const bool in = view.acquire_some(p + pso_pages, left, slot);
            if (!bam::ballot(in)) break;                      /* the wait was given up (the controller is marked aborted): the rest is not visited */
            left = left && !in;
            if (in) last = slot;
            if constexpr (PARTS) {
                /* the pages of a segment follow one another in the list, but for those that are not in it */
                const uint32_t per = 1u << g.part_log;
                for (uint64_t m = bam::ballot(in); m;) {
                    const uint32_t j = bam::first_lane(m);
                    const uint64_t seg = bam::bcast(p, j) >> g.part_log;
                    const uint64_t same = bam::ballot(in && p >> g.part_log == seg);
                    m &= ~same;
                    /* lane q: the slot of the segment's q-th page */
                    uint64_t held = 0;
                    uint32_t at = 0;
                    for (uint32_t q = 0; q < per; q++) {
                        const uint64_t of = bam::ballot((p & (per - 1u)) == q) & same;
                        if (!of) continue;
                        held |= 1ull << q;
                        const uint32_t s_q = bam::bcast(slot, bam::first_lane(of));
                        if (lane == q) at = s_q;
                    }
                    if (algo.prepare(g, s, seg, 1)) visit_parts(algo, g, s, view, seg, 0, held, 0, at, found, found_ahead);
                }
            } else for (uint64_t m = bam::ballot(in); m; m &= m - 1) {
                const uint32_t j = bam::first_lane(m);
                const uint64_t seg0 = bam::bcast(p, j) << g.seg_log;
                const uint64_t* payload = (const uint64_t*)view.slot_addr(bam::bcast(slot, j)) + lane;
                for (uint32_t k = 0; k < 1u << g.seg_log && seg0 + k < g.n_segs; k++) {
                    uint64_t id[BAM_SEG_ROWS];
#pragma unroll
                    for (uint32_t r = 0; r < BAM_SEG_ROWS; r++) id[r] = bam::ld_payload(payload + k * BAM_SEG_EDGES + r * BAM_WAVE_SIZE);
                    if (algo.prepare(g, s, seg0 + k, 1)) algo.visit(g, s, seg0 + k, 0, id, found, found_ahead);
                }
            }
            if (in) bam_release_refs(view.pages + p + pso_pages, 1, false);
        }
        if (A::again && again) { view.place = BAM_PLACE_AGAIN; view.again = last; }       /* the slots of the next chunk, unless the hand stands at others */
    }
    raise_flag(g.flags, found);
    raise_flag(g.flags + 1, found_ahead);
    view.flush_stats();
}

/* whether any vertex has this label */
__global__ void k_any_label(const uint32_t* label, const uint64_t n, const uint32_t which, unsigned long long* flag)
{
    bool any = false;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (uint64_t)gridDim.x * blockDim.x) any |= label[v] == which;
    raise_flag(flag, any);
}

// ---- PageRank by residual pushes (benchmarks/pagerank/main.cu:107-115 initialize, :252-273 kernel_coalesce_pc, :412-421 update) ----
__global__ void k_pr_initialize(bool* label, float* delta, float* residual, float* value, const uint64_t vertex_count, const uint64_t* vertexList, float alpha)
{
    const uint64_t tid = (uint64_t)blockDim.x * blockIdx.x + threadIdx.x;
    if (tid < vertex_count) {
        value[tid] = 1.0f - alpha;
        delta[tid] = (1.0f - alpha) * alpha / (vertexList[tid + 1] - vertexList[tid]);
        residual[tid] = 0.0f;
        label[tid] = true;
    }
}

/* every neighbour of a flagged vertex receives the vertex's delta: the group walk of the per-vertex graph kernels; the flags
 * are cleared by the host loop after the sweep */
__global__ __launch_bounds__(128) BAM_GRAPH_KERNEL_WAVES void k_pr_coalesce_pc(array_d_t<uint64_t>* da, const bool* label, const float* delta, float* residual,
                                                        const uint64_t vertex_count, const uint64_t* vertexList, uint64_t group,
                                                        const heavy_piece_t* heavy, uint64_t n_heavy, unsigned long long* next_work, uint32_t sweep)
{
    walk_vertex_groups(da, vertexList, vertex_count, group, heavy, n_heavy, next_work, (sweep & 1u) != 0,
                       [&](uint64_t v) { return label[v]; },
                       [&](uint64_t src, uint64_t next, uint64_t) { unsafeAtomicAdd(&residual[next], delta[src]); });
}

/* the same pushes taken page by page of the edge array; the flags are cleared by the host loop after the sweep */
__global__ __launch_bounds__(64) void k_pr_by_page(array_d_t<uint64_t>* da, const bool* label, const float* delta, float* residual, const uint64_t* offsets,
                                                    const uint64_t* first, uint64_t n_edges, uint32_t ppw, uint32_t sweep)
{
    graph_by_page(da, offsets, first, n_edges, ppw, (sweep & 1u) != 0,
                  [&](uint64_t v) { return label[v]; },
                  [&](uint64_t src, uint64_t next, uint64_t) { unsafeAtomicAdd(&residual[next], delta[src]); });
}

__global__ void k_pr_update(bool* label, float* delta, float* residual, float* value, const uint64_t vertex_count, const uint64_t* vertexList,
                            float tolerance, float alpha, bool* changed)
{
    const uint64_t tid = (uint64_t)blockDim.x * blockIdx.x + threadIdx.x;
    if (tid < vertex_count && residual[tid] > tolerance) {
        value[tid] += residual[tid];
        delta[tid] = residual[tid] * alpha / (vertexList[tid + 1] - vertexList[tid]);
        residual[tid] = 0.0f;
        label[tid] = true;
        *changed = true;
    }
}

// ---- SSSP (benchmarks/sssp/main.cu:174-201 kernel_coalesce_pc, :282-292 update): 32-bit costs, weights in their own array ----
/* relaxation of the edges of the flagged vertices with the cost each has at the time (any cost a vertex holds is the cost of a
 * path to it); the group walk of the per-vertex graph kernels, the weight of entry i read through a bam_ptr of its own */
template <bool FLOAT>
__device__ __forceinline__ void sssp_relax(uint32_t* newCostList, const bam_ptr<uint32_t>& weights, uint64_t src, uint64_t next, uint64_t i)
{
    const uint32_t have = __hip_atomic_load(&newCostList[src], __ATOMIC_RELAXED, BAM_AGENT), w = weights[i];
    /* single-precision costs (benchmarks/sssp_float/main.cu:69, 91-106, 194-217) travel as their bit patterns: for floats that
     * are not negative the order of the patterns is the order of the values, so the minimum is the integer one */
    const uint32_t cost = FLOAT ? __float_as_uint(__uint_as_float(have) + __uint_as_float(w)) : have + w;
    if (__hip_atomic_load(&newCostList[next], __ATOMIC_RELAXED, BAM_AGENT) > cost) atomicMin(&newCostList[next], cost);
}

template <bool FLOAT>
__global__ __launch_bounds__(128) BAM_GRAPH_KERNEL_WAVES void k_sssp_coalesce_pc(array_d_t<uint64_t>* de, array_d_t<uint32_t>* dw, const bool* label, uint32_t* newCostList,
                                                          const uint64_t vertex_count, const uint64_t* vertexList, uint64_t group,
                                                          const heavy_piece_t* heavy, uint64_t n_heavy, unsigned long long* next_work, uint32_t sweep)
{
    bam_ptr<uint32_t> wptr(dw);
    /* entry i of the weight array belongs to entry i of the edge array: what is touched ahead for the one is touched for the other */
    list_read_ahead<uint32_t> wahead;
    wahead.init(dw);
    walk_vertex_groups(de, vertexList, vertex_count, group, heavy, n_heavy, next_work, (sweep & 1u) != 0,
                       [&](uint64_t v) { return label[v]; },
                       [&](uint64_t src, uint64_t next, uint64_t i) { sssp_relax<FLOAT>(newCostList, wptr, src, next, i); }, &wahead);
}

__global__ void k_sssp_update(bool* label, uint32_t* costList, const uint32_t* newCostList, const uint64_t vertex_count, bool* changed)
{
    const uint64_t tid = (uint64_t)blockDim.x * blockIdx.x + threadIdx.x;
    if (tid < vertex_count && newCostList[tid] < costList[tid]) {
        costList[tid] = newCostList[tid];
        label[tid] = true;
        *changed = true;
    }
}

__global__ void k_iota(unsigned long long* p, uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

} // namespace

extern "C" {

namespace {
#define BAM_ALONG_WAVES 512u            /* waves that fetch what is missing, at most: as many as keep the store busy (k_fetch_wanted) */
/* launch shape of the by-page graph kernels: pages per wave trip and number of waves, so that what the waves hold
 * at any time stays under half of the cache */
struct by_page_plan { uint64_t n_edges = 0, n_pages = 0; uint32_t epp = 0, ppw = 0, blocks = 0; BufferPtr first; };

/* the end of a level: the device's `changed` word goes to the host through pinned memory, and it and the counter the next
 * sweep takes its work from start the next level at zero.  One small launch instead of two copies and a fill. */
/* words of a plan: [0] pieces, [1] next piece of work, [2] changed, [3] where the last list ends, [4] along_t::stretches; then, written by many waves and on lines of their own, the words
 * of along_t for each of the sweeps that are queued before the host looks */
#define BAM_PLAN_SWEEPS 6u
#define BAM_PLAN_STRETCHES 4u
#define BAM_PLAN_WORDS (16u + BAM_PLAN_SWEEPS * 48u)
#define BAM_PLAN_FLAGS(k) (16u + (k) * 48u)          /* along_t::flags of sweep k, */
#define BAM_PLAN_MISSING(k) (32u + (k) * 48u)        /* n_missing, */
#define BAM_PLAN_CHUNK(k) (48u + (k) * 48u)          /* next_chunk */
__global__ void k_level_end(unsigned long long* words, volatile uint64_t* host_flag)
{
    *host_flag = words[2];
    words[1] = words[2] = 0;
}
/* the end of the sweeps along the edges that were queued: two flags of each to the host; one wave */
__global__ void k_sweeps_end(unsigned long long* words, volatile uint64_t* host_flags)
{
    const uint32_t k = threadIdx.x;
    if (k >= BAM_PLAN_SWEEPS) return;
    host_flags[2 * k] = words[BAM_PLAN_FLAGS(k)];
    host_flags[2 * k + 1] = words[BAM_PLAN_FLAGS(k) + 1];
    words[BAM_PLAN_FLAGS(k)] = words[BAM_PLAN_FLAGS(k) + 1] = words[BAM_PLAN_MISSING(k)] = words[BAM_PLAN_CHUNK(k)] = 0;
}

/*
 * What the graph entry points need besides the graph, made once per graph (bam_array_set_graph) or, without that, once per
 * call: the pieces of the long edge lists (a list of d >= BAM_HEAVY_EDGES entries makes at most d / BAM_PIECE_EDGES + 1 <=
 * 2 d / BAM_HEAVY_EDGES pieces), the counter that hands out the work of a sweep, the `changed` word and its pinned copy,
 * the first-vertex table of the by-page kernels, and the per-vertex buffers of the algorithms, which come when first asked for.
 */
struct graph_plan {
    const uint64_t* offsets = nullptr;
    uint64_t n_vertices = 0, n_edges = 0;
    uint64_t lists_end = 0;                  /* offsets[n_vertices] */
    BufferPtr buf, words, host_words;
    heavy_piece_t* pieces = nullptr;
    unsigned long long* count = nullptr;     /* [0] number of pieces, [1] next piece of work of the sweep */
    uint64_t* changed = nullptr;             /* device */
    volatile uint64_t* host_flag = nullptr;  /* pinned host memory */
    uint64_t n_pieces = 0;
    uint64_t group = 512;                    /* vertices handed to a wave at a time */
    uint64_t resident = 0;                   /* waves a sweep runs */
    bool all_cached = false;                 /* the cache has a slot for every page of the edge array */
    std::atomic<uint32_t> cc_calls{0};
    /* Where some edges are on the store, calls that read all of them run forwards and backwards by turns: what the last one left
     * in the cache is what the next asks for first (2^22 vertices, a quarter cached: 7.4 ms along the pages, 8.4 always
     * forwards).  Where all are cached always forwards: from the back, chains grow long, each vertex hooked by the one before
     * it (2^19 vertices: 0.3 and 2.5 ms along the pages, 1.46 and 1.80 per vertex) */
    bool cc_backwards() { return !all_cached && (cc_calls++ & 1u) != 0; }
    by_page_plan bp;
    bool bp_built = false;
    along_t along{};                         /* n_segs = 0: the array or its pages do not qualify, or there is no memory for the tables */
    along_tables along_mem;
    uint64_t along_budget = 0;               /* pages that the waves of a launch may hold */
    BufferPtr bytes_a, bytes_b, floats_a, floats_b, words_a;      /* per-vertex buffers: flags, PageRank's delta and residual, SSSP's new costs */
    BufferPtr queue_a, queue_b, queue_bits, queue_totals;         /* bam_bfs_frontier: the two queues, the bit map that puts a queue in order and its counts per 4096 vertices */

    int build(bam_array_t* edges, const uint64_t* d_offsets, uint64_t nv, uint64_t other_cache_pages, hipStream_t st)
    {
        offsets = d_offsets; n_vertices = nv; n_edges = edges->a->adt.n_elems;
        const uint64_t cap = 2 * (n_edges / BAM_HEAVY_EDGES) + 1;
        buf = createBuffer(cap * sizeof(heavy_piece_t), 0);
        words = createBuffer(BAM_PLAN_WORDS * sizeof(unsigned long long), 0);
        host_words = createHostBuffer(2 * BAM_PLAN_SWEEPS * sizeof(uint64_t));
        pieces = (heavy_piece_t*)buf.get();
        count = (unsigned long long*)words.get();
        changed = (uint64_t*)words.get() + 2;
        host_flag = (volatile uint64_t*)host_words.get();
        int dev = 0, cus = 0;
        hip_err_chk(hipGetDevice(&dev));
        hip_err_chk(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        resident = (uint64_t)cus * 16;
        /* every lane of a running wave may hold a page of its own (its bam_ptr keeps the last one it read): more waves
         * than the cache has pages for would wait for slots that only they can give back */
        uint64_t cache_pages = edges->a->adt.n_ranges ? edges->a->h_ranges[0].cache.n_pages : 0;
        all_cached = true;
        for (uint64_t k = 0; k < edges->a->adt.n_ranges; k++) all_cached &= edges->a->h_ranges[k].page_count <= edges->a->h_ranges[k].cache.n_pages;
        if (other_cache_pages && other_cache_pages < cache_pages) cache_pages = other_cache_pages;
        if (cache_pages && resident > cache_pages / BAM_WAVE_SIZE) resident = cache_pages / BAM_WAVE_SIZE;
        if (resident < 2) resident = 2;
        hip_err_chk(hipMemsetAsync(words.get(), 0, BAM_PLAN_WORDS * sizeof(unsigned long long), st));
        hipLaunchKernelGGL(k_heavy_pieces, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, d_offsets, n_vertices, pieces, count, count + 3);
        hip_err_chk(hipGetLastError());
        unsigned long long got[4] = {};
        hip_err_chk(hipMemcpyAsync(got, count, sizeof(got), hipMemcpyDeviceToHost, st));
        hip_err_chk(hipStreamSynchronize(st));
        n_pieces = got[0];
        lists_end = got[3];
        return 0;
    }
    /* workgroups of two waves for a sweep over `n_items` items in groups of `grp` */
    uint32_t blocks(uint64_t n_items, uint64_t grp) const
    {
        const uint64_t units = (n_pieces + BAM_PIECE_BUNDLE - 1) / BAM_PIECE_BUNDLE + (n_items + grp - 1) / grp;
        return (uint32_t)(((units < resident ? units : resident) + 1) / 2);
    }
    unsigned long long* next_work() const { return count + 1; }
    /* between sweeps `changed` and the work counter are zero; true if the sweep just queued on `st` changed anything */
    bool level_end(hipStream_t st)
    {
        hipLaunchKernelGGL(k_level_end, dim3(1), dim3(1), 0, st, count, host_flag);
        hip_err_chk(hipGetLastError());
        hip_err_chk(hipStreamSynchronize(st));
        return *host_flag != 0;
    }
    /* the same for the sweeps along the edges: host_flag[2 k], [2 k + 1] are what sweep k found */
    void sweeps_end(hipStream_t st)
    {
        hipLaunchKernelGGL(k_sweeps_end, dim3(1), dim3(BAM_WAVE_SIZE), 0, st, count, host_flag);
        hip_err_chk(hipGetLastError());
        hip_err_chk(hipStreamSynchronize(st));
    }
    int by_page(bam_array_t* edges, hipStream_t st, bool can_do_without = false);
    bool along_edges(bam_array_t* edges, hipStream_t st, bool levels);
    static void* sized(BufferPtr& b, uint64_t bytes) { if (!b) b = createBuffer(bytes ? bytes : 8, 0); return b.get(); }
};

extern "C++" {
/* device memory, or NULL where it is refused */
BufferPtr spare_buffer(size_t bytes, int dev)
{
    void* p = nullptr;
    hip_err_chk(hipSetDevice(dev));
    if (hipMalloc(&p, bytes) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    return BufferPtr(p, [](void* q) { (void)hipFree(q); });
}
}

/* not 0, with nothing changed, where the array does not qualify, or, if the caller can do without, where memory is refused */
int graph_plan::by_page(bam_array_t* edges, hipStream_t st, const bool can_do_without)
{
    if (bp_built) return 0;
    by_page_plan& pl = bp;
    array_t<uint64_t>* a = edges->a;
    if (a->adt.n_ranges != 1) return fail(EINVAL, "by-page graph kernels take an array of one range");
    const range_d_t<uint64_t>& r = a->h_ranges[0];
    if (r.index_start != 0 || r.page_start_offset % r.cache.page_size) return fail(EINVAL, "by-page graph kernels need a range that starts on a page boundary");
    pl.n_edges = a->adt.n_elems;
    pl.epp = (uint32_t)(r.cache.page_size / 8);
    pl.n_pages = (pl.n_edges + pl.epp - 1) / pl.epp;
    const uint64_t budget = r.cache.n_pages / 2;               /* pages all waves together may hold */
    if (!budget) return fail(EINVAL, "by-page graph kernels need a cache of at least two pages");
    int dev = 0, cus = 0;
    hip_err_chk(hipGetDevice(&dev));
    hip_err_chk(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const uint64_t max_waves = (uint64_t)cus * 8;              /* eight waves per compute unit */
    uint64_t ppw = budget / max_waves;
    if (ppw > BAM_WAVE_SIZE) ppw = BAM_WAVE_SIZE;
    if (ppw < 1) ppw = 1;
    uint64_t waves = budget / ppw;
    if (waves > max_waves) waves = max_waves;
    const uint64_t trips = (pl.n_pages + ppw - 1) / ppw;
    if (waves > trips) waves = trips;
    pl.ppw = (uint32_t)ppw;
    pl.blocks = (uint32_t)waves;                               /* one wave per workgroup */
    if (can_do_without) {
        if (!(pl.first = spare_buffer((pl.n_pages + 1) * sizeof(uint64_t), dev))) return ENOMEM;
    } else
        pl.first = createBuffer((pl.n_pages + 1) * sizeof(uint64_t), dev);
    hipLaunchKernelGGL(k_page_first_vertex, dim3(blocks_for(pl.n_pages + 1, 256)), dim3(256), 0, st, offsets, n_vertices, (uint64_t)pl.epp, pl.n_pages,
                       (uint64_t*)pl.first.get());
    hip_err_chk(hipGetLastError());
    bp_built = true;
    return 0;
}

/*
 * Whether BFS and components of an array are read along its pages, whichever entry point asks for them: the array has one
 * range that begins on a page boundary, and pages the two launches take, and its number of elements covers the lists (it may be
 * less than its range holds, and an entry behind it is found all the same by who looks it up in the range).  Per vertex, and over a queue of vertices, the same
 * levels took 2.9 ms (2^20 vertices, all cached; 0.47 along the pages), 10.4 and 13.6 ms (2^18, a quarter cached; 1.8), 0.72
 * and 1.27 (2^12; 0.12; without a plan made for the graph 0.80 and 1.44, 0.25).
 */
bool graph_plan::along_edges(bam_array_t* edges, hipStream_t st, const bool levels)
{
    if (edges->a->adt.n_ranges != 1) return false;
    const range_d_t<uint64_t>& r = edges->a->h_ranges[0];
    if (r.index_start != 0 || r.page_start_offset % r.cache.page_size || r.cache.n_pages < 2) return false;
    if (by_page(edges, st, true)) return false;
    by_page_plan& pl = bp;
    /* pages of less than a segment: of a row or more, as many to a trip of the first launch as a wave has lanes */
    const uint64_t segs_per_page = std::max<uint64_t>(1, r.cache.page_size / (BAM_SEG_EDGES * 8));
    const uint64_t pages_per_seg = std::max<uint64_t>(1, BAM_SEG_EDGES * 8 / r.cache.page_size);
    if (pages_per_seg > BAM_SEG_ROWS || segs_per_page > BAM_TRIP_SEGS || !pl.n_pages || pl.n_pages > 0xFFFFFFFFull || n_vertices > 1ull << 32 || pl.n_edges > r.count || lists_end > pl.n_edges) return false;
    /* the first vertices of the segments where those are not the pages, the list of missing pages; and the bits, only where some edges
     * are on the store: there are no sweeps to spare otherwise */
    const uint64_t n_segs = (pl.n_edges + BAM_SEG_EDGES - 1) / BAM_SEG_EDGES, seg_words = segs_per_page > 1 || pages_per_seg > 1 ? n_segs + 1 : 0;
    int dev = 0;
    hip_err_chk(hipGetDevice(&dev));
    if (!along_mem.get(seg_words * sizeof(uint64_t) + pl.n_pages * sizeof(uint32_t), levels && !all_cached ? n_segs * BAM_SEG_ROWS * sizeof(uint64_t) : 0,
                       [&](size_t bytes) { return spare_buffer(bytes, dev); })) return false;
    along.ahead = (uint64_t*)along_mem.bits.get();
    if (!along.n_segs) {
        uint64_t* const seg_first = seg_words ? (uint64_t*)along_mem.tables.get() : (uint64_t*)pl.first.get();
        along.offsets = offsets; along.n_vertices = n_vertices; along.n_edges = pl.n_edges; along.n_pages = pl.n_pages; along.n_segs = n_segs;
        along.seg_log = (uint32_t)__builtin_ctzll(segs_per_page);
        along.part_log = (uint32_t)__builtin_ctzll(pages_per_seg);
        along.trip_segs = (uint32_t)segs_per_page;
        /* a wave's share as small as leaves 16384 waves or more (2^20 vertices, all cached, BFS: 0.47 ms, with 8192 0.50, 4096 0.56, 2048 0.70) */
        while (along.trip_segs < std::min<uint64_t>(BAM_TRIP_SEGS, BAM_WAVE_SIZE / pages_per_seg) && n_segs / along.trip_segs >= 32768) along.trip_segs *= 2;
        along.first = seg_first;
        if (seg_words)
            hipLaunchKernelGGL(k_page_first_vertex, dim3(blocks_for(n_segs + 1, 256)), dim3(256), 0, st, offsets, n_vertices, (uint64_t)BAM_SEG_EDGES, n_segs, seg_first);
        along.missing = (uint32_t*)((uint64_t*)along_mem.tables.get() + seg_words);
        along.n_missing = count + BAM_PLAN_MISSING(0);
        along.next_chunk = count + BAM_PLAN_CHUNK(0);
        along.flags = count + BAM_PLAN_FLAGS(0);
        along.sure = 1;
        along_budget = r.cache.n_pages / 2;
        hip_err_chk(hipGetLastError());
    }
    return true;
}

extern "C++" {
/*
 * One reading of the edge array, or of what the algorithm wants of it, with the words g names.
 * Joins: chains grow with the entries that are joined at a time (2^22 vertices, all cached, 2.6 ms with 16384 waves), and where they meet.
 * On a graph of neighbours side by side they grow along the array, and waves that take its next pieces by turns hook them to each other
 * as they grow: a stretch of the array to each workgroup.  On a graph without such an order stretches join trees all over it before there
 * is a large one, which the pieces in order grow from the front.  So where all edges are cached and make two turns or more, a
 * look at some of them (k_cc_look, 5 us) says which.  By turns and in stretches, two workgroups on a compute unit, us, medians: grids of 64 x 32768,
 * 1024 x 2048, 512 x 8192, 2048 x 2048, 4096 x 4096 3580, 2000, 2780, 2790, 9200 and 830, 860, 630, 1140, 2580; paths of 2^22 and 2^24 1560,
 * 5360 and 1340, 5130; uniform, 2^20, 2^21, 2^22 vertices 370, 610, 1200 and 570, 660, 1250; power-law, 2^18, 2^19, 2^20 310, 690, 620 and
 * 260, 400, 670; with two to five turns, grids of 64 x 8192, 1024 x 1024, 64 x 16384, 512 x 2048, 256 x 5095 1150, 1290, 1880, 1690, 2500 and
 * 1100, 1400, 840, 600, 450, paths of 2^20 and 2^21 445, 840 and 410, 750.  Three workgroups on a unit, in stretches, took 620, 650, 1400 on the uniform ones and 1600 and 2300 on square grids.
 * Where some edges are on the store, those that are not often lie together, and stretches would leave the most of them to few: a quarter of 2^22
 * vertices' cached 5.6 by turns, 6.2 in stretches; a half 4.1 and 4.2 (4.4 and more by turns with three workgroups on a unit, hence the LDS).
 */
template <typename A>
void along_sweep(bam_array_t* edges, const graph_plan* pl, along_t g, const A& algo, hipStream_t st)
{
    const uint64_t n_blk = (g.n_segs + BAM_TRIP_WAVES * g.trip_segs - 1) / (BAM_TRIP_WAVES * g.trip_segs);
    const bool look = A::joins && pl->all_cached && n_blk >= 2 * 512 && edges->a->h_ranges[0].cache.fast_reads;
    if (look) {
        unsigned long long* const stretches = pl->count + BAM_PLAN_STRETCHES;
        hipLaunchKernelGGL(k_cc_look, dim3(1), dim3(256), 0, st, edges->a->d_array_ptr, g, stretches);
        g.stretches = stretches;
    }
    const uint32_t blocks = (uint32_t)std::min<uint64_t>(!A::joins ? 1ull << 31 : look ? 512 : 1024, n_blk);
    const uint32_t lds = A::joins ? 48u << 10 : 0;
    if (g.part_log) hipLaunchKernelGGL((k_along_resident<A, true>), dim3(blocks), dim3(BAM_TRIP_WAVES * BAM_WAVE_SIZE), lds, st, edges->a->d_array_ptr, g, algo);
    else hipLaunchKernelGGL((k_along_resident<A, false>), dim3(blocks), dim3(BAM_TRIP_WAVES * BAM_WAVE_SIZE), lds, st, edges->a->d_array_ptr, g, algo);
    /* As many waves as leave each a batch worth sending (pages a wave, ms: 29 500 cached, BFS of 2^21 vertices 64 11.8, 32 11.4, 16
     * 11.6, 8 11.9; 7 500, 2^19 16 3.18, 8 3.11, 4 3.27; 3 700, 2^18 16 1.89, 8 1.73, 4 1.79; 2 048, 2^16 16 0.88, 8 0.72, 4 0.62, 2 0.70).
     * Under four pages a wave where the cache is small and what a wave fetched, visited one page after the other, is much: for joins, which
     * visit every entry, and for levels in pages of more than 8 KiB.  In batches of four and as here, and by k_bfs_by_page and k_cc_by_page, us:
     * 2^19 vertices, 8 entries each, pages of 64 KiB, 40 cached, BFS 23 200, 8 100, 10 400, components 23 900, 7 000, 9 000; of 16 KiB, 128 cached,
     * 8 900, 6 000, 6 000 and 8 600, 2 500, 3 100; components in pages of 8 KiB, 256 cached, 4 000, 1 800, 2 000, of 4 KiB, 256, 5 200, 3 400, 3 700.
     * Levels in small pages gain as much from it while their store alone is served, and lose it where another's is too (2^16, 8 KiB, 64
     * cached: 2.6 -> 1.6 ms, and 2.8 -> 3.7). */
    const uint64_t budget = pl->along_budget, enough = A::joins ? 128 : 64;
    const uint32_t least = A::joins || g.seg_log > 2 ? 1 : g.seg_log == 2 ? 2 : 4;
    const bool parts = g.part_log != 0;
    uint32_t chunk = parts ? 64 : 32;
    while ((chunk > 4 && budget / chunk < 256) || (chunk > least && budget / chunk < enough)) chunk /= 2;
    if (chunk > budget) chunk = (uint32_t)budget;
    /* Pages of less than a segment come in several times as fast: more of them to a wave, and more waves, as long as the cache is not
     * small (pages of 512 bytes, 64 to a wave with 1024 waves, 512 where slots are used again / 32 with 512 and 128 / 64 with 512 and 256, ms: BFS of 2^20
     * vertices, half cached, 3.9 / 7.7 / 4.9, a quarter 6.0 / 10.9 / 8.0; 2^16 vertices, a quarter, batches of 4, with 468, 256 and 128 waves 1.39,
     * 1.21, 1.23; components of 2^21, a quarter, 4.1 / 4.9 / 3.8). */
    const uint32_t waves = (uint32_t)std::min<uint64_t>(parts ? 2 * BAM_ALONG_WAVES : BAM_ALONG_WAVES, budget / chunk);
    /* 128 of them where they reuse their slots; 1024 pages on their way all the same (2^18 vertices, 3 700 cached, chunks of 4: 256 waves 1.59
     * ms, 128 1.93, all 469 1.58; the hand alone 1.76) */
    const uint32_t again_waves = std::min(waves, parts ? chunk == 64 ? 512u : 256u : std::max(128u, 1024u / chunk));
    if (parts) hipLaunchKernelGGL((k_along_missing<A, true>), dim3(waves), dim3(BAM_WAVE_SIZE), 0, st, edges->a->d_array_ptr, g, algo, chunk, again_waves);
    else hipLaunchKernelGGL((k_along_missing<A, false>), dim3(waves), dim3(BAM_WAVE_SIZE), 0, st, edges->a->d_array_ptr, g, algo, chunk, again_waves);
    hip_err_chk(hipGetLastError());
}
}

/*
 * All levels from labels of which the source's is set; the number of levels there are.  BAM_PLAN_SWEEPS sweeps are queued before
 * the host looks, each made only if the ones before found vertices for it: with a look after every level that look was most of a
 * small graph's time (all cached, 2^12 vertices, 5 levels: 118 -> 74 us; 2^16, 6: 197 -> 137; 2^20, 6: 479 -> 418; three sweeps at a time
 * 88, 150, 433, eight 84, 146, 424).
 */
uint32_t bfs_along_levels(bam_array_t* edges, graph_plan* pl, uint32_t* d_labels, hipStream_t st)
{
    const bool ahead = pl->along.ahead != nullptr;
    if (ahead) hip_err_chk(hipMemsetAsync(pl->along.ahead, 0, pl->along.n_segs * BAM_SEG_ROWS * sizeof(uint64_t), st));
    unsigned long long* const words = pl->count;
    /* a level has vertices for sure if the sweep before found some; it may have some if the one before that found some ahead */
    bool sure = true, next = false;
    for (uint32_t base = 0;; base += BAM_PLAN_SWEEPS) {
        for (uint32_t k = 0; k < BAM_PLAN_SWEEPS; k++) {
            along_t g = pl->along;
            g.flags = words + BAM_PLAN_FLAGS(k);
            g.n_missing = words + BAM_PLAN_MISSING(k);
            g.next_chunk = words + BAM_PLAN_CHUNK(k);
            g.sure = k == 0 || (k == 1 && next);
            g.gate[0] = k ? words + BAM_PLAN_FLAGS(k - 1) : nullptr;
            g.gate[1] = k > 1 ? words + BAM_PLAN_FLAGS(k - 2) + 1 : nullptr;
            if (ahead) along_sweep(edges, pl, g, bfs_along<true>{d_labels, base + k}, st);
            else along_sweep(edges, pl, g, bfs_along<false>{d_labels, base + k}, st);
        }
        pl->sweeps_end(st);
        for (uint32_t k = 0; k < BAM_PLAN_SWEEPS; k++) {
            const bool found = pl->host_flag[2 * k] != 0, found_ahead = pl->host_flag[2 * k + 1] != 0;
            if (found || next) { sure = found; next = found_ahead; continue; }
            if (sure) return base + k + 1;
            /* the last sweep was for vertices that a sweep ahead of their level had found; a nearer one may have found them since */
            hipLaunchKernelGGL(k_any_label, dim3(1024), dim3(256), 0, st, d_labels, pl->n_vertices, base + k, words + BAM_PLAN_FLAGS(0));
            pl->sweeps_end(st);
            return pl->host_flag[0] ? base + k + 1 : base + k;
        }
    }
}

/* the forest that cc_read_edges begins with: k_cc_begin, for the arrays whose pages are read along (elsewhere, and where entries are not read without a
 * reference on their page, every vertex by itself) */
void cc_begin(bam_array_t* edges, graph_plan* pl, unsigned long long* comp, hipStream_t st)
{
    const uint64_t nv = pl->n_vertices;
    if (!pl->along.n_segs || !edges->a->h_ranges[0].cache.fast_reads) { hipLaunchKernelGGL(k_iota, dim3(blocks_for(nv, 256)), dim3(256), 0, st, comp, nv); return; }
    const bool large = pl->all_cached && nv >= 1ull << 21;
    hipLaunchKernelGGL(k_cc_begin<false>, dim3(blocks_for(nv, 256)), dim3(256), 0, st, edges->a->d_array_ptr, pl->offsets, nv, comp, 1u);
    hipLaunchKernelGGL(k_cc_shorten, dim3(blocks_for(nv, 256)), dim3(256), 0, st, comp, nv);
    for (uint32_t round = large ? 1 : 0; round < 3; round++) {
        const uint32_t each = round < 2 ? 4 : 8;
        hipLaunchKernelGGL(k_cc_begin<true>, dim3(blocks_for((nv + each - 1) / each, 256)), dim3(256), 0, st, edges->a->d_array_ptr, pl->offsets, nv, comp, each);
        hipLaunchKernelGGL(k_cc_shorten, dim3(blocks_for(nv, 256)), dim3(256), 0, st, comp, nv);
    }
}
/* one reading of the edges that joins the trees of their ends.  In one launch where all are cached and few: 2^15 entries take 80 us, in two
 * 88 (in pages of 512 and 1024 bytes, which that launch goes over one after the other, 271 and 144, and 85); but that one goes over
 * the vertices between the lists of a page, so not where there may be many.  By page (bam_cc_by_page), in pages of less than 4 KiB, also where
 * all are cached and many: 2^24 entries of a uniform graph in pages of 512, 1024, 2048 bytes 690, 660, 630 us, in two launches 725, 730, 775
 * (vertex by vertex 990, 970, 1070). */
void cc_read_edges(bam_array_t* edges, graph_plan* pl, unsigned long long* comp, hipStream_t st, const bool by_page)
{
    const bool one = pl->bp.n_edges <= 1ull << 17 ? pl->along.part_log < 2 : by_page && pl->along.part_log;
    if (pl->along.n_segs && !(one && pl->all_cached && pl->n_vertices <= pl->bp.n_edges / 4)) along_sweep(edges, pl, pl->along, cc_along{comp}, st);
    else if (pl->bp.n_pages)
        hipLaunchKernelGGL(k_cc_by_page, dim3(pl->bp.blocks), dim3(BAM_WAVE_SIZE), 0, st, edges->a->d_array_ptr, pl->offsets, (const uint64_t*)pl->bp.first.get(), pl->bp.n_edges, pl->bp.ppw,
                           pl->cc_backwards(), comp);
}

/* the plan bam_array_set_graph made for this graph, or one made now in `local` that lives for the call */
graph_plan* plan_for(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t other_cache_pages, hipStream_t st, std::unique_ptr<graph_plan>& local)
{
    graph_plan* p = (graph_plan*)edges->graph.get();
    if (p && p->offsets == d_offsets && p->n_vertices == n_vertices && p->n_edges == edges->a->adt.n_elems && !other_cache_pages) return p;
    local.reset(new graph_plan());
    local->build(edges, d_offsets, n_vertices, other_cache_pages, st);
    return local.get();
}
} // namespace

int bam_array_set_graph(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, void* stream)
{
    if (!edges) return fail(EINVAL, "bam_array_set_graph: null argument");
    if (!d_offsets) { edges->graph.reset(); return 0; }
    if (!n_vertices) return fail(EINVAL, "bam_array_set_graph: empty graph");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::shared_ptr<graph_plan> p(new graph_plan());
    p->build(edges, d_offsets, n_vertices, 0, st);
    if (edges->a->adt.n_ranges == 1) {
        const range_d_t<uint64_t>& r = edges->a->h_ranges[0];
        if (r.index_start == 0 && r.page_start_offset % r.cache.page_size == 0 && r.cache.n_pages >= 2) p->by_page(edges, st);
    }
    const bool along = p->along_edges(edges, st, true);
    /* the per-vertex buffers the sweeps use, so that no later call has to allocate */
    graph_plan::sized(p->bytes_a, n_vertices); graph_plan::sized(p->bytes_b, n_vertices);
    graph_plan::sized(p->floats_a, n_vertices * sizeof(float)); graph_plan::sized(p->floats_b, n_vertices * sizeof(float));
    if (n_vertices <= 0xFFFFFFFFull && !along) {
        /* bam_bfs_frontier's queues and what puts them in order */
        const uint64_t n_words = (n_vertices + 63) / 64;
        graph_plan::sized(p->queue_a, n_vertices * sizeof(uint32_t)); graph_plan::sized(p->queue_b, n_vertices * sizeof(uint32_t));
        graph_plan::sized(p->queue_bits, n_words * sizeof(unsigned long long));
        graph_plan::sized(p->queue_totals, (n_words + BAM_WAVE_SIZE - 1) / BAM_WAVE_SIZE * sizeof(uint32_t));
    }
    hip_err_chk(hipStreamSynchronize(st));
    edges->graph = p;
    BAM_API_END
}

int bam_bfs(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t src, uint32_t* d_labels,
            uint32_t coarse, uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_labels) return fail(EINVAL, "bam_bfs: null argument");
    if (src >= n_vertices || !coarse) return fail(EINVAL, "bam_bfs: source out of range or coarse = 0");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    hip_err_chk(hipMemsetAsync(d_labels, 0xFF, n_vertices * sizeof(uint32_t), st));
    hip_err_chk(hipMemsetAsync(d_labels + src, 0, sizeof(uint32_t), st));
    if (pl->along_edges(edges, st, true)) {
        const uint32_t levels = bfs_along_levels(edges, pl, d_labels, st);
        if (iterations) *iterations = levels;
        return 0;
    }
    /* a group's lists are asked for as one batch of commands: a few hundred vertices make that batch large enough for the
     * store path, and keep the one word all waves take their work from out of the way */
    const uint64_t group = coarse > 512 ? coarse : 512;
    const uint32_t threads = 128;
    uint32_t level = 0, iter = 0;
    bool changed;
    do {
        hipLaunchKernelGGL(k_bfs_coalesce_coarse_ptr_pc, dim3(pl->blocks(n_vertices, group)), dim3(threads), 0, st,
                           edges->a->d_array_ptr, d_labels, level, n_vertices, d_offsets, pl->changed, group, pl->pieces, pl->n_pieces, pl->next_work());
        hip_err_chk(hipGetLastError());
        iter++; level++;
        changed = pl->level_end(st);
    } while (changed);
    if (iterations) *iterations = iter;
    BAM_API_END
}

namespace {
/* units of a shaped launch and the waves that walk them (see walk_shaped): at most one wave per eight pages of the cache */
struct shaped_launch { uint64_t n_units; uint32_t blocks; };
shaped_launch shape_of(int shape, uint64_t n_vertices, uint64_t coarse, uint64_t stride, uint64_t cache_pages)
{
    shaped_launch sl{};
    if (shape == 3) sl.n_units = (n_vertices + BAM_SHAPE_CHUNK - 1) / BAM_SHAPE_CHUNK;
    else if (shape == 1) sl.n_units = ((n_vertices + stride * coarse) / (stride * coarse)) * stride;
    else sl.n_units = ((n_vertices + stride) / stride) * stride;
    const uint64_t per_wave = shape == 2 ? 4 : 1;
    uint64_t waves = (sl.n_units + per_wave - 1) / per_wave;
    int dev = 0, cus = 0;
    hip_err_chk(hipGetDevice(&dev));
    hip_err_chk(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (waves > (uint64_t)cus * 16) waves = (uint64_t)cus * 16;
    if (cache_pages && waves > cache_pages / 8) waves = cache_pages / 8;
    if (waves < 2) waves = 2;
    sl.blocks = (uint32_t)((waves + 1) / 2);            /* workgroups of two waves */
    return sl;
}
} // namespace

int bam_bfs_shaped(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t src, uint32_t* d_labels,
                   int shape, uint32_t coarse, uint32_t stride, uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_labels) return fail(EINVAL, "bam_bfs_shaped: null argument");
    if (src >= n_vertices || shape < 0 || shape > 3 || !coarse || !stride) return fail(EINVAL, "bam_bfs_shaped: source out of range, shape not 0..3, or coarse / stride = 0");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    const shaped_launch sl = shape_of(shape, n_vertices, coarse, stride, edges->a->adt.n_ranges ? edges->a->h_ranges[0].cache.n_pages : 0);
    hip_err_chk(hipMemsetAsync(d_labels, 0xFF, n_vertices * sizeof(uint32_t), st));
    hip_err_chk(hipMemsetAsync(d_labels + src, 0, sizeof(uint32_t), st));
    uint32_t level = 0, iter = 0;
    bool changed;
    do {
        const dim3 grid(sl.blocks), block(128);
        array_d_t<uint64_t>* d = edges->a->d_array_ptr;
        switch (shape) {
        case 0: hipLaunchKernelGGL(k_bfs_shaped<0>, grid, block, 0, st, d, d_labels, level, n_vertices, d_offsets, pl->changed, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        case 1: hipLaunchKernelGGL(k_bfs_shaped<1>, grid, block, 0, st, d, d_labels, level, n_vertices, d_offsets, pl->changed, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        case 2: hipLaunchKernelGGL(k_bfs_shaped<2>, grid, block, 0, st, d, d_labels, level, n_vertices, d_offsets, pl->changed, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        default: hipLaunchKernelGGL(k_bfs_shaped<3>, grid, block, 0, st, d, d_labels, level, n_vertices, d_offsets, pl->changed, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        }
        hip_err_chk(hipGetLastError());
        iter++; level++;
        changed = pl->level_end(st);
    } while (changed);
    if (iterations) *iterations = iter;
    BAM_API_END
}

int bam_cc_shaped(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t* d_labels,
                  int shape, uint32_t coarse, uint32_t stride, uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_labels) return fail(EINVAL, "bam_cc_shaped: null argument");
    if (!n_vertices || shape < 0 || shape > 3 || !coarse || !stride) return fail(EINVAL, "bam_cc_shaped: empty graph, shape not 0..3, or coarse / stride = 0");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    const shaped_launch sl = shape_of(shape, n_vertices, coarse, stride, edges->a->adt.n_ranges ? edges->a->h_ranges[0].cache.n_pages : 0);
    bool* curr = (bool*)graph_plan::sized(pl->bytes_a, n_vertices);
    bool* next = (bool*)graph_plan::sized(pl->bytes_b, n_vertices);
    hipLaunchKernelGGL(k_iota, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, (unsigned long long*)d_labels, n_vertices);
    hip_err_chk(hipMemsetAsync(curr, 0x01, n_vertices, st));
    hip_err_chk(hipMemsetAsync(next, 0x00, n_vertices, st));
    uint32_t iter = 0;
    bool changed;
    do {
        const dim3 grid(sl.blocks), block(128);
        array_d_t<uint64_t>* d = edges->a->d_array_ptr;
        unsigned long long* comp = (unsigned long long*)d_labels;
        bool* ch = (bool*)pl->changed;
        switch (shape) {
        case 0: hipLaunchKernelGGL(k_cc_shaped<0>, grid, block, 0, st, d, curr, next, n_vertices, d_offsets, comp, ch, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        case 1: hipLaunchKernelGGL(k_cc_shaped<1>, grid, block, 0, st, d, curr, next, n_vertices, d_offsets, comp, ch, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        case 2: hipLaunchKernelGGL(k_cc_shaped<2>, grid, block, 0, st, d, curr, next, n_vertices, d_offsets, comp, ch, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        default: hipLaunchKernelGGL(k_cc_shaped<3>, grid, block, 0, st, d, curr, next, n_vertices, d_offsets, comp, ch, (uint64_t)coarse, (uint64_t)stride, sl.n_units); break;
        }
        hip_err_chk(hipGetLastError());
        hip_err_chk(hipMemsetAsync(curr, 0x00, n_vertices, st));
        bool* t = curr; curr = next; next = t;
        iter++;
        changed = pl->level_end(st);
    } while (changed);
    if (iterations) *iterations = iter;
    BAM_API_END
}

int bam_bfs_frontier(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t src, uint32_t* d_labels,
                     uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_labels) return fail(EINVAL, "bam_bfs_frontier: null argument");
    if (src >= n_vertices) return fail(EINVAL, "bam_bfs_frontier: source out of range");
    if (n_vertices > 0xFFFFFFFFull) return fail(EINVAL, "bam_bfs_frontier: the queues hold 32-bit vertex numbers");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    if (pl->along_edges(edges, st, true)) {
        hip_err_chk(hipMemsetAsync(d_labels, 0xFF, n_vertices * sizeof(uint32_t), st));
        hip_err_chk(hipMemsetAsync(d_labels + src, 0, sizeof(uint32_t), st));
        const uint32_t levels = bfs_along_levels(edges, pl, d_labels, st);
        if (iterations) *iterations = levels;
        return 0;
    }
    /* two queues of at most every vertex once (benchmarks/bfs/main.cu:1489-1492); the size of the next one is the reference's `changed`.
     * They, and what puts a queue in order, belong to the plan: with bam_array_set_graph nothing is allocated here */
    uint32_t* curr = (uint32_t*)graph_plan::sized(pl->queue_a, n_vertices * sizeof(uint32_t));
    uint32_t* next = (uint32_t*)graph_plan::sized(pl->queue_b, n_vertices * sizeof(uint32_t));
    const uint64_t n_words = (n_vertices + 63) / 64, n_bit_waves = (n_words + BAM_WAVE_SIZE - 1) / BAM_WAVE_SIZE;
    unsigned long long* bits = (unsigned long long*)graph_plan::sized(pl->queue_bits, n_words * sizeof(unsigned long long));      /* zero between levels */
    uint32_t* totals = (uint32_t*)graph_plan::sized(pl->queue_totals, n_bit_waves * sizeof(uint32_t));
    unsigned long long* next_size = (unsigned long long*)pl->changed;
    const uint32_t src32 = (uint32_t)src;
    hip_err_chk(hipMemsetAsync(d_labels, 0xFF, n_vertices * sizeof(uint32_t), st));
    hip_err_chk(hipMemsetAsync(d_labels + src, 0, sizeof(uint32_t), st));
    hip_err_chk(hipMemcpyAsync(curr, &src32, sizeof(uint32_t), hipMemcpyHostToDevice, st));
    const uint32_t threads = 128;
    uint64_t group = BAM_WAVE_SIZE;                 /* queue entries handed to a wave at a time: one per lane, more of a sorted queue */
    bool sorted = true;                             /* the first queue holds the source alone */
    uint32_t level = 0, iter = 0;
    unsigned long long active = 1;
    const char* e = getenv("BAM_FRONTIER_SORT");
    const bool sort_queue = !e || atoi(e) != 0;
    do {
        hipLaunchKernelGGL(k_bfs_frontier_coalesce_ptr_pc, dim3(pl->blocks(active, group)), dim3(threads), 0, st, edges->a->d_array_ptr, d_labels, level,
                           d_offsets, curr, (uint64_t)active, next, next_size, group, pl->pieces, pl->n_pieces, pl->next_work(), sorted);
        hip_err_chk(hipGetLastError());
        iter++; level++;
        pl->level_end(st);
        active = *pl->host_flag;
        sorted = sort_queue;
        group = sorted ? pl->group : BAM_WAVE_SIZE;
        if (sorted && active > 1) {
            /* the queue comes out in the order of discovery; in the order of the vertices the level reads the edge array
             * front to back (neighbouring lists share pages, a page is not evicted between two of its lists, and the pages
             * under the lists of a group of entries can be asked for together as in the sweep over all vertices).  The
             * ordered queue goes into the buffer the level just walked, so the two do not change places. */
            hipLaunchKernelGGL(k_queue_mark, dim3(blocks_for(active, 256)), dim3(256), 0, st, next, (uint64_t)active, bits);
            hipLaunchKernelGGL(k_bits_count, dim3(blocks_for(n_bit_waves * BAM_WAVE_SIZE, 256)), dim3(256), 0, st, bits, n_words, totals);
            hipLaunchKernelGGL(k_totals_scan, dim3(1), dim3(1024), 0, st, totals, n_bit_waves);
            hipLaunchKernelGGL(k_bits_emit, dim3(blocks_for(n_bit_waves * BAM_WAVE_SIZE, 256)), dim3(256), 0, st, bits, n_words, totals, curr);
            hip_err_chk(hipGetLastError());
        } else
            std::swap(curr, next);
    } while (active);
    if (iterations) *iterations = iter;
    BAM_API_END
}

int bam_cc(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t* d_labels,
           uint32_t coarse, uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_labels) return fail(EINVAL, "bam_cc: null argument");
    if (!coarse || !n_vertices) return fail(EINVAL, "bam_cc: empty graph or coarse = 0");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    const uint64_t group = coarse > 512 ? coarse : 512;
    unsigned long long* comp = (unsigned long long*)d_labels;
    const bool along = pl->along_edges(edges, st, false);
    if (along) { cc_begin(edges, pl, comp, st); cc_read_edges(edges, pl, comp, st, false); }
    else {
        hipLaunchKernelGGL(k_iota, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, comp, n_vertices);
        hipLaunchKernelGGL(k_cc_coalesce_coarse_ptr_pc, dim3(pl->blocks(n_vertices, group)), dim3(128), 0, st, edges->a->d_array_ptr, n_vertices, d_offsets, comp, group,
                       pl->pieces, pl->n_pieces, pl->next_work(), pl->cc_backwards());
    }
    hipLaunchKernelGGL(k_cc_settle, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, comp, n_vertices, pl->along.n_missing, pl->along.next_chunk);
    hip_err_chk(hipGetLastError());
    if (along) { hip_err_chk(hipStreamSynchronize(st)); }
    else pl->level_end(st);
    if (iterations) *iterations = 2;
    BAM_API_END
}

int bam_bfs_by_page(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t src, uint32_t* d_labels,
                    uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_labels) return fail(EINVAL, "bam_bfs_by_page: null argument");
    if (src >= n_vertices) return fail(EINVAL, "bam_bfs_by_page: source out of range");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    if (int rc = pl->by_page(edges, st)) return rc;
    hip_err_chk(hipMemsetAsync(d_labels, 0xFF, n_vertices * sizeof(uint32_t), st));
    hip_err_chk(hipMemsetAsync(d_labels + src, 0, sizeof(uint32_t), st));
    if (pl->along_edges(edges, st, true)) {
        const uint32_t iter = bfs_along_levels(edges, pl, d_labels, st);
        if (iterations) *iterations = iter;
        return 0;
    }
    uint32_t level = 0, iter = 0;
    bool changed;
    do {
        if (pl->bp.n_pages)
            hipLaunchKernelGGL(k_bfs_by_page, dim3(pl->bp.blocks), dim3(BAM_WAVE_SIZE), 0, st, edges->a->d_array_ptr, d_labels, level, d_offsets,
                               (const uint64_t*)pl->bp.first.get(), pl->bp.n_edges, pl->bp.ppw, pl->changed);
        hip_err_chk(hipGetLastError());
        iter++; level++;
        changed = pl->level_end(st);
    } while (changed);
    if (iterations) *iterations = iter;
    BAM_API_END
}

int bam_cc_by_page(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t* d_labels, uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_labels) return fail(EINVAL, "bam_cc_by_page: null argument");
    if (!n_vertices) return fail(EINVAL, "bam_cc_by_page: empty graph");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    if (int rc = pl->by_page(edges, st)) return rc;
    pl->along_edges(edges, st, false);
    unsigned long long* comp = (unsigned long long*)d_labels;
    uint32_t iter = 0;
    bool changed = true;
    /*
     * With every edge cached a sweep of label propagation costs 40 to 60 us up to 2^22 entries, and a reading that joins as much
     * as its longest chain of loads and exchanges that failed, which differs from call to call by twice and more: sweeps / joins in us, medians,
     * for 0.03, 0.13, 0.26, 0.5, 1, 2.1, 4.2, 8.4 million entries of a uniform random graph 116 / 78, 140 / 106, 157 / 315, 177 / 495,
     * 220 / 450, 290 / 450, 456 / 510, 735 / 560; of a power-law graph of 0.1, 0.5, 1.9, 7.7, 15 million 105 / 83, 140 / 106, 187 / 171,
     * 437 / 254, 886 / 354; of a grid of 64 x 4096 (1 million, six sweeps and joins) 460 / 660.
     * A graph that is long rather than wide would take a sweep per step: after six the edges are joined, from the labels as they
     * are, each of which names a smaller vertex of the component or the vertex itself, and so the roots the labels lead to do.
     */
    if (pl->bp.n_pages && pl->all_cached && pl->bp.n_edges > (1ull << 17) && pl->bp.n_edges < (1ull << 22)) {
        bool* curr = (bool*)graph_plan::sized(pl->bytes_a, n_vertices);
        bool* next = (bool*)graph_plan::sized(pl->bytes_b, n_vertices);
        hipLaunchKernelGGL(k_iota, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, comp, n_vertices);
        hip_err_chk(hipMemsetAsync(curr, 0x01, n_vertices, st));
        hip_err_chk(hipMemsetAsync(next, 0x00, n_vertices, st));
        while (changed && iter < 6) {
            hipLaunchKernelGGL(k_cc_sweep_by_page, dim3(pl->bp.blocks), dim3(BAM_WAVE_SIZE), 0, st, edges->a->d_array_ptr, curr, next, d_offsets,
                               (const uint64_t*)pl->bp.first.get(), pl->bp.n_edges, pl->bp.ppw, comp, (bool*)pl->changed);
            hip_err_chk(hipGetLastError());
            hip_err_chk(hipMemsetAsync(curr, 0x00, n_vertices, st));
            std::swap(curr, next);
            iter++;
            changed = pl->level_end(st);
        }
    }
    if (changed) {
        if (iter) hipLaunchKernelGGL(k_cc_shorten, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, comp, n_vertices);
        else cc_begin(edges, pl, comp, st);
        cc_read_edges(edges, pl, comp, st, true);
        hipLaunchKernelGGL(k_cc_settle, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, comp, n_vertices, pl->along.n_missing, pl->along.next_chunk);
        hip_err_chk(hipGetLastError());
        hip_err_chk(hipStreamSynchronize(st));
        iter += 2;
    }
    if (iterations) *iterations = iter;
    BAM_API_END
}

int bam_pagerank(bam_array_t* edges, const uint64_t* d_offsets, uint64_t n_vertices, float alpha, float tolerance, uint32_t max_iterations,
                 int by_page, float* d_value, uint32_t* iterations, void* stream)
{
    if (!edges || !d_offsets || !d_value) return fail(EINVAL, "bam_pagerank: null argument");
    if (iterations) *iterations = 0;
    if (!n_vertices) return 0;
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, 0, st, local);
    if (by_page)
        if (int rc = pl->by_page(edges, st)) return rc;
    float* delta_d = (float*)graph_plan::sized(pl->floats_a, n_vertices * sizeof(float));
    float* residual_d = (float*)graph_plan::sized(pl->floats_b, n_vertices * sizeof(float));
    bool* label_d = (bool*)graph_plan::sized(pl->bytes_a, n_vertices);
    const uint32_t upd_blocks = blocks_for(n_vertices, 256);
    hipLaunchKernelGGL(k_pr_initialize, dim3(upd_blocks), dim3(256), 0, st, label_d, delta_d, residual_d, d_value, n_vertices, d_offsets, alpha);
    uint32_t iter = 0;
    bool changed;
    do {
        if (by_page) {
            if (pl->bp.n_pages)
                hipLaunchKernelGGL(k_pr_by_page, dim3(pl->bp.blocks), dim3(BAM_WAVE_SIZE), 0, st, edges->a->d_array_ptr, label_d, delta_d, residual_d, d_offsets,
                                   (const uint64_t*)pl->bp.first.get(), pl->bp.n_edges, pl->bp.ppw, iter);
        } else
            hipLaunchKernelGGL(k_pr_coalesce_pc, dim3(pl->blocks(n_vertices, pl->group)), dim3(128), 0, st, edges->a->d_array_ptr, label_d, delta_d, residual_d,
                               n_vertices, d_offsets, pl->group, pl->pieces, pl->n_pieces, pl->next_work(), iter);
        hip_err_chk(hipMemsetAsync(label_d, 0, n_vertices, st));
        iter++;
        hipLaunchKernelGGL(k_pr_update, dim3(upd_blocks), dim3(256), 0, st, label_d, delta_d, residual_d, d_value, n_vertices, d_offsets, tolerance, alpha, (bool*)pl->changed);
        hip_err_chk(hipGetLastError());
        changed = pl->level_end(st);
    } while (changed && iter < max_iterations);
    if (iterations) *iterations = iter;
    BAM_API_END
}

namespace {
/* the loop of benchmarks/sssp/main.cu:663-725 (and of sssp_float, :624-700): relax from the flagged vertices, adopt what got
 * cheaper, flag it, until nothing does.  FLOAT: costs and weights are single-precision values, unreached = 1e9 (sssp_float :529) */
void sssp_run(const bool FLOAT, bam_array_t* edges, bam_array32_t* weights, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t src, uint32_t* d_costs,
              uint32_t* iterations, hipStream_t st)
{
    /* a lane holds a page of the weights beside its page of the edges: the waves a sweep runs must fit the smaller cache too */
    const uint64_t weight_pages = weights->a->adt.n_ranges ? weights->a->h_ranges[0].cache.n_pages : 0;
    std::unique_ptr<graph_plan> local;
    graph_plan* pl = plan_for(edges, d_offsets, n_vertices, weight_pages ? weight_pages : 1, st, local);
    uint32_t* new_d = (uint32_t*)graph_plan::sized(pl->words_a, n_vertices * sizeof(uint32_t));
    bool* label_d = (bool*)graph_plan::sized(pl->bytes_a, n_vertices);
    const uint32_t zero = 0;                    /* the pattern of 0.0f as well */
    const bool one = true;
    const float far = 1000000000.0f;
    uint32_t unreached = 0xFFFFFFFFu;
    if (FLOAT) memcpy(&unreached, &far, sizeof(unreached));
    hip_err_chk(hipMemsetD32Async((hipDeviceptr_t)d_costs, (int)unreached, n_vertices, st));
    hip_err_chk(hipMemsetD32Async((hipDeviceptr_t)new_d, (int)unreached, n_vertices, st));
    hip_err_chk(hipMemsetAsync(label_d, 0, n_vertices, st));
    hip_err_chk(hipMemcpyAsync(label_d + src, &one, sizeof(bool), hipMemcpyHostToDevice, st));
    hip_err_chk(hipMemcpyAsync(d_costs + src, &zero, sizeof(uint32_t), hipMemcpyHostToDevice, st));
    hip_err_chk(hipMemcpyAsync(new_d + src, &zero, sizeof(uint32_t), hipMemcpyHostToDevice, st));
    const uint32_t threads = 128;
    uint32_t iter = 0;
    bool changed;
    do {
        hipLaunchKernelGGL(FLOAT ? k_sssp_coalesce_pc<true> : k_sssp_coalesce_pc<false>, dim3(pl->blocks(n_vertices, pl->group)), dim3(threads), 0, st,
                           edges->a->d_array_ptr, weights->a->d_array_ptr, label_d, new_d, n_vertices, d_offsets, pl->group, pl->pieces, pl->n_pieces, pl->next_work(), iter);
        hip_err_chk(hipMemsetAsync(label_d, 0, n_vertices, st));
        hipLaunchKernelGGL(k_sssp_update, dim3(blocks_for(n_vertices, 256)), dim3(256), 0, st, label_d, d_costs, new_d, n_vertices, (bool*)pl->changed);
        hip_err_chk(hipGetLastError());
        iter++;
        changed = pl->level_end(st);
    } while (changed);
    if (iterations) *iterations = iter;
}
} // namespace

int bam_sssp(bam_array_t* edges, bam_array32_t* weights, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t src, uint32_t* d_costs,
             uint32_t* iterations, void* stream)
{
    if (!edges || !weights || !d_offsets || !d_costs) return fail(EINVAL, "bam_sssp: null argument");
    if (src >= n_vertices) return fail(EINVAL, "bam_sssp: source out of range");
    if (edges->a->adt.n_elems != weights->a->adt.n_elems) return fail(EINVAL, "bam_sssp: one weight per edge");
    BAM_API_BEGIN
    sssp_run(false, edges, weights, d_offsets, n_vertices, src, d_costs, iterations, (hipStream_t)stream);
    BAM_API_END
}

int bam_sssp_float(bam_array_t* edges, bam_array32_t* weights, const uint64_t* d_offsets, uint64_t n_vertices, uint64_t src, float* d_costs,
                   uint32_t* iterations, void* stream)
{
    if (!edges || !weights || !d_offsets || !d_costs) return fail(EINVAL, "bam_sssp_float: null argument");
    if (src >= n_vertices) return fail(EINVAL, "bam_sssp_float: source out of range");
    if (edges->a->adt.n_elems != weights->a->adt.n_elems) return fail(EINVAL, "bam_sssp_float: one weight per edge");
    BAM_API_BEGIN
    sssp_run(true, edges, weights, d_offsets, n_vertices, src, (uint32_t*)d_costs, iterations, (hipStream_t)stream);
    BAM_API_END
}

} // extern "C"
