// vectoradd, reduction and scan of the C-ABI library (benchmarks/vectoradd, reduction, scan of the reference): kernels
// in which consecutive threads read consecutive elements through bam_ptr, and the scan that allocates nothing.
#include "bam_capi_internal.h"

namespace {

// ---- vectoradd (benchmarks/vectoradd/main.cu:102-117 kernel_baseline_ptr_pc): C[i] = A[i] + B[i], all three behind the cache ----
__global__ __launch_bounds__(64) void k_vectoradd_ptr_pc(array_d_t<uint64_t>* da, array_d_t<uint64_t>* db, uint64_t n_elems, array_d_t<uint64_t>* dc, const fetch_plan fp)
{
    if (fp.done && blockIdx.x < fp.blocks) {
        array_d_t<uint64_t>* const arrays[3] = {da, db, dc};
        fetch_role(arrays, n_elems, fp);
        return;
    }
    /* once each, or by turns where the cache does not let as many waves hold pages at a time (bam_vectoradd) */
    const uint32_t fetching = fp.done ? fp.blocks : 0u;
    for (uint64_t first = (uint64_t)(blockIdx.x - fetching) * BAM_WAVE_SIZE; first < n_elems; first += (uint64_t)(gridDim.x - fetching) * BAM_WAVE_SIZE) {
        const uint64_t tid = first + threadIdx.x;
        bam_ptr<uint64_t> Aptr(da);
        bam_ptr<uint64_t> Bptr(db);
        bam_ptr<uint64_t> Cptr(dc);
        const bam_ptr<uint64_t>& A = Aptr;
        const bam_ptr<uint64_t>& B = Bptr;
        touch_ahead(da, first, n_elems, BAM_WAVE_SIZE, 0);
        touch_ahead(db, first, n_elems, BAM_WAVE_SIZE, 1);
        touch_ahead(dc, first, n_elems, BAM_WAVE_SIZE, 2);
        if (tid < n_elems) Cptr[tid] = A[tid] + B[tid];
        if (fp.done && threadIdx.x == 0) __hip_atomic_fetch_add(fp.done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

/*
 * The same sums a page at a time, for arrays whose pages are 4 or 8 KiB and fit a staging page.  A wave holds up to 16 or 32
 * pages of A and of B, loads them in 16-byte pieces and writes the sums, past the caches, straight to where they go:
 *  - into the slot of C's page where that is resident;
 *  - where it is not, and the three arrays are larger than the cache, to the store: into the staging pages of a batch of write
 *    commands.  Read by read, a page of C would come in only to be written over, push out a page of A or B, and be pushed out
 *    in turn, a command at a time, by whoever needs its slot.  The page's descriptor is BUSY until its write has completed, as
 *    under an evictor, so nobody brings the old content in meanwhile.
 * First the pages of which A and B are resident (k_vectoradd_resident), so that what a call left in the cache is there for the
 * next one, then the others in batches (k_vectoradd_missing).  What neither could do (C's page was being loaded or evicted, a
 * command failed) is left to k_vectoradd_rest.
 * Bound by the store: 10^7 elements and a cache of half their pages, with the flush, 10.6 ms element by element (58 600 page
 * reads, 19 500 writes), here 2.9 (13 600 reads); the cache holds all: 6.1 and 2.05, of which the flush takes 1.9; 10^6
 * elements, half: 5.6 and 0.5.
 */
struct vadd_t {
    array_d_t<uint64_t>* a;
    array_d_t<uint64_t>* b;
    array_d_t<uint64_t>* c;
    uint64_t n_elems, n_full;                   /* pages that the elements fill */
    uint32_t past_cache;                        /* C's pages that are not resident go to the store */
    uint8_t* done;                              /* [n_full] pages that are finished */
    uint32_t* list;                             /* [n_full] pages left to the second launch */
    unsigned long long* n_list;                 /* zero between calls, like the next one */
    unsigned long long* next_chunk;
    uint32_t* finished;
    uint32_t call;
};
#define BAM_VADD_PAGES 32u                      /* pages of C a wave of the first launch looks after */

/* the place of a page of C for the lane to write its sums to, taken in one of the two ways above */
struct vadd_dest { data_page_t* dp; uint8_t* at; bool in_place, claimed; };
__device__ __forceinline__ vadd_dest vadd_take(const bam::range_view<uint64_t>& view, const uint64_t page, const bool has, const bool past_cache)
{
    vadd_dest d{view.pages + (has ? page : 0), nullptr, false, false};
    if (!has) return d;
    const uint32_t st = bam::ld_relaxed(&d.dp->state) >> (CNT_SHIFT + 1);
    if (st == V_NB) {
        uint64_t sv;
        uint32_t slot = 0;
        d.in_place = bam_try_hit(d.dp, 1, true, sv, slot);
        if (d.in_place) d.at = view.slot_addr(slot);
        else __hip_atomic_fetch_add(&d.dp->state, 0u - 1u, __ATOMIC_RELAXED, BAM_AGENT);
    } else if (st == NV_NB && past_cache) {
        const uint32_t o = __hip_atomic_fetch_or(&d.dp->state, BUSY, __ATOMIC_RELAXED, BAM_AGENT);
        if ((o & BUSY) == 0) {
            if ((o >> (CNT_SHIFT + 1)) == NV_NB) d.claimed = true;
            else __hip_atomic_fetch_and(&d.dp->state, DISABLE_BUSY_MASK, __ATOMIC_RELAXED, BAM_AGENT);      /* it came in meanwhile */
        }
    }
    return d;
}

/* by the whole wave: the sums of the lanes' pages (payload of A at pa, of B at pb) to their places, which are given back; true for the lanes whose sums are there */
__device__ __forceinline__ bool vadd_pages(const bam::range_view<uint64_t>& view, const uint64_t page, vadd_dest d, const uint8_t* pa, const uint8_t* pb)
{
    using bam::u64x2_t;
    const uint32_t lane = bam::lane();
    page_cache_d_t* const cache = &view.r->cache;
    Controller* const ctl = cache->d_ctrls[0];
    QueuePair* const qp = ctl->d_qps + bam::first(bam::wave_slot_hash() % ctl->n_qps);
    /* more commands than half the queue's slots go through it in rounds */
    const uint32_t step = qp->sq.qs >> 1 ? qp->sq.qs >> 1 : 1u;
    uint64_t todo = bam::ballot(d.claimed);
    bool ok = false, pending = d.in_place;
    do {
        const bool mine = ((todo >> lane) & 1) != 0 && bam::rank_in(todo) < step;
        uint32_t ticket = 0, id = 0;
        if (mine) {
            ticket = bam::sq_reserve_group(&qp->sq);
            id = ticket & qp->sq.qs_minus_1;
            d.at = qp->stage + (size_t)id * qp->stage_stride;
        }
        for (uint64_t m = bam::ballot(mine || pending); m; m &= m - 1) {
            const uint32_t j = bam::first_lane(m);
            const uint8_t* qa = (const uint8_t*)bam::bcast((uint64_t)pa, j) + lane * 16u;
            const uint8_t* qb = (const uint8_t*)bam::bcast((uint64_t)pb, j) + lane * 16u;
            uint8_t* to = (uint8_t*)bam::bcast((uint64_t)d.at, j) + lane * 16u;
            for (uint32_t o = 0; o < view.page_size; o += 4096u) {
                const u64x2_t* p[8];
                u64x2_t x[8];
#pragma unroll
                for (uint32_t r = 0; r < 4; r++) { p[r] = (const u64x2_t*)(qa + o + r * 1024u); p[r + 4] = (const u64x2_t*)(qb + o + r * 1024u); }
                bam::ld_payload_stream8x2(p, x);
#pragma unroll
                for (uint32_t r = 0; r < 4; r++) {
                    const u64x2_t sum = {x[r].x + x[r + 4].x, x[r].y + x[r + 4].y};
                    bam::st16_sys(to + o + r * 1024u, __builtin_bit_cast(bam::u32x4_t, sum));
                }
            }
        }
        bam::wait_stores();                     /* in memory, or in the staging pages, before anybody is told */
        if (mine) {
            const uint64_t stage = qp->stage_ioaddr + (uint64_t)id * qp->stage_stride;
            nvm_cmd_t cmd;
#pragma unroll
            for (int i = 0; i < 16; i++) cmd.dword[i] = 0;
            nvm_cmd_header(&cmd, (uint16_t)id, NVM_IO_WRITE, qp->nvmNamespace);
            nvm_cmd_data_ptr(&cmd, stage, view.page_size > qp->pageSize ? stage + qp->pageSize : 0);
            nvm_cmd_rw_blks(&cmd, view.r->get_backing_page(page) * cache->n_blocks_per_page, (uint16_t)cache->n_blocks_per_page);
            bam::sq_submit_group(&qp->sq, &cmd, ticket);
            ok = bam::cq_wait_group(&qp->cq, &qp->sq, id);
            bam::sq_release_group(&qp->sq, id);
        }
        pending = false;
        todo &= ~bam::ballot(mine);
    } while (todo);
    if (d.claimed) __hip_atomic_fetch_and(&d.dp->state, DISABLE_BUSY_MASK, __ATOMIC_RELAXED, BAM_AGENT);
    if (d.in_place) bam_release_refs(d.dp, 1, false);         /* written through: nothing to make visible */
    return d.in_place || (d.claimed && ok);
}

/* the accesses of `pages` pages, an element each, as the bam_ptrs of k_vectoradd_ptr_pc count them; all lanes */
__device__ __forceinline__ void vadd_account(bam::range_view<uint64_t>& view, const uint32_t pages, const uint32_t hits)
{
    view.n_access = pages * (view.page_size / (8u * BAM_WAVE_SIZE));
    view.n_hit = hits * (view.page_size / (8u * BAM_WAVE_SIZE));
    view.flush_stats();
}

/* elements [first, last) of one page, through bam_ptr; the whole wave */
__device__ __forceinline__ void vadd_elements(const vadd_t& g, const uint64_t first, const uint64_t last)
{
    for (uint64_t e = first + bam::lane(); e < last; e += BAM_WAVE_SIZE) {
        bam_ptr<uint64_t> Aptr(g.a);
        bam_ptr<uint64_t> Bptr(g.b);
        bam_ptr<uint64_t> Cptr(g.c);
        const bam_ptr<uint64_t>& A = Aptr;
        const bam_ptr<uint64_t>& B = Bptr;
        Cptr[e] = A[e] + B[e];
    }
}

__global__ __launch_bounds__(BAM_WAVE_SIZE) void k_vectoradd_resident(const vadd_t g)
{
    const uint32_t lane = bam::lane();
    bam::range_view<uint64_t> va, vb, vc;
    va.load(g.a->d_ranges);
    const uint64_t per_page = va.page_size / 8;
    const uint32_t n_main = (uint32_t)((g.n_full + BAM_VADD_PAGES - 1) / BAM_VADD_PAGES);
    if (blockIdx.x >= n_main) {                 /* what is behind the last full page, 64 elements to a wave: one wave took 35 us for a page less one */
        const uint64_t first = g.n_full * per_page + (uint64_t)(blockIdx.x - n_main) * BAM_WAVE_SIZE;
        vadd_elements(g, first, first + BAM_WAVE_SIZE < g.n_elems ? first + BAM_WAVE_SIZE : g.n_elems);
        return;
    }
    vb.load(g.b->d_ranges);
    vc.load(g.c->d_ranges);
    const uint64_t i = (uint64_t)blockIdx.x * BAM_VADD_PAGES + lane;
    const bool mine = lane < BAM_VADD_PAGES && i < g.n_full;
    data_page_t* const da = va.pages + (va.pso >> va.page_size_log) + (mine ? i : 0);
    data_page_t* const db = vb.pages + (vb.pso >> vb.page_size_log) + (mine ? i : 0);
    bool has = false;
    uint32_t slot_a = 0, slot_b = 0;
    if (mine && bam::ld_relaxed(&da->state) >> (CNT_SHIFT + 1) == V_NB && bam::ld_relaxed(&db->state) >> (CNT_SHIFT + 1) == V_NB) {
        uint64_t sv;
        if (bam_try_hit(da, 1, false, sv, slot_a)) {
            has = bam_try_hit(db, 1, false, sv, slot_b);
            if (!has) __hip_atomic_fetch_add(&db->state, 0u - 1u, __ATOMIC_RELAXED, BAM_AGENT);
        }
        if (!has) __hip_atomic_fetch_add(&da->state, 0u - 1u, __ATOMIC_RELAXED, BAM_AGENT);
    }
    const uint64_t page_c = (vc.pso >> vc.page_size_log) + i;
    vadd_dest d = vadd_take(vc, page_c, has, g.past_cache != 0);
    const uint32_t pages = bam::popc(bam::ballot(d.in_place || d.claimed)), placed = bam::popc(bam::ballot(d.in_place));
    bool took = false;
    if (pages) took = vadd_pages(vc, page_c, d, va.slot_addr(slot_a), vb.slot_addr(slot_b));
    if (has) { bam_release_refs(da, 1, false); bam_release_refs(db, 1, false); }
    if (mine) g.done[i] = took ? 1 : 0;
    const uint64_t left = bam::ballot(mine && !took);
    if (left) {
        uint64_t at = 0;
        if (lane == 0) at = __hip_atomic_fetch_add(g.n_list, (unsigned long long)bam::popc(left), __ATOMIC_RELAXED, BAM_AGENT);
        at = bam::bcast(at, 0);
        if (mine && !took) g.list[at + bam::popc(left & bam::lanes_below(lane))] = (uint32_t)i;
    }
    if (!pages) return;
    vadd_account(va, pages, pages);
    vadd_account(vb, pages, pages);
    vadd_account(vc, pages, placed);
}

/* a wave holds at most 3 x `chunk` pages at a time; the launch keeps what all hold under half the cache */
__global__ __launch_bounds__(BAM_WAVE_SIZE) void k_vectoradd_missing(const vadd_t g, const uint32_t chunk)
{
    const uint64_t n = *g.n_list;
    if (!n) return;
    const uint32_t lane = bam::lane();
    bam::range_view<uint64_t> va, vb, vc;
    va.load(g.a->d_ranges);
    vb.load(g.b->d_ranges);
    vc.load(g.c->d_ranges);
    va.place = vb.place = vc.place = BAM_PLACE_PULLED;
    const uint64_t pso_a = va.pso >> va.page_size_log, pso_b = vb.pso >> vb.page_size_log, pso_c = vc.pso >> vc.page_size_log;
    bool any_left = false;
    uint32_t pages = 0, placed = 0;
    for (;;) {
        uint64_t k = 0;
        if (lane == 0) k = __hip_atomic_fetch_add(g.next_chunk, 1ull, __ATOMIC_RELAXED, BAM_AGENT) * chunk;
        k = bam::bcast(k, 0);
        if (k >= n) break;
        const bool want = lane < chunk && k + lane < n;
        const uint64_t i = g.list[want ? k + lane : k];
        uint32_t slot_a = BAM_NO_SLOT, slot_b = BAM_NO_SLOT;
        auto keep_a = [&](uint32_t s_) { slot_a = s_; return false; };
        auto keep_b = [&](uint32_t s_) { slot_b = s_; return false; };
        auto touch = [](uint32_t) { return true; };
        va.acquire_helped(pso_a + i, want, false, keep_a, keep_a);
        vb.acquire_helped(pso_b + i, want, false, keep_b, keep_b);
        if (!g.past_cache) vc.acquire_helped(pso_c + i, want, false, touch, touch);
        const bool has = want && slot_a != BAM_NO_SLOT && slot_b != BAM_NO_SLOT;
        vadd_dest d = vadd_take(vc, pso_c + i, has, g.past_cache != 0);
        pages += bam::popc(bam::ballot(d.in_place || d.claimed));
        placed += bam::popc(bam::ballot(d.in_place));
        bool took = false;
        if (bam::ballot(d.in_place || d.claimed)) took = vadd_pages(vc, pso_c + i, d, va.slot_addr(has ? slot_a : 0), vb.slot_addr(has ? slot_b : 0));
        if (want) { va.release(pso_a + i, false); vb.release(pso_b + i, false); }
        if (took) g.done[i] = 1;
        any_left |= want && !took;
    }
    if (bam::ballot(any_left)) note_work_left(g.finished, g.call);
    vadd_account(va, pages, 0);
    vadd_account(vb, pages, 0);
    vadd_account(vc, pages, placed);
}

__global__ __launch_bounds__(BAM_WAVE_SIZE) void k_vectoradd_rest(const vadd_t g)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *g.n_list = *g.next_chunk = 0;
    if (g.finished[BAM_LEFT_WORD] != g.call) return;
    const uint64_t per_page = g.a->d_ranges[0].cache.page_size / 8;
    for (uint64_t i = blockIdx.x; i < g.n_full; i += gridDim.x)
        if (!g.done[i]) vadd_elements(g, i * per_page, (i + 1) * per_page);
}

// ---- reduction (benchmarks/reduction/main.cu:166-195 kernel_reduce_baseline_ptr_pc): output[b] = sum of the 2 x blockDim elements of block b ----
/* output `bid` by `half` consecutive threads of the workgroup (a multiple of 64; each such group its own output, or none: take =
 * false); all threads of the workgroup come in */
__device__ __forceinline__ void reduce_output(array_d_t<uint64_t>* da, unsigned long long* output, const uint64_t len, const uint64_t bid, const uint32_t half, const bool take, uint64_t* wave_total)
{
    const uint64_t tid = threadIdx.x % half, start = 2ull * half * bid;
    const uint32_t w = threadIdx.x / BAM_WAVE_SIZE;
    uint64_t v = 0;
    if (take) {
        bam_ptr<uint64_t> in_ptr(da);
        const bam_ptr<uint64_t>& input = in_ptr;
        /* a group reads 2 x half consecutive elements: its waves' first elements */
        const uint64_t first = start + tid - tid % BAM_WAVE_SIZE;
        if (first < len) touch_ahead(da, first, len);
        if (first + half < len) touch_ahead(da, first + half, len);
        if (start + tid < len) v = input[start + tid];
        if (half + start + tid < len) v += input[half + start + tid];
    }
    v = wave_sum(v);
    if (half == BAM_WAVE_SIZE) {                /* a wave's own output: nothing to wait for */
        if (tid == 0 && take) output[bid] = v;
        return;
    }
    if (bam::lane() == 0) wave_total[w] = v;
    __syncthreads();
    if (tid < BAM_WAVE_SIZE) {
        v = wave_sum(tid < half / BAM_WAVE_SIZE ? wave_total[w + tid] : 0);
        if (tid == 0 && take) output[bid] = v;
    }
}

__global__ void k_reduce_ptr_pc(array_d_t<uint64_t>* da, unsigned long long* output, uint64_t len, const fetch_plan fp)
{
    __shared__ uint64_t wave_total[1024 / BAM_WAVE_SIZE];
    if (fp.done && blockIdx.x < fp.blocks) {
        array_d_t<uint64_t>* const arrays[1] = {da};
        fetch_role(arrays, len, fp);
        return;
    }
    const uint64_t bid = blockIdx.x - (fp.done ? fp.blocks : 0u);
    reduce_output(da, output, len, bid, blockDim.x, true, wave_total);
    if (fp.done && threadIdx.x == 0) __hip_atomic_fetch_add(fp.done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/*
 * The outputs k_reduce_resident left, by at most 32768 waves: what is resident was summed there, and a grid with a workgroup
 * per output takes as long to find nothing to do as that kernel takes (2^24 elements, blocks of 64, all resident: 71 us a call,
 * 47 with 32768 workgroups of a wave, 42 with 8192 of four).  So small outputs are taken `blockDim / half` to a workgroup.
 * notes[k] covers `per_note` consecutive outputs.  Bound by the store where all is missing (2^24 elements, blocks of 64: 8.7 ms
 * in one launch of a workgroup per output, 7.7 here; with 4096 waves 11).  The word that says whether anything was left is read as an ordinary
 * load, and is on another line than *done: read past the caches by every wave, on the line the workgroups count themselves off
 * in, it cost some 12 ns a wave, one after the other (2^22 elements in workgroups of a wave: 2.35 ms, as here 1.9).
 */
#define BAM_REST_WAVES 32768u
__global__ void k_reduce_rest(array_d_t<uint64_t>* da, unsigned long long* output, uint64_t len, uint64_t n_outputs, uint32_t half, uint32_t per_note, const uint8_t* notes,
                              const uint32_t* finished, uint32_t call, const fetch_plan fp)
{
    __shared__ uint64_t wave_total[1024 / BAM_WAVE_SIZE];
    if (finished[BAM_LEFT_WORD] != call) return;      /* nothing was left */
    const uint32_t fetching = fp.done ? fp.blocks : 0u;
    if (blockIdx.x < fetching) {
        array_d_t<uint64_t>* const arrays[1] = {da};
        fetch_role(arrays, len, fp);
        return;
    }
    const uint32_t groups = blockDim.x / half;
    for (uint64_t b0 = (uint64_t)(blockIdx.x - fetching) * groups; b0 < n_outputs; b0 += (uint64_t)(gridDim.x - fetching) * groups) {
        const uint64_t bid = b0 + threadIdx.x / half;
        reduce_output(da, output, len, bid, half, bid < n_outputs && notes[bid / per_note] != 0, wave_total);
        if (half > BAM_WAVE_SIZE) __syncthreads();
        if (fp.done && threadIdx.x % half == 0) __hip_atomic_fetch_add(fp.done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---- reading consecutive elements that are resident ----
/*
 * Eight rows of 128 elements from element `first` (a multiple of 128; the same in every lane) of a range that starts on a
 * page boundary with element 0: lane l gets elements first + 128 r + 2 l and the one behind it in x[r], zero from element n
 * on.  True (in every lane) if every page with elements below n was resident, by two looks at its descriptor, before and
 * after the loads, as in bam_read_unpinned; nothing is counted.  The look is one load per page and wave instead of one
 * atomic pair per page and wave, and a page's payload one 16-byte load per lane and KiB.
 */
#define BAM_ROW_ELEMS (2u * BAM_WAVE_SIZE)
#define BAM_WAVE_ROWS 8u
#define BAM_WAVE_ELEMS (BAM_WAVE_ROWS * BAM_ROW_ELEMS)
__device__ __forceinline__ bool read_rows_resident(const bam::range_view<uint64_t>& view, const uint64_t first, const uint64_t n, bam::u64x2_t (&x)[BAM_WAVE_ROWS])
{
    using bam::u64x2_t;
    const uint32_t lane = bam::lane(), log = view.page_size_log;
#pragma unroll
    for (uint32_t r = 0; r < BAM_WAVE_ROWS; r++) x[r] = u64x2_t{0, 0};
    if (first >= n) return true;
    const uint64_t end = first + BAM_WAVE_ELEMS < n ? first + BAM_WAVE_ELEMS : n;
    const uint64_t byte0 = first * 8, p0 = byte0 >> log;
    const uint32_t np = (uint32_t)(((end - 1) * 8 >> log) - p0) + 1;          /* at most 16: pages are of 512 bytes and more */
    const uint64_t* dp = (const uint64_t*)(view.pages + p0 + (lane < np ? lane : 0));
    const uint64_t s1 = __hip_atomic_load(dp, __ATOMIC_RELAXED, BAM_AGENT);
    if (bam::ballot(((uint32_t)s1 >> (CNT_SHIFT + 1)) != V_NB)) return false;
    const uint32_t slot = (uint32_t)(s1 >> 32) & BAM_SLOT_MASK;
    const u64x2_t* p[BAM_WAVE_ROWS];
#pragma unroll
    for (uint32_t r = 0; r < BAM_WAVE_ROWS; r++) {
        /* a row spans two pages of 512 bytes or lies in one larger one; rows behind the last page with elements below n read
         * that page once more */
        const uint64_t byte = byte0 + r * (BAM_ROW_ELEMS * 8u);
        const uint32_t a = (uint32_t)((byte >> log) - p0), b = (uint32_t)(((byte + BAM_ROW_ELEMS * 4u) >> log) - p0);
        const uint32_t slot_a = bam::bcast(slot, a < np ? a : np - 1), slot_b = bam::bcast(slot, b < np ? b : np - 1);
        p[r] = (const u64x2_t*)(view.base_addr + ((uint64_t)(lane < BAM_WAVE_SIZE / 2 ? slot_a : slot_b) << log) + ((byte + lane * 16u) & (view.page_size - 1)));
    }
    bam::ld_payload_stream8x2(p, x);                /* with its wait: the elements are here before the second look goes out */
    const uint64_t s2 = __hip_atomic_load(dp, __ATOMIC_RELAXED, BAM_AGENT);
    if (end - first < BAM_WAVE_ELEMS) {
#pragma unroll
        for (uint32_t r = 0; r < BAM_WAVE_ROWS; r++) {
            const uint64_t e = first + r * BAM_ROW_ELEMS + 2u * lane;
            if (e >= n) x[r].x = 0;
            if (e + 1 >= n) x[r].y = 0;
        }
    }
    return bam::ballot(((s1 ^ s2) & 0xFFFFFFFFC0000000ull) != 0) == 0;
}

/*
 * The outputs of bam_reduce whose elements are resident.  A wave takes as many outputs at a time as fit its 1024 elements,
 * or one larger one, and goes on to the next; the outputs it could not read are left to k_reduce_rest (a byte per turn says
 * so).  The accesses are counted as the bam_ptr of k_reduce_ptr_pc counts them: one per lane and page, the lane's second
 * element, block_size further on, on its own only where it lies on another page.
 * Bound by HBM: 8 bytes read per element.  2^26 elements in outputs of 512: 95 us, 5.6 TB/s (4221 through bam_ptr); the call takes 16 us
 * whatever its size below 2^22.
 */
__global__ __launch_bounds__(256) void k_reduce_resident(array_d_t<uint64_t>* da, unsigned long long* output, uint64_t len, uint64_t n_outputs, uint32_t half_groups, uint32_t per_note,
                                                         uint8_t* notes, uint32_t* finished, uint32_t call, unsigned long long* done)
{
    const uint32_t lane = bam::lane(), rows = half_groups;          /* rows of an output: 2 x 64 x half_groups elements, 128 to a row */
    const uint64_t wave = bam::first(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / BAM_WAVE_SIZE), n_waves = (uint64_t)gridDim.x * blockDim.x / BAM_WAVE_SIZE;
    if (blockIdx.x == 0 && threadIdx.x == 0) *done = 0;              /* for the fetching workgroups of the launch behind this one */
    bam::range_view<uint64_t> view;
    view.load(da->d_ranges);
    const uint64_t n_turns = (n_outputs + per_note - 1) / per_note;
    bool any_left = false;
    for (uint64_t t = wave; t < n_turns; t += n_waves) {
        const uint64_t o0 = t * per_note, first = o0 * rows * BAM_ROW_ELEMS;
        bam::u64x2_t x[BAM_WAVE_ROWS];
        /* what the lanes hold of the output at hand, and how many of its rows are still to come */
        uint64_t acc = 0, o = o0;
        uint32_t rest = rows;
        bool left = false;
        const uint32_t turn_rows = per_note * rows;
        for (uint32_t r0 = 0; r0 < turn_rows && !left; r0 += BAM_WAVE_ROWS) {
            if (!read_rows_resident(view, first + (uint64_t)r0 * BAM_ROW_ELEMS, len, x)) { left = true; break; }
#pragma unroll
            for (uint32_t r = 0; r < BAM_WAVE_ROWS; r++) {
                if (r0 + r < turn_rows) {
                    acc += x[r].x + x[r].y;
                    if (--rest == 0) {
                        const uint64_t sum = bam::wave_running_sum(acc);
                        if (lane == BAM_WAVE_SIZE - 1 && o < n_outputs) output[o] = sum;
                        acc = 0; rest = rows; o++;
                    }
                }
            }
        }
        if (lane == 0) notes[t] = left ? 1 : 0;
        any_left |= left;
        if (!left && lane < 2u * turn_rows) {
            /* lane l: the l-th group of 64 elements of the turn; the first half of an output's groups are read by its threads first */
            const uint64_t e = first + lane * 64ull;
            const uint32_t within = lane % (2u * rows);
            if (within < half_groups && e < len) {
                const uint64_t e2 = e + half_groups * 64ull;
                uint32_t n = (uint32_t)(len - e < 64 ? len - e : 64);
                if (e2 < len && view.page_of(e) != view.page_of(e2)) n += (uint32_t)(len - e2 < 64 ? len - e2 : 64);
                view.n_access += n;
                view.n_hit += n;
            }
        }
    }
    if (any_left) note_work_left(finished, call);
    view.flush_stats();
}

// ---- scan (benchmarks/scan/main.cu:147-190 kernel_scan_baseline_ptr_pc, :89-100 finalsum) ----
/* inclusive sums over the 64 lanes of a wave (all lanes active) */
__device__ __forceinline__ uint64_t wave_inclusive_sum(uint64_t v)
{
    const uint32_t lane = bam::lane();
#pragma unroll
    for (uint32_t o = 1; o < BAM_WAVE_SIZE; o <<= 1) {
        const uint64_t u = bam::shfl(v, lane >= o ? lane - o : lane);
        if (lane >= o) v += u;
    }
    return v;
}

/*
 * Block b scans its 2 x blockDim elements: output[i] = sum of the block's elements up to and including i,
 * intermediate[b] = the block's total.  The elements are read as the reference reads them (thread t takes t and
 * t + blockDim, so a wave reads consecutive elements through one page reference); the scan itself runs over wave
 * shuffles on pairs of neighbours rather than the two tree passes over shared memory.
 */
__global__ void k_scan_ptr_pc(array_d_t<uint64_t>* da, unsigned long long* output, unsigned long long* intermediate, uint64_t len, const fetch_plan fp)
{
    extern __shared__ uint64_t scan_mem[];                      /* 2 x blockDim elements, then one total per wave */
    if (fp.done && blockIdx.x < fp.blocks) {
        array_d_t<uint64_t>* const arrays[1] = {da};
        fetch_role(arrays, len, fp);
        return;
    }
    const uint32_t bid = blockIdx.x - (fp.done ? fp.blocks : 0u);
    const uint32_t B = blockDim.x, t = threadIdx.x;
    uint64_t* wave_total = scan_mem + 2 * B;
    const uint64_t idx = 2ull * bid * B + t;
    {
        bam_ptr<uint64_t> in_ptr(da);
        const bam_ptr<uint64_t>& ptr = in_ptr;
        const uint64_t first = idx - t % BAM_WAVE_SIZE;
        if (first < len) touch_ahead(da, first, len);
        if (first + B < len) touch_ahead(da, first + B, len);
        scan_mem[t] = idx < len ? ptr[idx] : 0;
        scan_mem[t + B] = idx + B < len ? ptr[idx + B] : 0;
    }
    __syncthreads();
    const uint64_t a = scan_mem[2 * t], b = a + scan_mem[2 * t + 1];
    const uint64_t s = wave_inclusive_sum(b);
    if (bam::lane() == BAM_WAVE_SIZE - 1) wave_total[t / BAM_WAVE_SIZE] = s;
    __syncthreads();
    uint64_t before = s - b;
    for (uint32_t w = 0; w < t / BAM_WAVE_SIZE; w++) before += wave_total[w];
    scan_mem[2 * t] = before + a;
    scan_mem[2 * t + 1] = before + b;
    __syncthreads();
    if (idx < len) output[idx] = scan_mem[t];
    if (idx + B < len) output[idx + B] = scan_mem[t + B];
    if (intermediate && t == B - 1) intermediate[bid] = before + b;
    if (fp.done && t == 0) __hip_atomic_fetch_add(fp.done, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

/*
 * The scan of elements that are resident, in one reading.  A workgroup holds a tile of 16384 elements in registers, tells the
 * others its sum, adds up what lies before it and writes the running sums.  What lies before: the tiles' sums, back to the nearest
 * tile that has told the sum of everything up to its end; a wave looks at 64 of them at a time (the decoupled look-back of Merrill
 * and Garland, "Single-pass parallel prefix scan with decoupled look-back", 2016).
 *   The workgroups of a launch are started in the order of their numbers on each cluster of compute units, so of one scan the first
 * unfinished tile runs, or will once something ends that waits for no tile.  Two scans at a time, on different streams,
 * could each fill a cluster that a tile of the other's is to run on, and wait for each other: a scan that begins while another is on
 * its way draws the numbers of its tiles from one word instead (next_tile), so that all before a tile have begun, and of those that do
 * not draw there is never more than one (host_word::alone).  Always drawing costs the device 20 ns a tile: 2^26 elements 239 -> 257 us,
 * 2^22 28.4 -> 33.1.  Against another process's scan there is the end of all waits, after 20 ms or when somebody has given up.
 *   A word of a tile is 32 bits of a sum and the number of the call: it says by itself whether it has been written, and nothing
 * has to be cleared or ordered.
 *   Bound by HBM: 16 bytes per element.  2^26 elements: 314 -> 245 us a call (4.4 TB/s; a copy of as much on this device 4.9), 2^25
 * 171 -> 130, 2^22 45 -> 34, 2^16 30 -> 27, 4099 28 -> 22, against two launches of which the first added up and the second
 * read the elements again.  While a tile waits another has to load: two of 16 waves fit a compute unit with 64 registers a lane
 * (four are spilled); with 68, one, 272 us; tiles of 8 waves, three to a compute unit, 293 (twice as many sums to look back over).
 *   A page that is not resident: the wave tells the other workgroups and the host, which then runs the kernels that can miss.
 */
#define BAM_TILE_WAVES 16u
#define BAM_TILE_ELEMS (BAM_TILE_WAVES * BAM_WAVE_ELEMS)
#define BAM_SCAN_WAIT_TICKS 2000000ull      /* of the 100 MHz clock */
#define BAM_COUNTED_WORD 98u      /* of the scratch's words: the call whose accesses were counted */
__device__ __forceinline__ void scan_gives_up(uint32_t* finished, const uint32_t call, volatile uint32_t* host_left)
{
    if (bam::lane() == 0 && __hip_atomic_load(finished + BAM_LEFT_WORD, __ATOMIC_RELAXED, BAM_AGENT) != call &&
        __hip_atomic_exchange(finished + BAM_LEFT_WORD, call, __ATOMIC_RELAXED, BAM_AGENT) != call) *host_left = call;
}
/* [0, 1] the tile's sum, [2, 3] the sum of all elements up to its end */
struct scan_tile_t { uint64_t word[4]; };
__device__ __forceinline__ void scan_tell(uint64_t* word, const uint64_t sum, const uint32_t call)
{
    bam::st_relaxed(word, ((uint64_t)call << 32) | (uint32_t)sum);
    bam::st_relaxed(word + 1, ((uint64_t)call << 32) | (uint32_t)(sum >> 32));
}
/* by a whole wave: the sum of everything before tile `tile` */
__device__ __forceinline__ uint64_t scan_look_back(const scan_tile_t* tiles, const uint64_t tile, const uint32_t call, uint32_t* finished, volatile uint32_t* host_left)
{
    const uint32_t lane = bam::lane();
    uint64_t acc = 0, t0 = 0;
    for (uint64_t end = tile;; end -= BAM_WAVE_SIZE) {
        /* lane l: tile end - 1 - l; before the first there is nothing, known for sure */
        const bool there = lane < end;
        const scan_tile_t* const at = tiles + (there ? end - 1 - lane : 0);
        uint64_t sum = 0;
        bool known = !there, all = !there;
        for (uint32_t looks = 1;; looks++) {
            if (!known || !all) {
                const uint64_t a0 = bam::ld_relaxed(&at->word[0]), a1 = bam::ld_relaxed(&at->word[1]), b0 = bam::ld_relaxed(&at->word[2]), b1 = bam::ld_relaxed(&at->word[3]);
                if ((uint32_t)(b0 >> 32) == call && (uint32_t)(b1 >> 32) == call) { sum = (b1 << 32) | (uint32_t)b0; known = all = true; }
                else if ((uint32_t)(a0 >> 32) == call && (uint32_t)(a1 >> 32) == call) { sum = (a1 << 32) | (uint32_t)a0; known = true; }
            }
            const uint64_t m = bam::ballot(all);
            const uint64_t need = m ? (m & (0ull - m)) | ((m & (0ull - m)) - 1) : ~0ull;      /* up to the nearest that has it all */
            if ((bam::ballot(known) & need) == need) {
                acc += wave_sum((need >> lane) & 1 ? sum : 0);
                if (m) return acc;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            if ((looks & 1023u) == 0) {
                const uint64_t now = wall_clock64();
                if (!t0) t0 = now;
                else if (now - t0 > BAM_SCAN_WAIT_TICKS) { scan_gives_up(finished, call, host_left); return acc; }
                if (__hip_atomic_load(finished + BAM_LEFT_WORD, __ATOMIC_RELAXED, BAM_AGENT) == call) return acc;      /* nobody wants the result */
            }
        }
    }
}
/* n_access: what the scan counts, as the kernels that can miss count it */
__global__ __launch_bounds__(BAM_TILE_WAVES * BAM_WAVE_SIZE) __attribute__((amdgpu_waves_per_eu(8))) void k_scan_tiles(array_d_t<uint64_t>* da, uint64_t* result, const uint64_t n, scan_tile_t* tiles, uint32_t* finished,
                                                                               const uint32_t call, volatile uint32_t* host_left, const uint64_t n_access, uint32_t* next_tile)
{
    __shared__ uint64_t wave_sums[BAM_TILE_WAVES], before_s;

    const uint32_t lane = bam::lane(), w = bam::first(threadIdx.x / BAM_WAVE_SIZE);
    bam::range_view<uint64_t> view;
    view.load(da->d_ranges);
    uint32_t tile_drawn = blockIdx.x;
    if (next_tile) {
        __shared__ uint32_t drawn;
        if (threadIdx.x == 0) {
            drawn = __hip_atomic_fetch_add(next_tile, 1u, __ATOMIC_RELAXED, BAM_AGENT);
            if (drawn == gridDim.x - 1) bam::st_relaxed(next_tile, 0u);      /* the last one: the next scan starts over */
        }
        __syncthreads();
        tile_drawn = bam::first(drawn);
    }
    const uint64_t tile = tile_drawn, first = tile * BAM_TILE_ELEMS + w * BAM_WAVE_ELEMS;
    /* once somebody has given up the result is not wanted: the tile is told as it is */
    const bool given_up = __hip_atomic_load(finished + BAM_LEFT_WORD, __ATOMIC_RELAXED, BAM_AGENT) == call;
    bam::u64x2_t x[BAM_WAVE_ROWS];
    if (given_up || !read_rows_resident(view, first, n, x)) {
        if (!given_up) scan_gives_up(finished, call, host_left);
#pragma unroll
        for (uint32_t r = 0; r < BAM_WAVE_ROWS; r++) x[r] = bam::u64x2_t{0, 0};
    }
    uint64_t v = 0;
#pragma unroll
    for (uint32_t r = 0; r < BAM_WAVE_ROWS; r++) v += x[r].x + x[r].y;
    v = wave_sum(v);
    if (lane == 0) wave_sums[w] = v;
    __syncthreads();
    if (w == 0) {
        uint64_t total = 0;
#pragma unroll
        for (uint32_t k = 0; k < BAM_TILE_WAVES; k++) total += wave_sums[k];
        if (lane == 0 && tile) scan_tell(tiles[tile].word, total, call);
        const uint64_t before = tile ? scan_look_back(tiles, tile, call, finished, host_left) : 0;
        if (lane == 0) { scan_tell(tiles[tile].word + 2, before + total, call); before_s = before; }
    }
    __syncthreads();
    if (!given_up && first <= n) {
        uint64_t carry = before_s;
#pragma unroll
        for (uint32_t k = 0; k < BAM_TILE_WAVES; k++) carry += k < w ? wave_sums[k] : 0;
        /* entry e is the sum of the elements before element e, the last one, n, the total */
#pragma unroll
        for (uint32_t r = 0; r < BAM_WAVE_ROWS; r++) {
            const uint64_t pair = x[r].x + x[r].y, incl = bam::wave_running_sum(pair), sum = carry + (incl - pair);
            carry += bam::bcast(incl, BAM_WAVE_SIZE - 1);
            const uint64_t e = first + r * BAM_ROW_ELEMS + 2u * lane;
            if (first + BAM_WAVE_ELEMS <= n + 1) __builtin_nontemporal_store(bam::u64x2_t{sum, sum + x[r].x}, (bam::u64x2_t*)(result + e));
            else {
                if (e <= n) result[e] = sum;
                if (e + 1 <= n) result[e + 1] = sum + x[r].x;
            }
        }
    }
    if (tile == 0 && threadIdx.x == 0) {
        bam_stat_shard_t* const sh = view.r->shard();
        __hip_atomic_fetch_add(&sh->access_cnt, (unsigned long long)n_access, __ATOMIC_RELAXED, BAM_AGENT);
        __hip_atomic_fetch_add(&sh->hit_cnt, (unsigned long long)n_access, __ATOMIC_RELAXED, BAM_AGENT);
        finished[BAM_COUNTED_WORD] = call;
    }
}
/* behind a k_scan_tiles of which some wave gave up: the kernels that can miss count the whole scan, so what its first
 * workgroup counted (it does not wait for the others) is taken off again */
__global__ void k_scan_uncount(array_d_t<uint64_t>* da, const uint32_t* finished, const uint32_t call, const uint64_t n_access)
{
    if (finished[BAM_COUNTED_WORD] != call) return;
    bam_stat_shard_t* const sh = da->d_ranges->shard();
    __hip_atomic_fetch_add(&sh->access_cnt, 0ull - n_access, __ATOMIC_RELAXED, BAM_AGENT);
    __hip_atomic_fetch_add(&sh->hit_cnt, 0ull - n_access, __ATOMIC_RELAXED, BAM_AGENT);
}

/* one block: v[i] = v[0] + ... + v[i] in place (the reference calls cub::DeviceScan::InclusiveSum here, scan/main.cu:416-418) */
__global__ void k_scan_block_totals(unsigned long long* v, uint64_t n)
{
    __shared__ uint64_t wave_total[1024 / BAM_WAVE_SIZE];
    __shared__ uint64_t carry_s;
    const uint32_t t = threadIdx.x;
    if (t == 0) carry_s = 0;
    __syncthreads();
    for (uint64_t base = 0; base < n; base += blockDim.x) {
        const uint64_t x = base + t < n ? v[base + t] : 0;
        const uint64_t s = wave_inclusive_sum(x);
        if (bam::lane() == BAM_WAVE_SIZE - 1) wave_total[t / BAM_WAVE_SIZE] = s;
        __syncthreads();
        uint64_t r = carry_s + s;
        for (uint32_t w = 0; w < t / BAM_WAVE_SIZE; w++) r += wave_total[w];
        if (base + t < n) v[base + t] = r;
        __syncthreads();
        if (t == blockDim.x - 1) carry_s = r;
        __syncthreads();
    }
}

__global__ void k_scan_finalsum(const unsigned long long* scanned_totals, unsigned long long* output, uint64_t len)
{
    if (blockIdx.x == 0) return;
    const uint64_t B = blockDim.x, idx = 2ull * blockIdx.x * B + threadIdx.x;
    const uint64_t add = scanned_totals[blockIdx.x - 1];
    if (idx < len) output[idx] += add;
    if (idx + B < len) output[idx + B] += add;
}

/*
 * Whether bam_reduce and bam_scan read what is resident first, without references: arrays of one range whose element 0 is
 * the first of a page, with the elements asked for in no more pages than the cache has (otherwise some are missing for sure,
 * and the kernels that can miss do it all), and no capture (the launches work in buffers that are kept between calls).
 */
bool resident_first(bam_array_t* a, uint64_t n_elems, hipStream_t st)
{
    if (!two_launches_ok(a)) return false;
    const range_d_t<uint64_t>& r = a->a->h_ranges[0];
    if (r.index_start || r.page_start_offset || n_elems > r.count || r.cache.page_size < 512) return false;
    if ((n_elems * sizeof(uint64_t) + r.cache.page_size - 1) / r.cache.page_size > r.cache.n_pages) return false;
    return !is_captured(st);
}

/*
 * The accesses a reduction or scan of n elements counts with workgroups of `half` threads when all is resident: thread t of
 * a workgroup reads elements t and t + half of its 2 half, one access each unless they lie on the same page.  The second
 * elements on another page than their first are those within `half` behind a page boundary; where boundaries lie in a
 * workgroup repeats, and one period stands for all that are complete.
 */
uint64_t paired_accesses(uint64_t n, uint64_t half, uint64_t page_elems)
{
    if (half >= page_elems) return n;
    auto behind = [&](uint64_t boundary) {
        const uint64_t in_half = boundary % half, lo = boundary / half & 1 ? boundary : boundary + half - in_half, hi = boundary / half & 1 ? boundary + half - in_half : boundary + half;
        return std::min(hi, n) - std::min(lo, n);
    };
    uint64_t total = n / (2 * half) * half + std::min(half, n % (2 * half)), period = 1;
    while (period * page_elems % (2 * half)) period++;
    const uint64_t complete = n > half ? (n - half) / page_elems / period * period : 0;
    if (complete) {
        uint64_t one = 0;
        for (uint64_t k = 1; k <= period; k++) one += behind(k * page_elems);
        total += one * (complete / period);
    }
    for (uint64_t k = complete + 1; k * page_elems < n; k++) total += behind(k * page_elems);
    return total;
}

/*
 * A word in host memory that the device can write, one call's own for as long as it lasts: a scan waits for its result, and
 * finds there whether it is whole.  Page-locked memory takes far longer to get than a scan does, so the words are kept for the
 * next call, whichever array or thread makes it; there are as many as calls were ever waiting at a time, in steps of 64.
 * Words that launches may still write (the wait failed) are not given back.  `at` is NULL where no memory is to be had.
 */
struct host_word {
    volatile uint32_t* at = nullptr;
    bool idle = true;
    bool alone = false;             /* no other word was out when this one was taken */
    host_word()
    {
        pool& p = shared();
        std::lock_guard<std::mutex> guard(p.mu);
        if (p.free.empty()) {
            const relaxed_capture relaxed;
            void* mem = nullptr;
            if (hipHostMalloc(&mem, 64 * sizeof(uint32_t), hipHostMallocMapped | hipHostMallocPortable) != hipSuccess) { (void)hipGetLastError(); return; }
            for (uint32_t k = 0; k < 64; k++) p.free.push_back((volatile uint32_t*)mem + k);
            p.made += 64;
        }
        alone = p.free.size() == p.made;
        at = p.free.back();
        p.free.pop_back();
        at[0] = 0;                  /* never the number of a call */
    }
    ~host_word()
    {
        if (!at || !idle) return;
        pool& p = shared();
        std::lock_guard<std::mutex> guard(p.mu);
        p.free.push_back(at);
    }
    host_word(const host_word&) = delete;
    host_word& operator=(const host_word&) = delete;

private:
    struct pool { std::mutex mu; std::vector<volatile uint32_t*> free; size_t made = 0; };
    static pool& shared() { static pool* p = new pool(); return *p; }      /* never taken down: the runtime may be gone by then */
};

/*
 * Whole pages of the three arrays (k_vectoradd_resident); false, with nothing launched, where they do not lend themselves to it:
 * arrays of one range whose element 0 is the first of a page, behind one cache of pages that fit a staging page, one
 * controller, no capture (the launches keep notes for each other), memory for the notes.
 */
bool vectoradd_by_page(bam_array_t* a, bam_array_t* b, bam_array_t* c, uint64_t n_elems, hipStream_t st)
{
    uint64_t pages = 0;
    bam_array_t* const all[3] = {a, b, c};
    const page_cache_d_t* cache = nullptr;
    for (int k = 0; k < 3; k++) {
        if (all[k]->a->adt.n_ranges != 1) return false;
        const range_d_t<uint64_t>& r = all[k]->a->h_ranges[0];
        if (r.index_start || r.page_start_offset % r.cache.page_size || n_elems > r.count) return false;
        if (cache && cache->base_addr != r.cache.base_addr) return false;
        cache = &r.cache;
        pages += (n_elems * sizeof(uint64_t) + r.cache.page_size - 1) / r.cache.page_size;
    }
    if (cache->n_ctrls != 1 || (cache->page_size != 4096 && cache->page_size != 8192) || cache->page_size > cache->stage_bytes) return false;
    const uint64_t n_full = n_elems * sizeof(uint64_t) / cache->page_size;
    if (!n_full || n_full > 0xFFFFFFFFull || is_captured(st)) return false;
    uint32_t chunk = 16;
    const uint64_t budget = cache->n_pages / 2;
    while (chunk > 4 && budget / (3 * chunk) < 256) chunk /= 2;
    const uint64_t waves = budget / (3 * chunk);
    if (!waves) return false;
    std::lock_guard<std::mutex> guard(c->scratch.mu);
    scratch_set* set = scratch_for(c, st, n_full * (sizeof(uint32_t) + 1), 0);
    if (!set) return false;
    vadd_t g{a->a->d_array_ptr, b->a->d_array_ptr, c->a->d_array_ptr, n_elems, n_full, pages > cache->n_pages ? 1u : 0u, (uint8_t*)set->notes.get() + n_full * sizeof(uint32_t),
             (uint32_t*)set->notes.get(), set->listed(), set->next_chunk(), set->finished(), set->next_call()};
    hipLaunchKernelGGL(k_vectoradd_resident, dim3((uint32_t)((n_full + BAM_VADD_PAGES - 1) / BAM_VADD_PAGES) + blocks_for(n_elems - n_full * (cache->page_size / sizeof(uint64_t)), BAM_WAVE_SIZE)),
                       dim3(BAM_WAVE_SIZE), 0, st, g);
    hipLaunchKernelGGL(k_vectoradd_missing, dim3((uint32_t)std::min<uint64_t>(waves, (n_full + chunk - 1) / chunk)), dim3(BAM_WAVE_SIZE), 0, st, g, chunk);
    hipLaunchKernelGGL(k_vectoradd_rest, dim3((uint32_t)std::min<uint64_t>(n_full, std::min<uint64_t>(4096, cache->n_pages / 8))), dim3(BAM_WAVE_SIZE), 0, st, g);      /* a wave holds a page of each array */
    hip_err_chk(hipGetLastError());
    return true;
}

/*
 * Waves for k_vectoradd_ptr_pc: one per 64 elements, unless those that the device runs at a time could hold the pages of all slots.  A
 * wave keeps its page of A while it waits for a slot for B's, and both while it waits for C's, so that they then wait for each
 * other until the bounded waits give up, and the sums are wrong (three times 65 pages of 8 KiB behind 97 slots: now and then).  As
 * many as have a slot for each of their three pages do not.
 */
uint32_t vectoradd_waves(bam_array_t* a, bam_array_t* b, bam_array_t* c, uint64_t n_elems)
{
    uint64_t slots = ~0ull, held = 0;
    for (bam_array_t* x : {a, b, c}) {
        uint64_t pages = 0;
        for (uint32_t k = 0; k < x->a->adt.n_ranges; k++) {
            const range_d_t<uint64_t>& r = x->a->h_ranges[k];
            slots = std::min<uint64_t>(slots, r.cache.n_pages);
            pages += r.page_count;
        }
        if (x != c) held += pages;                /* who holds a page of C waits for nothing */
    }
    const uint32_t waves = blocks_for(n_elems, BAM_WAVE_SIZE);
    int dev = 0, units = 0, per_unit = 0;
    hip_err_chk(hipGetDevice(&dev));
    hip_err_chk(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, dev));
    hip_err_chk(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_unit, k_vectoradd_ptr_pc, BAM_WAVE_SIZE, 0));
    held = std::min(held, 2 * std::min<uint64_t>(waves, (uint64_t)units * per_unit));
    return held < slots ? waves : (uint32_t)std::min<uint64_t>(waves, std::max<uint64_t>(1, slots / 3));
}

/* the scan of resident elements; false if some were not, and then the result is not written in full, or if there is no
 * memory for the sums */
bool scan_resident(bam_array_t* a, uint64_t n_elems, uint32_t block_size, uint64_t* d_result, hipStream_t st)
{
    host_word left;
    if (!left.at) return false;
    uint32_t call;
    uint32_t* finished;
    const uint64_t n_access = paired_accesses(n_elems, block_size, a->a->h_ranges[0].cache.page_size / 8);
    {
        const uint64_t n_tiles = n_elems / BAM_TILE_ELEMS + 1;          /* entry n of the result is in the last */
        std::lock_guard<std::mutex> guard(a->scratch.mu);
        scratch_set* set = scratch_for(a, st, 0, 0, n_tiles * sizeof(scan_tile_t));
        if (!set) return false;
        call = set->next_call();
        finished = set->finished();
        left.idle = false;          /* (until the wait is over) */
        hipLaunchKernelGGL(k_scan_tiles, dim3((uint32_t)n_tiles), dim3(BAM_TILE_WAVES * BAM_WAVE_SIZE), 0, st, a->a->d_array_ptr, d_result, n_elems, (scan_tile_t*)set->tiles.get(), finished, call,
                           left.at, n_access, left.alone ? nullptr : set->next_tile());
        hip_err_chk(hipGetLastError());
    }
    const hipError_t e = hipStreamSynchronize(st);
    left.idle = e == hipSuccess;
    hip_err_chk(e);
    if (left.at[0] != call) return true;
    hipLaunchKernelGGL(k_scan_uncount, dim3(1), dim3(1), 0, st, a->a->d_array_ptr, finished, call, n_access);
    hip_err_chk(hipGetLastError());
    return false;
}

} // namespace

extern "C" {

int bam_vectoradd(bam_array_t* a, bam_array_t* b, bam_array_t* c, uint64_t n_elems, void* stream)
{
    if (!a || !b || !c) return fail(EINVAL, "bam_vectoradd: null argument");
    if (n_elems > a->a->adt.n_elems || n_elems > b->a->adt.n_elems || n_elems > c->a->adt.n_elems) return fail(EINVAL, "bam_vectoradd: more elements than the arrays hold");
    if (!n_elems) return 0;
    BAM_API_BEGIN
    if (vectoradd_by_page(a, b, c, n_elems, (hipStream_t)stream)) return 0;
    const fetch_plan fp = make_fetch_plan(a, 3, 64, 64, (hipStream_t)stream);
    hipLaunchKernelGGL(k_vectoradd_ptr_pc, dim3(vectoradd_waves(a, b, c, n_elems) + fp.blocks), dim3(64), 0, (hipStream_t)stream,
                       a->a->d_array_ptr, b->a->d_array_ptr, n_elems, c->a->d_array_ptr, fp);
    hip_err_chk(hipGetLastError());
    BAM_API_END
}

int bam_reduce(bam_array_t* a, uint64_t n_elems, uint32_t block_size, uint64_t* d_partials, void* stream)
{
    if (!a || !d_partials) return fail(EINVAL, "bam_reduce: null argument");
    if (!block_size || block_size % BAM_WAVE_SIZE || block_size > 1024) return fail(EINVAL, "bam_reduce: block size must be a multiple of 64, at most 1024");
    if (n_elems > a->a->adt.n_elems) return fail(EINVAL, "bam_reduce: more elements than the array holds");
    if (!n_elems) return 0;
    BAM_API_BEGIN
    const uint64_t n_outputs = blocks_for(n_elems, 2ull * block_size);
    /* two launches instead of one: 4 us more per call, made up for from here on (blocks of 64: 21 against 16 us at 2^16 elements;
     * blocks of 256: 15 against 17 there, 17 both at 2^17, 20 against 17 at 2^18) */
    if ((n_elems >= 1ull << 17 || n_outputs >= 512) && resident_first(a, n_elems, (hipStream_t)stream)) {
        hipStream_t st = (hipStream_t)stream;
        /* outputs per turn of a wave: as many as its rows hold, one at least (of more than eight rows, read in two goes) */
        const uint32_t rows = block_size / BAM_WAVE_SIZE, per_note = rows < BAM_WAVE_ROWS ? BAM_WAVE_ROWS / rows : 1;
        const uint64_t n_turns = (n_outputs + per_note - 1) / per_note;
        std::lock_guard<std::mutex> guard(a->scratch.mu);
        if (scratch_set* set = scratch_for(a, st, n_turns, 0)) {
            uint8_t* notes = (uint8_t*)set->notes.get();
            const uint32_t call = set->next_call();
            hipLaunchKernelGGL(k_reduce_resident, dim3((uint32_t)std::min<uint64_t>((n_turns + 3) / 4, 2048)), dim3(256), 0, st, a->a->d_array_ptr, (unsigned long long*)d_partials, n_elems,
                               n_outputs, rows, per_note, notes, set->finished(), call, set->done());
            const uint32_t groups = block_size <= 128 ? 256 / block_size : 1, threads = groups * block_size;
            const fetch_plan fp = make_fetch_plan(a, 1, threads, 2ull * block_size, st, set->done());
            const uint64_t at_a_time = (uint64_t)BAM_REST_WAVES * BAM_WAVE_SIZE / threads;
            hipLaunchKernelGGL(k_reduce_rest, dim3((uint32_t)std::min<uint64_t>((n_outputs + groups - 1) / groups, at_a_time) + fp.blocks), dim3(threads), 0, st, a->a->d_array_ptr,
                               (unsigned long long*)d_partials, n_elems, n_outputs, block_size, per_note, notes, set->finished(), call, fp);
            hip_err_chk(hipGetLastError());
            return 0;
        }
    }
    const fetch_plan fp = make_fetch_plan(a, 1, block_size, 2ull * block_size, (hipStream_t)stream);
    hipLaunchKernelGGL(k_reduce_ptr_pc, dim3(n_outputs + fp.blocks), dim3(block_size), 0, (hipStream_t)stream,
                       a->a->d_array_ptr, (unsigned long long*)d_partials, n_elems, fp);
    hip_err_chk(hipGetLastError());
    BAM_API_END
}

int bam_scan(bam_array_t* a, uint64_t n_elems, uint32_t block_size, uint64_t* d_result, void* stream)
{
    if (!a || !d_result) return fail(EINVAL, "bam_scan: null argument");
    if (!block_size || block_size % BAM_WAVE_SIZE || block_size > 1024) return fail(EINVAL, "bam_scan: block size must be a multiple of 64, at most 1024");
    if (n_elems > a->a->adt.n_elems) return fail(EINVAL, "bam_scan: more elements than the array holds");
    BAM_API_BEGIN
    hipStream_t st = (hipStream_t)stream;
    const bool kept = n_elems && (uintptr_t)d_result % 16 == 0 && resident_first(a, n_elems, st);
    if (kept && scan_resident(a, n_elems, block_size, d_result, st)) return 0;
    hip_err_chk(hipMemsetAsync(d_result, 0, sizeof(uint64_t), st));
    if (n_elems) {
        const uint64_t n_blocks = blocks_for(n_elems, 2ull * block_size);
        /* the block totals: in the scratch of a call that has just looked for resident pages, else in memory of their own */
        BufferPtr own;
        unsigned long long* totals = nullptr;
        std::unique_lock<std::mutex> guard(a->scratch.mu, std::defer_lock);
        if (kept) {
            guard.lock();
            if (scratch_set* set = scratch_for(a, st, n_blocks * sizeof(uint64_t), 0)) totals = (unsigned long long*)set->notes.get();
            else guard.unlock();
        }
        if (!totals) {
            own = createBuffer(n_blocks * sizeof(uint64_t), 0);
            totals = (unsigned long long*)own.get();
        }
        unsigned long long* out = (unsigned long long*)d_result + 1;
        const size_t lds = (2 * block_size + 1024 / BAM_WAVE_SIZE) * sizeof(uint64_t);
        const fetch_plan fp = make_fetch_plan(a, 1, block_size, 2ull * block_size, st);
        hipLaunchKernelGGL(k_scan_ptr_pc, dim3(n_blocks + fp.blocks), dim3(block_size), lds, st, a->a->d_array_ptr, out, totals, n_elems, fp);
        hipLaunchKernelGGL(k_scan_block_totals, dim3(1), dim3(1024), 0, st, totals, n_blocks);
        hipLaunchKernelGGL(k_scan_finalsum, dim3(n_blocks), dim3(block_size), 0, st, totals, out, n_elems);
        hip_err_chk(hipGetLastError());
        if (guard.owns_lock()) guard.unlock();
        hip_err_chk(hipStreamSynchronize(st));         /* `own` is released on return */
    }
    BAM_API_END
}

} // extern "C"

/*
 * bam_scan for callers that cannot allocate (code under stream capture, serving loops, harnesses that forbid it): the block
 * totals, which bam_scan keeps in a buffer it allocates and frees per call, live in a file-scope device array of fixed size.
 * Every device the library runs on holds its own copy of the array at its own address until the process ends; the address is
 * looked up once per device (the array's name means nothing to the host) and handed to the kernels like any other buffer.
 */
/* BAM_SCAN_NOALLOC_MAX_BLOCKS (bam_amd.h): 65536 block totals, 512 KiB */
#define BAM_SCAN_NOALLOC_MAX_DEVICES 64
static __device__ __align__(256) unsigned long long scratch[BAM_SCAN_NOALLOC_MAX_BLOCKS];

namespace {
std::mutex g_scratch_mu;
unsigned long long* g_scratch_ptr[BAM_SCAN_NOALLOC_MAX_DEVICES];      /* per device: where its copy of `scratch` lives */

/* the current device's copy of the array; NULL (and the error recorded) if it cannot be found */
unsigned long long* scan_scratch_of_current_device()
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= BAM_SCAN_NOALLOC_MAX_DEVICES) { g_err = "bam_scan_noalloc: no current device"; return nullptr; }
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) { g_err = std::string("bam_scan_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e); return nullptr; }
        g_scratch_ptr[dev] = (unsigned long long*)p;
    }
    return g_scratch_ptr[dev];
}

} // namespace

extern "C" {

int bam_scan_noalloc(bam_array_t* a, uint64_t n_elems, uint32_t block_size, uint64_t* d_result, void* stream)
{
    if (!a || !d_result) return fail(EINVAL, "bam_scan_noalloc: null argument");
    if (!block_size || block_size % BAM_WAVE_SIZE || block_size > 1024) return fail(EINVAL, "bam_scan_noalloc: block size must be a multiple of 64, at most 1024");
    if (n_elems > a->a->adt.n_elems) return fail(EINVAL, "bam_scan_noalloc: more elements than the array holds");
    const uint64_t n_blocks = (n_elems + 2ull * block_size - 1) / (2ull * block_size);
    if (n_blocks > BAM_SCAN_NOALLOC_MAX_BLOCKS)
        return fail(E2BIG, "bam_scan_noalloc: " + std::to_string(n_elems) + " elements in blocks of " + std::to_string(2ull * block_size) + " need " + std::to_string(n_blocks) +
                           " block totals, the fixed scratch array holds " + std::to_string(BAM_SCAN_NOALLOC_MAX_BLOCKS) + " (use bam_scan, or a larger block size)");
    unsigned long long* totals = scan_scratch_of_current_device();
    if (!totals) return EIO;
    hipStream_t st = (hipStream_t)stream;
    unsigned long long* out = (unsigned long long*)d_result + 1;
    /* no memset node: a fill kernel clears the first word (a caller may be capturing this stream) */
    hipLaunchKernelGGL(k_store_zero64, dim3(1), dim3(1), 0, st, (unsigned long long*)d_result);
    if (n_elems) {
        /* totals[0 .. n_blocks) are written by the first kernel before the second reads them; what an earlier, longer call
         * left behind them is never read, so nothing has to be cleared */
        const size_t lds = (2 * block_size + 1024 / BAM_WAVE_SIZE) * sizeof(uint64_t);
        /* no fetch waves here: their counter would have to be allocated and cleared */
        const fetch_plan none{nullptr, 0, 0, 0, 0};
        hipLaunchKernelGGL(k_scan_ptr_pc, dim3((uint32_t)n_blocks), dim3(block_size), lds, st, a->a->d_array_ptr, out, totals, n_elems, none);
        hipLaunchKernelGGL(k_scan_block_totals, dim3(1), dim3(1024), 0, st, totals, n_blocks);
        hipLaunchKernelGGL(k_scan_finalsum, dim3((uint32_t)n_blocks), dim3(block_size), 0, st, (const unsigned long long*)totals, out, n_elems);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(EIO, std::string("bam_scan_noalloc: ") + hipGetErrorString(e));
    return 0;
}

} // extern "C"
