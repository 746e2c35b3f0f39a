// Checks of what calls in several launches keep between them (bam_amd/csrc/scratch_sets.h), with an allocator that can be made
// to refuse.  No GPU.  Prints "ok <name>" per check; exit 0 = all passed.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <thread>
#include "along_tables.h"
#include "scratch_sets.h"

static int failures = 0;
#define CHECK(name, cond) do { if (cond) printf("ok %s\n", name); else { printf("FAIL %s (%s:%d)\n", name, __FILE__, __LINE__); failures++; } } while (0)

struct Memory {
    int allocs = 0, frees = 0, refuse_from = -1;
    std::map<void*, size_t> live;
    std::shared_ptr<void> operator()(size_t bytes)
    {
        if (refuse_from >= 0 && allocs >= refuse_from) return nullptr;
        allocs++;
        void* p = calloc(1, bytes);
        live[p] = bytes;
        return std::shared_ptr<void>(p, [this](void* q) { live.erase(q); frees++; free(q); });
    }
    bool holds(const std::shared_ptr<void>& b, size_t bytes) const { auto it = live.find(b.get()); return it != live.end() && it->second >= bytes; }
};
static void* stream(uintptr_t k) { return (void*)(0x1000 * k); }
static bool whole(const Memory& m, scratch_set* s, size_t notes, size_t wanted)
{
    return s && m.holds(s->words, BAM_SCRATCH_WORDS_BYTES) && m.holds(s->notes, notes) && (!wanted || m.holds(s->wanted, wanted));
}

int main()
{
    /* a refusal at every place a call can meet one: the call gets nothing, and the next one a whole set */
    for (int at = 0; at < 3; at++) {
        Memory mem;
        {
            scratch_sets sets;
            auto alloc = [&](size_t b) { return mem(b); };
            mem.refuse_from = at;
            scratch_set* s = sets.get(stream(1), 0, 4096, 512, alloc);
            CHECK("refused: nothing", s == nullptr);
            mem.refuse_from = -1;
            s = sets.get(stream(1), 0, 4096, 512, alloc);
            CHECK("then a whole set", whole(mem, s, 4096, 512));
            mem.refuse_from = mem.allocs;
            CHECK("a larger call is refused", sets.get(stream(1), 0, 8192, 512, alloc) == nullptr);
            CHECK("and the smaller still has its set", sets.get(stream(1), 0, 4096, 512, alloc) == s && whole(mem, s, 4096, 512));
        }
        CHECK("all is given back", mem.live.empty() && mem.frees == mem.allocs);
    }
    /* what the tiles of a scan tell each other, refused: the scan gets nothing, the calls that need none their set, the next scan all of it */
    {
        Memory mem;
        scratch_sets sets;
        auto alloc = [&](size_t b) { return mem(b); };
        mem.refuse_from = 1;
        CHECK("tiles refused", sets.get(stream(1), 0, 0, 0, alloc, 640) == nullptr);
        scratch_set* s = sets.get(stream(1), 0, 0, 0, alloc);
        CHECK("a call without tiles has its set", s && !s->tiles && mem.allocs == 1);
        mem.refuse_from = -1;
        CHECK("then tiles", sets.get(stream(1), 0, 0, 0, alloc, 640) == s && mem.holds(s->tiles, 640));
        /* notes come from an allocator of their own */
        Memory raw;
        CHECK("notes apart", sets.get(stream(1), 0, 4096, 512, alloc, 640, [&](size_t b) { return raw(b); }) == s && raw.holds(s->notes, 4096) && mem.holds(s->wanted, 512));
        s->notes.reset();
    }
    /* one handle that is another stream in each thread: two threads share nothing, each finds its own again */
    {
        Memory mem;
        scratch_sets sets;
        auto alloc = [&](size_t b) { return mem(b); };
        scratch_set* got[2][2] = {};
        uint64_t number[2] = {};
        for (int k = 0; k < 2; k++)
            std::thread([&] {
                number[k] = scratch_thread_number();
                for (int rep = 0; rep < 2; rep++) {
                    std::lock_guard<std::mutex> guard(sets.mu);
                    got[k][rep] = sets.get((void*)2, scratch_thread_number(), 1024, 512, alloc);
                }
            }).join();
        CHECK("threads have numbers of their own", number[0] != number[1] && number[0] && number[1]);
        CHECK("each thread finds its set again", got[0][0] == got[0][1] && got[1][0] == got[1][1]);
        CHECK("threads share no set", got[0][0] != got[1][0] && got[0][0]->notes != got[1][0]->notes && got[0][0]->words != got[1][0]->words && got[0][0]->wanted != got[1][0]->wanted);
    }
    /* streams by turns: after the first round nothing is allocated and nothing moves; a buffer that was replaced is still
     * there (its launches may be queued); beyond the bound a stream gets nothing, and the others keep what they have */
    {
        Memory mem;
        {
            scratch_sets sets;
            auto alloc = [&](size_t b) { return mem(b); };
            std::shared_ptr<void> first[8];
            for (uintptr_t k = 0; k < 8; k++) first[k] = sets.get(stream(k + 1), 0, 1000 + k, 512, alloc)->notes;
            const int allocs = mem.allocs;
            bool same = true;
            for (int rep = 0; rep < 3; rep++)
                for (uintptr_t k = 0; k < 8; k++) same &= sets.get(stream(k + 1), 0, 1000, 512, alloc)->notes == first[k];
            CHECK("eight streams by turns allocate once", same && mem.allocs == allocs && mem.frees == 0);
            void* const before = first[0].get();
            first[0].reset();
            scratch_set* s = sets.get(stream(1), 0, 1001, 512, alloc);
            CHECK("a larger buffer is twice the size, the smaller one stays", whole(mem, s, 2000, 512) && s->notes.get() != before && mem.live.count(before) && mem.frees == 0);
            mem.refuse_from = mem.allocs;
            CHECK("refused: the set keeps what it has", sets.get(stream(1), 0, 5000, 512, alloc) == nullptr && sets.get(stream(1), 0, 2000, 512, alloc) == s);
            mem.refuse_from = -1;
            for (uintptr_t k = 8; k < BAM_SCRATCH_SETS; k++) sets.get(stream(k + 1), 0, 64, 0, alloc);
            const int full = mem.allocs;
            CHECK("no set beyond the bound", sets.get(stream(BAM_SCRATCH_SETS + 1), 0, 64, 0, alloc) == nullptr && mem.allocs == full);
            CHECK("the others keep theirs", sets.get(stream(1), 0, 64, 0, alloc) == s && sets.get(stream(BAM_SCRATCH_SETS), 0, 64, 0, alloc) && mem.frees == 0);
        }
        CHECK("all is given back", mem.live.empty());
    }
    /* the tables of readings along the edge pages: refused, the call goes another way; the bits refused, it goes without them; nothing
     * is asked for that nobody wants, and nothing twice */
    {
        Memory mem;
        {
            along_tables t;
            auto alloc = [&](size_t b) { return mem(b); };
            mem.refuse_from = 0;
            CHECK("tables refused", !t.get(4096, 512, alloc) && !t.tables && !t.bits);
            mem.refuse_from = 1;
            CHECK("bits refused", t.get(4096, 512, alloc) && mem.holds(t.tables, 4096) && !t.bits);
            CHECK("components want none", t.get(4096, 0, alloc) && !t.bits && mem.allocs == 1);
            mem.refuse_from = -1;
            CHECK("a later call gets them", t.get(4096, 512, alloc) && mem.holds(t.bits, 512) && mem.allocs == 2);
            CHECK("once", t.get(4096, 512, alloc) && t.get(4096, 0, alloc) && mem.allocs == 2 && mem.frees == 0);
        }
        CHECK("all is given back", mem.live.empty());
    }
    printf(failures ? "FAILED\n" : "PASSED\n");
    return failures != 0;
}
