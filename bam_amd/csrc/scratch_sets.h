// What the calls of one array that take several launches keep between the launches, and from call to call.  Host side only,
// no HIP in here: the memory comes from the caller's allocator (tests/native/test_scratch.cpp hands in one of its own).
#ifndef __BAM_SCRATCH_SETS_H__
#define __BAM_SCRATCH_SETS_H__
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <memory>
#include <mutex>
#include <vector>

#define BAM_SUM_PARTIALS 4096
#define BAM_SCRATCH_SETS 64
#define BAM_SCRATCH_WORDS_BYTES (BAM_SUM_PARTIALS * sizeof(uint64_t) + 1024)

/*
 * The bits of the requests a first launch leaves, a byte per page of the range that somebody waits for
 * or a count of its requests (zero between calls),
 * what the tiles of a scan tell each other (words that carry the number of their call), checksum shards and the count of finished
 * workgroups.
 */
struct scratch_set {
    void* stream = nullptr;
    uint64_t thread = 0;
    std::shared_ptr<void> words, notes, wanted, tiles;
    size_t notes_bytes = 0, wanted_bytes = 0, tiles_bytes = 0;
    uint32_t calls = 0, updates = 0;
    unsigned long long* partials() { return (unsigned long long*)words.get(); }
    uint32_t* finished() { return (uint32_t*)(partials() + BAM_SUM_PARTIALS); }
    uint32_t next_call() { if (++calls == 0) calls = 1; return calls; }
    /* the word the computing workgroups of a reduction count themselves off in for the fetching ones, on a line of its own */
    unsigned long long* done() { return (unsigned long long*)(finished() + 128); }
    /* how many pages a first launch has listed for the second, and which of them comes next: zero between calls, a line each */
    unsigned long long* listed() { return (unsigned long long*)(finished() + 160); }
    unsigned long long* next_chunk() { return (unsigned long long*)(finished() + 192); }
    /* requests dealt out to their pages so far, and turns of pages taken: the first launch clears them */
    uint32_t* cursor() { return finished() + 144; }
    uint32_t* turns() { return finished() + 176; }
    /* the number of the next tile of a scan that draws them: zero between calls */
    uint32_t* next_tile() { return finished() + 208; }
    /* how many updates a slice has left for its last launch, by turns: the one's word is cleared by the other */
    unsigned long long* left_over(uint32_t which) { return (unsigned long long*)(finished() + (which ? 240 : 224)); }
};

/* a number of the calling thread's own, given out once in the life of the process (the number of a thread that has ended may
 * not come back: its work may still run) */
inline uint64_t scratch_thread_number()
{
    static std::atomic<uint64_t> last{0};
    thread_local const uint64_t mine = ++last;
    return mine;
}

/*
 * One set per stream, because the launches of two calls on one stream run one after the other and those on two streams do
 * not; the set is picked and its launches are queued under the mutex, so the calls of two threads on one stream do not mix.
 * One handle, hipStreamPerThread, names another stream in each thread: its sets belong to the thread as well.
 * A set stays where it is until the array goes, and so does a buffer that a larger one has replaced (the larger one is twice
 * its size or more, so that all of them together are no larger than the last): launches that use them may still be queued, and
 * to wait for them would hold up every stream of the device.  BAM_SCRATCH_SETS bounds the sets; a stream for which none is left
 * takes the routes that need none.
 */
struct scratch_sets {
    std::mutex mu;
    std::vector<std::unique_ptr<scratch_set>> sets;
    std::vector<std::shared_ptr<void>> replaced;
    /*
     * The set of `stream` (and of `thread`, 0 where the handle names one stream everywhere) with at least these sizes, with `mu` held; NULL where the memory is refused, and then the caller
     * takes a route that needs none.  alloc(bytes) gives memory that is zero to what is queued on `stream` from now on, or NULL;
     * alloc_notes(bytes) memory for the notes, which every call writes before it reads them, whatever another left there.
     * A set is entered once all of it is there, and a buffer changes place with a larger one that is there.
     */
    template <typename Alloc>
    scratch_set* get(void* stream, uint64_t thread, size_t notes_bytes, size_t wanted_bytes, Alloc&& alloc, size_t tiles_bytes = 0)
    {
        return get(stream, thread, notes_bytes, wanted_bytes, alloc, tiles_bytes, alloc);
    }
    template <typename Alloc, typename AllocNotes>
    scratch_set* get(void* stream, uint64_t thread, size_t notes_bytes, size_t wanted_bytes, Alloc&& alloc, size_t tiles_bytes, AllocNotes&& alloc_notes)
    {
        scratch_set* s = nullptr;
        for (auto& x : sets) if (x->stream == stream && x->thread == thread) s = x.get();
        if (!s && sets.size() >= BAM_SCRATCH_SETS) return nullptr;
        if (!s) {
            std::unique_ptr<scratch_set> made(new scratch_set());
            made->stream = stream;
            made->thread = thread;
            if (!(made->words = alloc(BAM_SCRATCH_WORDS_BYTES))) return nullptr;
            sets.push_back(std::move(made));
            s = sets.back().get();
        }
        return grown(s->notes, s->notes_bytes, notes_bytes, alloc_notes) && grown(s->wanted, s->wanted_bytes, wanted_bytes, alloc) &&
               grown(s->tiles, s->tiles_bytes, tiles_bytes, alloc) ? s : nullptr;
    }

private:
    template <typename Alloc>
    bool grown(std::shared_ptr<void>& buf, size_t& have, size_t bytes, Alloc& alloc)
    {
        if (bytes <= have) return true;
        size_t size = bytes < 2 * have ? 2 * have : bytes;
        std::shared_ptr<void> larger = alloc(size);
        if (!larger && size > bytes) larger = alloc(size = bytes);
        if (!larger) return false;
        if (buf) replaced.push_back(buf);
        buf = larger;
        have = size;
        return true;
    }
};
#endif /* __BAM_SCRATCH_SETS_H__ */
