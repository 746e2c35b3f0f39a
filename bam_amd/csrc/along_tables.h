// The tables of a graph's plan that a reading of the edge array along its pages cannot do without, and the bits that one of the
// levels can.  Host side only, no HIP in here: the memory comes from the caller's allocator (tests/native/test_scratch.cpp hands
// in one of its own).
#ifndef __BAM_ALONG_TABLES_H__
#define __BAM_ALONG_TABLES_H__
#include <cstddef>
#include <memory>

struct along_tables {
    std::shared_ptr<void> tables, bits;      /* each made when first asked for; NULL: not yet, or refused */
    /*
     * False where the memory for the tables is refused: the call then reads the edges in a way that needs none.  Where it is
     * refused for the bits (0 bytes: none wanted) the levels are read without.  A later call asks again.  alloc(bytes) gives memory
     * or NULL.
     */
    template <typename Alloc>
    bool get(size_t table_bytes, size_t bit_bytes, Alloc&& alloc)
    {
        if (!tables) tables = alloc(table_bytes);
        if (tables && !bits && bit_bytes) bits = alloc(bit_bytes);
        return tables != nullptr;
    }
};
#endif /* __BAM_ALONG_TABLES_H__ */
