// Stable radix sort of (key, 32-bit position) pairs and the scans it needs
// (sort.hip).
#pragma once

#include "alto_internal.hpp"

namespace alto {

// 128-bit key, least significant word first
struct alignas(16) Key128 {
    uint64_t lo, hi;
};

// Work buffers of sort_pairs, reused from sort to sort on one stream.  Like
// every DevBuf they must outlive the work that uses them.  A sort may leave its
// buffers swapped: sorts of several key types over one space need keys and
// sp.keys both sized for the widest before the first.
struct SortSpace {
    DevBuf keys, pay;   // the alternate halves of the double buffers
    DevBuf hist, total;
};

// sizes the (unused) work buffers for up to n pairs with keys of key_bytes, so
// that the sorts allocate nothing
int reserve_sort(uint64_t n, size_t key_bytes, SortSpace& sp);

// Sorts n pairs by the low `bits` bits of the keys, stably and
// asynchronously on s.  keys / pay (refused where they are too small for n) are
// double-buffered with sp.keys / sp.pay: on return `keys` and `pay` hold the result (the buffers may have
// been swapped).  identity: pay is not read, the position of key i is i.
template <typename K>
int sort_pairs(DevBuf& keys, DevBuf& pay, bool identity, uint64_t n, int bits, SortSpace& sp, hipStream_t s);

// exclusive scan of each of `rows` rows of m counts in place; total[r] = sum
// of row r
int scan_rows(uint32_t* a, uint64_t rows, uint64_t m, uint32_t* total, hipStream_t s);

}  // namespace alto
