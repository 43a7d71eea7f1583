// gather.hpp -- integer arithmetic of the products' gathers and tile loops
// (plain C++: tested on the host at sizes no test matrix has).
#pragma once
#include <cstdint>

namespace hala_amd {

// Byte offset of element c of a vector whose elements lie step bytes apart.
template <class TO>
constexpr TO gather_offset(int c, TO step) {
    return (TO)c * step;
}

// Whether the offsets of an n-element vector need 64 bits.
constexpr bool gather_wide(int64_t n, int64_t step) { return n * step > (int64_t)UINT32_MAX; }

// Whether the threads of a product walk their rows in memory instead of in staged tiles.  A staged block
// keeps only the rows of the present tile at work: with more entries than a tile (`tile`) it waits for
// one tile after the other, which other workgroups of the CU hide if there are any.  So the rows are
// walked where the CUs hold at most per_cu of them (walk_per_cu), and where one row alone (max_row, 0: not
// known) takes a good part of a tile.  Walking many blocks per CU loses the lines that neighbouring rows
// share.  Staged -> walked (us), x vectors:
//   27-point complex FP64, 250 blocks x1 35 -> 11, 432 x1 41 -> 18, 1024 x1 44 -> 61; transposed 432 57 -> 43, 1024 78 -> 133
//   27-point FP64, 250 blocks x8 31 -> 20, 420 x8 34 -> 27, 762 x8 47 -> 54
//   30 random entries FP64 per row, 235 blocks x8 83 -> 70, 293 x8 117 -> 142
//   rows of 2 .. 3000 FP64, 391 blocks x2 325 -> 207
constexpr bool walk_rows(int64_t entries, int blocks, int max_row, int tile, int num_cus, int per_cu) {
    return (blocks <= num_cus * per_cu && entries > (int64_t)blocks * tile) || max_row > tile / 4;
}
// One, but two for 16-byte values, whose tiles are half as long; not for a transposed product of more than
// two vectors (313 blocks of 15 entries a row, x1 33 -> 28, x3 50 -> 58).
constexpr int walk_per_cu(int elem_bytes, bool trans, int ncols) {
    return elem_bytes >= 16 && (!trans || ncols <= 2) ? 2 : 1;
}

// Vectors of `bytes` each that a product takes at once (8, 4, 2 or 1) where neighbouring rows seldom gather
// neighbouring elements (hala_csr_s::spread: random and ragged patterns): as many as an XCD's 4 MiB of L2
// hold together, or every gather of a group goes out to the MALL.  Eight at once -> by this rule, 8 FP64
// vectors: 600 000 rows of 10 random entries 736 -> 441 us (one by one), 300 000 rows of a ragged
// mesh 271 -> 188 us (one by one), 200 000 rows of 8 random entries 134 -> 91 us (pairs).
constexpr int64_t GATHER_CACHE = int64_t(4) << 20;
constexpr int gather_group(int64_t bytes) {
    return bytes * 8 <= GATHER_CACHE ? 8 : bytes * 4 <= GATHER_CACHE ? 4 : bytes * 2 <= GATHER_CACHE ? 2 : 1;
}

// Where a loop over the entries [.., end) in tiles goes after base (never past
// end: entry counts reach INT_MAX - 1).
constexpr int tile_next(int base, int end, int tile) { return end - base > tile ? base + tile : end; }

}  // namespace hala_amd
