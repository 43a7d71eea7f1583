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

// Where a loop over the entries [.., end) in tiles goes after base (never past
// end: entry counts reach INT_MAX - 1).
constexpr int tile_next(int base, int end, int tile) { return end - base > tile ? base + tile : end; }

}  // namespace hala_amd
