// tile_order.hpp -- tickets of the grid sweeps' tiles (plain C++: tested on the host).
#pragma once

namespace hala_amd {

// Place of tile (tj, tk) of ntj x ntk in the order by diagonals tj + tk, by tk inside one: a tile's
// neighbours (tj - 1, tk) and (tj, tk - 1) come before it.
constexpr int tile_ticket(int tj, int tk, int ntj, int ntk) {
    const int d = tj + tk, a = ntj < ntk ? ntj : ntk, b = ntj < ntk ? ntk : ntj, left = ntj + ntk - 1 - d;
    const int before = d <= a   ? d * (d + 1) / 2
                       : d <= b ? a * (a + 1) / 2 + (d - a) * a
                                : ntj * ntk - left * (left + 1) / 2;
    return before + tk - (d < ntj ? 0 : d - ntj + 1);
}

}  // namespace hala_amd
