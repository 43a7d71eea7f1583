// Every tile's ticket (hala_amd/csrc/tile_order.hpp) against a stable sort by diagonals; exits 1 on a failure.
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <vector>

#include "../../hala_amd/csrc/tile_order.hpp"

int main() {
    std::vector<int> sizes(24);
    std::iota(sizes.begin(), sizes.end(), 1);
    for (int big : {100, 1563, 2499}) sizes.push_back(big);
    for (int ntj : sizes)
        for (int ntk : sizes) {
            if ((long)ntj * ntk > 300000) continue;
            std::vector<int> order(ntj * ntk);
            std::iota(order.begin(), order.end(), 0);
            std::stable_sort(order.begin(), order.end(),
                             [&](int x, int y) { return x % ntj + x / ntj < y % ntj + y / ntj; });
            for (int k = 0; k < ntj * ntk; k++)
                if (hala_amd::tile_ticket(order[k] % ntj, order[k] / ntj, ntj, ntk) != k) {
                    std::printf("%d x %d: ticket %d\n", ntj, ntk, k);
                    return 1;
                }
        }
    return 0;
}
