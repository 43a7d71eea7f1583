// Gathers and tile loops at the largest sizes the entry points accept
// (hala_amd/csrc/gather.hpp); prints one line per check, exits 1 on a failure.
#include <climits>
#include <cstdio>
#include <initializer_list>

#include "../../hala_amd/csrc/gather.hpp"

using namespace hala_amd;

static int failures = 0;
static void check(bool ok, const char *what) {
    std::printf("%s %s\n", ok ? "ok" : "FAIL", what);
    failures += !ok;
}

// the last element's offset by the rule's choice of type, against 64-bit arithmetic
static bool reaches(int64_t n, int64_t step) {
    const int c = (int)(n - 1);
    const uint64_t want = (uint64_t)c * (uint64_t)step;
    const uint64_t got = gather_wide(n, step) ? gather_offset<uint64_t>(c, (uint64_t)step)
                                              : gather_offset<uint32_t>(c, (uint32_t)step);
    return got == want;
}

// a tile loop visits every entry of [begin, end) once and ends
static bool covers(int begin, int end, int tile) {
    int64_t seen = 0;
    int at = begin;
    for (int base = begin; base < end; base = tile_next(base, end, tile)) {
        if (base != at) return false;
        const int cnt = end - base < tile ? end - base : tile;
        seen += cnt;
        at = base + cnt;
        if (seen > (int64_t)end - begin) return false;
    }
    return seen == (int64_t)end - begin && at == end;
}

int main() {
    const int64_t lim = int64_t(1) << 29;  // 2^29 doubles are 2^32 bytes
    for (int64_t step : {4, 8, 16})
        for (int64_t d = -2; d <= 2; d++) check(reaches((int64_t(1) << 32) / step + d, step), "offset around 4 GiB");
    check(!gather_wide(lim - 1, 8) && gather_wide(lim + 1, 8), "doubles need 64-bit offsets past 2^29");
    check(reaches(INT_MAX, 8) && reaches(INT_MAX, 16) && reaches(1, 8), "extremes");
    check(reaches(1000, int64_t(8) * 3000000), "a row of a wide dense matrix");
    for (int tile : {64, 1024, 2048, 4096})
        for (int end : {0, 1, tile - 1, tile, tile + 1, 3 * tile + 5, INT_MAX - 1, INT_MAX})
            for (int len : {0, 1, tile - 1, tile, tile + 1, 5 * tile - 3})
                if (len <= end) check(covers(end - len, end, tile), "tile loop");
    check(walk_rows(257 * 2048, 256, 9, 2048, 256, 1) && !walk_rows(257 * 2048, 257, 9, 2048, 256, 1) &&
              walk_rows(513 * 1024, 512, 9, 1024, 256, 2) && !walk_rows(100 * 2048, 100, 9, 2048, 256, 1) &&
              walk_rows(100, 1000, 513, 2048, 256, 1) && walk_rows(INT_MAX, 200, 0, 2048, 256, 1) &&
              walk_per_cu(16, false, 8) == 2 && walk_per_cu(16, true, 2) == 2 && walk_per_cu(16, true, 3) == 1 &&
              walk_per_cu(8, false, 1) == 1,
          "walked rows");
    check(gather_group(1) == 8 && gather_group(1 << 19) == 8 && gather_group((1 << 19) + 1) == 4 &&
              gather_group((1 << 20) + 1) == 2 && gather_group((1 << 21) + 1) == 1 &&
              gather_group(int64_t(INT_MAX) * 16) == 1,
          "vectors at once");
    return failures ? 1 : 0;
}
