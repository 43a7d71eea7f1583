// Gathers at the largest sizes the entry points accept
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

int main() {
    const int64_t lim = int64_t(1) << 29;  // 2^29 doubles are 2^32 bytes
    for (int64_t step : {4, 8, 16})
        for (int64_t d = -2; d <= 2; d++) check(reaches((int64_t(1) << 32) / step + d, step), "offset around 4 GiB");
    check(!gather_wide(lim - 1, 8) && gather_wide(lim + 1, 8), "doubles need 64-bit offsets past 2^29");
    check(reaches(INT_MAX, 8) && reaches(INT_MAX, 16) && reaches(1, 8), "extremes");
    check(reaches(1000, int64_t(8) * 3000000), "a row of a wide dense matrix");
    return failures ? 1 : 0;
}
