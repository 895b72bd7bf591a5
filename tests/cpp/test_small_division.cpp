// CPU test of the division by a launch constant that the few-row product stages its activations with: exact wherever the number times
// the divisor stays below 2^32, the last number of that range included.  Built with g++ (no GPU needed).
#include <cstdio>

#include "../../tscale_amd/csrc/wg_map.h"

using namespace tsattn;

int main()
{
    for (uint32_t d = 2; d <= 70000; d = d < 2100 ? d + 1 : d * 9 / 8) {
        const WgDiv by = wg_make_div(d);
        const uint32_t top = 0xffffffffu / d; // the largest x with x * d < 2^32
        for (uint32_t q = 0;; q = q < 40 ? q + 1 : q * 3 / 2) { // around multiples of the divisor
            const uint64_t at = (uint64_t)q * d;
            if (at > top) break;
            for (int64_t x = (int64_t)at - 1; x <= (int64_t)at + 1; ++x)
                if (x >= 0 && x <= (int64_t)top && wg_div_small((uint32_t)x, by) != (uint32_t)x / d) {
                    printf("FAIL %lld / %u\n", (long long)x, d);
                    return 1;
                }
        }
        if (wg_div_small(top, by) != top / d) {
            printf("FAIL %u / %u\n", top, d);
            return 1;
        }
    }
    printf("OK\n");
    return 0;
}
