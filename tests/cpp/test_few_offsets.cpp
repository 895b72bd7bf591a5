// CPU test of the bound on the normalising few-row products: whatever it lets through is reached with 32-bit byte offsets, and the
// widest layer that is served (2^20 values, a feed-forward block of 2^21, 16 rows) is let through.  Built with g++ (no GPU needed).
#include <cstdio>

#include "../../tscale_amd/csrc/few_offsets.h"

using tsattn::few_offsets_fit;

int main()
{
    bool ok = few_offsets_fit(16, (int64_t)1 << 21, (int64_t)1 << 20) && few_offsets_fit(1, 768, 768) && !few_offsets_fit(16, 128, (int64_t)1 << 40);
    for (int64_t rows = 1; rows <= 16; ++rows)
        for (int64_t pitch = 128; pitch < ((int64_t)1 << 33); pitch = pitch * 5 / 4 + 1) {
            const bool reached = (rows * pitch - 1) * 4 <= (int64_t)0xffffffff; // the last value of the last row
            if ((few_offsets_fit(rows, pitch, 128) && !reached) || (few_offsets_fit(rows, 128, pitch) && !reached)) ok = false;
        }
    printf(ok ? "OK\n" : "FAIL\n");
    return ok ? 0 : 1;
}
