// CPU test of the K offsets that the wide int8 product requests: inside the rows for every step, those ahead of the last one
// included, and the step's own tile wherever there is one.  Built with g++ (no GPU needed).
#include <cstdio>

#include "../../tscale_amd/csrc/wg_map.h"

int main()
{
    const int tile = 64, ahead = 3;
    for (int k = tile; k <= 8192; k += tile)
        for (int step = 0; step < k / tile + ahead; ++step) {
            const int at = tsattn::wide_k_offset(step, tile, k);
            if (at < 0 || at + tile > k || (step < k / tile && at != step * tile)) {
                printf("FAIL k %d step %d: offset %d\n", k, step, at);
                return 1;
            }
        }
    printf("OK\n");
    return 0;
}
