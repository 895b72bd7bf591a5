// CPU test of the request walk of the streamed product (tscale_amd/csrc/stream_walk.h) with the kernel's shares of a matrix: every
// stage of every block is asked for exactly once, in order; every request, those past a wave's share included, stays inside
// its descriptor and the matrix.  Built with g++ (no GPU needed).
#include <cstdio>
#include <vector>

#include "../../tscale_amd/csrc/stream_walk.h"

using namespace tsattn;

static bool check(int n, int k, int pitch, int groups)
{
    const int waves = 8, in_flight = 5, ns = (k + 127) / 128, blocks = (n + 15) / 16;
    std::vector<int> seen((size_t)blocks * ns, 0);
    for (int wg = 0; wg < groups; ++wg) {
        const int b0 = (int)((int64_t)wg * blocks / groups), b1 = (int)(((int64_t)wg + 1) * blocks / groups), total = (b1 - b0) * ns;
        for (int w = 0; w < waves; ++w) {
            const int t0 = (int)((int64_t)w * total / waves), t1 = (int)(((int64_t)w + 1) * total / waves);
            StreamWalk walk = stream_walk(b0, t0, t1, ns);
            for (int i = t0; i < t1 + in_flight; ++i) { // in_flight stages ahead of the last multiplication
                const StreamStage s = stream_next(walk, n, k, pitch);
                const bool real = i < t1;
                const int rows = n - s.block * 16 < 16 ? n - s.block * 16 : 16;
                if (s.block < 0 || s.block >= blocks || s.scalar_off < 0 || s.scalar_off > s.size || (real ? s.size != (rows - 1) * pitch + k : s.size != 0)) {
                    printf("FAIL n %d k %d pitch %d, workgroup %d of %d, wave %d, stage %d of %d..%d: block %d, size %d, offset %d\n", n, k, pitch, wg, groups, w, i, t0,
                           t1, s.block, s.size, s.scalar_off);
                    return false;
                }
                if (real && (s.block * ns + s.scalar_off / 128 != b0 * ns + i || seen[(size_t)s.block * ns + s.scalar_off / 128]++)) {
                    printf("FAIL n %d k %d: stage %d is not the next\n", n, k, i);
                    return false;
                }
            }
        }
    }
    for (int x : seen)
        if (x != 1) { printf("FAIL n %d k %d: a stage is missing\n", n, k); return false; }
    return true;
}

int main()
{
    for (int n : {1, 15, 16, 17, 500, 4095, 4096, 4111, 50257})
        for (int k : {64, 128, 192, 512, 2048, 4160})
            for (int groups : {1, 7, 256})
                if (!check(n, k, k, groups) || !check(n, k, k + 16, groups)) return 1;
    printf("OK\n");
    return 0;
}
