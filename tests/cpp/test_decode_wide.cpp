// CPU test of the choice between four and sixteen waves per workgroup of a decode launch.  The times are microseconds of launches in a
// replayed graph (MI355X, int8 cache, bf16 queries) with four and with sixteen; the rule has to choose one that is at most 7 % slower
// than the other (3 % is the worst of these lines, all launches on one cache), and four from one workgroup more than there are compute units.  Built
// with g++ (no GPU needed).
#include <cstdio>

#include "../../tscale_amd/csrc/decode_splits.h"

using namespace tsattn;

static const struct {
    int pairs, splits, head_dim, rows;
    double four, sixteen;
} LINES[] = {
    {12, 1, 64, 300, 4.47, 4.85},
    {12, 1, 64, 701, 5.87, 5.51},
    {12, 1, 64, 1500, 7.09, 7.28},
    {12, 1, 64, 2500, 9.74, 9.18},
    {12, 1, 64, 4096, 13.62, 12.62},
    {12, 4, 64, 2500, 8.79, 8.46},
    {16, 1, 128, 300, 6.09, 5.48},
    {16, 1, 128, 701, 7.20, 7.23},
    {16, 1, 128, 1500, 11.13, 10.87},
    {16, 1, 128, 4096, 24.55, 22.65},
    {16, 4, 128, 4096, 14.07, 12.84},
    {64, 1, 64, 701, 6.08, 5.81},
    {64, 2, 64, 4096, 14.18, 12.77},
    {64, 1, 128, 300, 6.29, 5.62},
    {64, 4, 128, 2500, 13.06, 11.99},
    {64, 4, 128, 4096, 17.14, 15.61},
    {96, 2, 64, 2500, 11.87, 10.56},
    {96, 1, 64, 4096, 18.11, 16.33},
    {128, 2, 128, 2500, 18.75, 18.14},
    {128, 1, 128, 4096, 33.56, 28.76},
    {156, 1, 64, 1500, 8.69, 8.67},
    {156, 1, 64, 4096, 19.65, 17.45},
    {156, 1, 128, 1500, 15.51, 13.94},
    {156, 2, 128, 1500, 16.63, 18.75},
    {256, 1, 64, 701, 6.72, 6.33},
    {256, 1, 64, 4096, 23.57, 22.52},
    {256, 1, 128, 2500, 28.23, 27.55},
    {288, 1, 64, 300, 5.60, 8.34},
    {288, 1, 64, 1500, 12.88, 15.69},
    {512, 1, 64, 701, 9.74, 11.33},
    {512, 1, 128, 1500, 31.58, 33.49},
};

int main()
{
    bool ok = true;
    for (const auto &l : LINES) {
        const bool wide = decode_wide((l.rows + l.splits - 1) / l.splits, l.head_dim, (int64_t)l.pairs * l.splits);
        const double got = wide ? l.sixteen : l.four, best = l.four < l.sixteen ? l.four : l.sixteen;
        if (got > 1.07 * best) {
            printf("FAIL %d pairs of width %d, %d rows in %d splits: %s waves, %.2f us, best %.2f\n", l.pairs, l.head_dim, l.rows, l.splits, wide ? "sixteen" : "four", got, best);
            ok = false;
        }
    }
    for (int d = 64; d <= 128; d += 64)
        for (int64_t rows = 1; rows < ((int64_t)1 << 31); rows = rows * 5 / 3 + 1)
            for (int64_t groups = 257; groups < 100000; groups *= 3) ok = ok && !decode_wide(rows, d, groups);
    if (ok) printf("OK\n");
    return ok ? 0 : 1;
}
