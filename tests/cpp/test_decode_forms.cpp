// CPU test of the choice between four and sixteen waves per workgroup of a decode launch, by what the launch has to do.  Two lines drawn
// from every range of rows per workgroup (a quarter to a half of a step of the four waves, up to 0.54, 3/4, 1, 1 1/2, 2, 3 steps and
// more), up to 256 workgroups.  The times are microseconds of launches in a replayed graph (MI355X), each on a cache of its own, for int8
// and e4m3 caches under bf16 queries, and of a whole layer's launches for the form with the front.  A launch alone may be at most 0.1 us
// slower than with the other form; the layers' times, in which four other launches vary along, 0.1 us on average.  Built with g++.
#include <cstdio>

#include "../../tscale_amd/csrc/decode_splits.h"

using namespace tsattn;

enum Kind { I8, E4M3, FRONT };

static const struct {
    Kind kind;
    int pairs, splits, head_dim, rows;
    double four, sixteen;
} LINES[] = {
    {I8, 16, 1, 64, 200, 4.61, 4.61},
    {I8, 64, 2, 64, 400, 7.14, 7.15},
    {I8, 16, 1, 64, 260, 4.63, 4.89},
    {I8, 16, 12, 64, 3100, 10.85, 11.15},
    {I8, 64, 1, 64, 300, 4.86, 5.08},
    {I8, 192, 1, 64, 300, 5.24, 5.51},
    {I8, 8, 6, 64, 2875, 8.37, 9.38},
    {I8, 156, 1, 64, 400, 5.32, 6.39},
    {I8, 8, 1, 64, 701, 6.56, 5.70},
    {I8, 96, 1, 64, 701, 7.04, 6.25},
    {I8, 16, 2, 64, 2048, 9.21, 9.09},
    {I8, 48, 1, 64, 900, 7.10, 7.07},
    {I8, 16, 2, 64, 2500, 10.81, 9.58},
    {I8, 16, 1, 64, 1300, 8.71, 7.87},
    {I8, 128, 2, 64, 3100, 16.74, 14.91},
    {I8, 192, 1, 64, 2500, 15.60, 14.35},
    {I8, 96, 2, 128, 160, 7.17, 7.27},
    {I8, 48, 3, 128, 260, 7.54, 7.63},
    {I8, 32, 1, 128, 130, 4.76, 5.03},
    {I8, 64, 3, 128, 400, 8.00, 8.25},
    {I8, 12, 6, 128, 900, 8.30, 8.53},
    {I8, 16, 3, 128, 560, 7.67, 7.88},
    {I8, 12, 6, 128, 1300, 8.83, 9.86},
    {I8, 64, 3, 128, 701, 8.55, 9.49},
    {I8, 24, 8, 128, 2875, 11.48, 10.81},
    {I8, 8, 1, 128, 300, 6.37, 5.59},
    {I8, 8, 6, 128, 2875, 10.40, 10.42},
    {I8, 12, 8, 128, 3100, 11.12, 11.21},
    {I8, 8, 4, 128, 2500, 11.25, 9.99},
    {I8, 32, 2, 128, 1300, 11.18, 10.39},
    {I8, 8, 3, 128, 2500, 12.92, 10.82},
    {I8, 32, 1, 128, 2048, 18.72, 15.69},
    {E4M3, 24, 6, 64, 1500, 8.86, 8.68},
    {E4M3, 48, 1, 64, 200, 4.98, 4.83},
    {E4M3, 16, 12, 64, 3100, 10.74, 10.87},
    {E4M3, 12, 12, 64, 3100, 10.54, 10.75},
    {E4M3, 156, 1, 64, 300, 5.30, 5.52},
    {E4M3, 32, 1, 64, 300, 4.97, 5.34},
    {E4M3, 24, 6, 64, 2500, 9.16, 10.22},
    {E4M3, 128, 2, 64, 1024, 8.83, 9.44},
    {E4M3, 64, 3, 64, 2048, 10.54, 9.56},
    {E4M3, 32, 6, 64, 3100, 11.22, 10.26},
    {E4M3, 12, 4, 64, 3100, 10.14, 10.08},
    {E4M3, 32, 4, 64, 3100, 10.33, 10.26},
    {E4M3, 12, 3, 64, 3100, 11.76, 10.57},
    {E4M3, 8, 3, 64, 3100, 11.52, 10.43},
    {E4M3, 16, 2, 64, 4096, 13.71, 12.15},
    {E4M3, 240, 1, 64, 2500, 17.60, 16.62},
    {E4M3, 12, 12, 128, 1500, 10.86, 10.71},
    {E4M3, 16, 3, 128, 200, 7.97, 7.48},
    {E4M3, 192, 1, 128, 130, 5.34, 5.47},
    {E4M3, 64, 1, 128, 130, 5.03, 5.33},
    {E4M3, 16, 12, 128, 2048, 11.23, 11.17},
    {E4M3, 32, 2, 128, 300, 7.46, 7.74},
    {E4M3, 24, 8, 128, 2048, 10.11, 11.00},
    {E4M3, 240, 1, 128, 200, 6.03, 6.78},
    {E4M3, 24, 1, 128, 300, 6.94, 6.15},
    {E4M3, 48, 1, 128, 300, 7.06, 6.19},
    {E4M3, 24, 2, 128, 1024, 9.75, 9.74},
    {E4M3, 32, 8, 128, 4096, 13.88, 13.28},
    {E4M3, 64, 4, 128, 2500, 14.65, 13.29},
    {E4M3, 32, 3, 128, 2048, 12.42, 11.36},
    {E4M3, 64, 1, 128, 2048, 19.98, 16.48},
    {E4M3, 16, 3, 128, 2500, 14.07, 11.68},
    {FRONT, 12, 8, 64, 2048, 27.47, 27.21},
    {FRONT, 24, 8, 64, 2048, 27.99, 27.54},
    {FRONT, 8, 1, 64, 260, 22.62, 22.74},
    {FRONT, 16, 1, 64, 260, 23.15, 23.08},
    {FRONT, 24, 6, 64, 2112, 27.70, 27.43},
    {FRONT, 48, 2, 64, 560, 29.08, 29.16},
    {FRONT, 96, 2, 64, 800, 30.16, 30.67},
    {FRONT, 12, 1, 64, 512, 23.74, 23.73},
    {FRONT, 48, 3, 64, 2048, 31.99, 31.66},
    {FRONT, 256, 1, 64, 701, 35.66, 35.18},
    {FRONT, 24, 2, 64, 2048, 28.55, 28.43},
    {FRONT, 156, 1, 64, 1024, 35.34, 35.52},
    {FRONT, 256, 1, 64, 1100, 38.95, 37.56},
    {FRONT, 12, 1, 64, 1100, 27.03, 26.15},
    {FRONT, 156, 1, 64, 3100, 44.79, 42.24},
    {FRONT, 96, 2, 64, 4096, 40.00, 38.54},
    {FRONT, 16, 4, 128, 300, 32.30, 31.93},
    {FRONT, 128, 2, 128, 150, 37.13, 36.91},
    {FRONT, 16, 6, 128, 800, 32.90, 32.80},
    {FRONT, 128, 2, 128, 260, 37.64, 37.34},
    {FRONT, 8, 4, 128, 701, 27.06, 26.74},
    {FRONT, 8, 3, 128, 512, 26.52, 26.36},
    {FRONT, 128, 1, 128, 200, 35.64, 35.51},
    {FRONT, 8, 4, 128, 1024, 27.13, 26.94},
    {FRONT, 16, 4, 128, 1100, 34.21, 33.53},
    {FRONT, 48, 4, 128, 1500, 37.85, 37.65},
    {FRONT, 8, 3, 128, 1500, 28.72, 28.57},
    {FRONT, 32, 8, 128, 4096, 39.86, 40.11},
    {FRONT, 8, 6, 128, 4096, 31.33, 30.82},
    {FRONT, 8, 1, 128, 701, 27.55, 26.86},
    {FRONT, 32, 2, 128, 2048, 39.55, 38.46},
    {FRONT, 48, 1, 128, 2112, 47.33, 43.42},
};

int main()
{
    bool ok = true;
    double layers = 0.0;
    int n_layers = 0;
    for (const auto &l : LINES) {
        const bool wide = decode_wide((l.rows + l.splits - 1) / l.splits, l.head_dim, (int64_t)l.pairs * l.splits);
        const double lost = (wide ? l.sixteen : l.four) - (l.four < l.sixteen ? l.four : l.sixteen);
        if (l.kind == FRONT) { layers += lost; ++n_layers; }
        else if (lost > 0.1) {
            printf("FAIL kind %d, %d pairs of width %d, %d rows in %d splits: %s waves, %.2f and %.2f us\n", (int)l.kind, l.pairs, l.head_dim, l.rows, l.splits,
                   wide ? "sixteen" : "four", l.four, l.sixteen);
            ok = false;
        }
    }
    if (layers > 0.1 * n_layers) { printf("FAIL layers %.3f us lost on average\n", layers / n_layers); ok = false; }
    for (int d = 64; d <= 128; d += 64)
        for (int64_t rows = 1; rows < ((int64_t)1 << 31); rows = rows * 5 / 3 + 1) ok = ok && !decode_wide(rows, d, 257) && !decode_wide(rows, d, 1, true);
    if (ok) printf("OK\n");
    return ok ? 0 : 1;
}
