// CPU test of the number of splits a decode launch takes.  The times are microseconds of launches (MI355X, int8 cache, bf16
// queries) with the numbers of splits behind them; the rule has to choose one that is at most 7 % slower than the best of its line,
// and never more than the caller's scratch or the rule's own limit allows.  Built with g++ (no GPU needed).
#include <cstdio>

#include "../../tscale_amd/csrc/decode_splits.h"

using namespace tsattn;

static const int SPLITS[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16};
struct Line {
    int pairs, head_dim, rows;
    double us[10]; // 0: not measured
};
static const Line LINES[] = {
    {16, 128, 512, {7.37, 7.90, 8.06, 7.86, 8.22, 8.71, 8.69, 9.73, 9.81, 11.16}},
    {16, 128, 1500, {15.28, 12.26, 10.87, 10.33, 10.71, 9.85, 10.15, 10.99, 11.11, 12.54}},
    {16, 128, 3000, {25.11, 17.94, 14.80, 12.99, 13.02, 11.98, 12.03, 12.88, 11.99, 13.42}},
    {16, 128, 4096, {31.90, 21.65, 18.39, 14.98, 14.98, 13.79, 12.75, 13.48, 13.58, 14.04}},
    {32, 128, 2048, {19.32, 14.52, 13.09, 11.38, 11.64, 12.08, 11.47, 13.16, 13.12, 14.26}},
    {64, 128, 1024, {12.15, 10.96, 11.23, 10.14, 11.35, 11.60, 11.84, 13.01, 13.22, 14.78}},
    {64, 128, 4096, {32.48, 22.85, 20.49, 18.37, 21.06, 19.75, 19.10, 21.22, 20.58, 21.73}},
    {128, 128, 1500, {16.46, 15.15, 15.83, 15.33, 16.03, 15.62, 17.15, 19.36, 0, 0}},
    {128, 128, 4096, {33.85, 28.03, 30.04, 27.14, 29.42, 29.14, 29.27, 30.57, 0, 0}},
    {240, 128, 2048, {24.53, 25.59, 27.32, 26.67, 0, 0, 0, 0, 0, 0}},
    {12, 64, 701, {7.24, 7.80, 0, 0, 0, 0, 0, 0, 0, 0}},
    {12, 64, 2048, {11.71, 10.49, 10.64, 9.13, 9.39, 9.38, 9.65, 10.50, 11.07, 11.95}},
    {12, 64, 3000, {15.40, 12.41, 11.25, 10.57, 10.82, 9.81, 10.01, 10.75, 11.17, 12.49}},
    {12, 64, 4096, {18.90, 14.38, 12.95, 11.22, 11.23, 11.18, 10.26, 11.19, 11.62, 12.66}},
    {24, 64, 2048, {11.92, 10.56, 10.60, 9.24, 9.46, 9.96, 9.97, 10.96, 12.36, 12.95}},
    {96, 64, 1500, {10.57, 10.98, 11.67, 11.25, 11.40, 12.85, 12.71, 15.21, 0, 0}},
    {96, 64, 4096, {20.32, 16.43, 18.20, 16.28, 16.45, 19.39, 16.20, 18.57, 0, 0}},
    {180, 64, 4096, {21.81, 23.30, 25.44, 22.14, 23.92, 0, 0, 0, 0, 0}},
};

int main()
{
    bool ok = true;
    for (const Line &l : LINES) {
        double best = 1e9, got = 0.0;
        const int s = decode_choose_splits(l.rows, l.head_dim, l.pairs, 32);
        for (int i = 0; i < 10; ++i) {
            if (l.us[i] == 0.0) continue;
            if (l.us[i] < best) best = l.us[i];
            if (SPLITS[i] == s) got = l.us[i];
        }
        if (got == 0.0 || got > 1.07 * best) {
            printf("FAIL %d pairs of width %d, %d rows: %d splits, %.2f us, best %.2f\n", l.pairs, l.head_dim, l.rows, s, got, best);
            ok = false;
        }
    }
    for (int d = 64; d <= 128; d += 64)
        for (int64_t pairs = 1; pairs < 5000; pairs = pairs * 3 / 2 + 1)
            for (int64_t rows = 1; rows < ((int64_t)1 << 31); rows = rows * 5 / 3 + 1)
                for (int most = 1; most <= 40; most += 13) {
                    const int s = decode_choose_splits(rows, d, pairs, most);
                    if (s < 1 || s > most || (s > 1 && s * pairs > 1024)) { printf("FAIL %ld pairs, %ld rows: %d of %d splits\n", (long)pairs, (long)rows, s, most); return 1; }
                }
    if (ok) printf("OK\n");
    return ok ? 0 : 1;
}
