// CPU test of a decode launch's form: a range that the waves cover in one step of two rows per lane group takes such steps whatever the
// stride of the cache's tokens, and what exists with four waves only is never given sixteen.  Built with g++ (no GPU needed).
#include <cstdio>

#include "../../tscale_amd/csrc/decode_splits.h"

using namespace tsattn;

int main()
{
    bool ok = true;
    const auto want = [&](bool right, const char *what, int d, int64_t rows) {
        if (!right) { printf("FAIL %s: width %d, %ld rows\n", what, d, (long)rows); ok = false; }
    };
    for (int d = 64; d <= 128; d += 64)
        for (int far = 0; far < 2; ++far)
            for (int dump = 0; dump < 2; ++dump) {
                const bool general = decode_general(far ? (int64_t)1 << 24 : ((int64_t)1 << 24) - 16, dump);
                want(general == (far || dump), "general", d, 0);
                const int group = 64 / (d / 16); // rows of a wave's load
                for (int64_t rows = 0; rows < 6000; ++rows)
                    for (int64_t groups = 1; groups < 2000; groups = groups * 4 + 1) {
                        const DecodeForm f = decode_form(rows, d, groups, general);
                        want(f.general == general, "general kernel", d, rows);
                        want(f.waves == DEC_WAVES || (f.waves == DEC_WIDE_WAVES && !f.general && groups <= 256), "waves", d, rows);
                        want((f.rows == DEC_SHORT) == (rows <= f.waves * DEC_SHORT * group), "short steps", d, rows);
                        want(f.rows == DEC_SHORT || f.rows == (f.waves == DEC_WAVES ? DEC_LONG : DEC_WIDE_LONG), "long steps", d, rows);
                        if (rows <= 64) want(f.waves == DEC_WAVES && f.rows == DEC_SHORT, "a window of 64", d, rows);
                    }
            }
    // what tests/test_gpu_decode_wide.py and tests/test_gpu_token_step.py are about takes the forms they name
    const struct { int pairs, head_dim, rows, splits, per_group; } SIXTEEN[] = { // splits 0: chosen
        {12, 64, 513, 1, DEC_WIDE_LONG}, {12, 64, 1023, 1, DEC_WIDE_LONG}, {12, 64, 1025, 2, DEC_WIDE_LONG},
        {12, 64, 2100, 2, DEC_WIDE_LONG}, {12, 128, 257, 1, DEC_WIDE_LONG}, {12, 128, 511, 1, DEC_WIDE_LONG},
        {12, 128, 513, 2, DEC_WIDE_LONG}, {12, 128, 1100, 2, DEC_WIDE_LONG}, {12, 64, 129, 1, DEC_SHORT},
        {12, 64, 256, 1, DEC_SHORT}, {12, 128, 65, 1, DEC_SHORT}, {12, 128, 128, 1, DEC_SHORT},
        {6, 64, 200, 0, DEC_SHORT}, {6, 128, 100, 0, DEC_SHORT}, {6, 64, 700, 0, DEC_WIDE_LONG},
        {6, 128, 400, 0, DEC_WIDE_LONG}, {156, 64, 1025, 0, DEC_WIDE_LONG}, {6, 64, 4500, 0, DEC_WIDE_LONG},
        {6, 128, 2300, 0, DEC_WIDE_LONG}};
    int several = 0;
    for (const auto &l : SIXTEEN) {
        const int s = l.splits ? l.splits : decode_choose_splits(l.rows, l.head_dim, l.pairs, 32);
        const DecodeForm f = decode_form((l.rows + s - 1) / s, l.head_dim, (int64_t)l.pairs * s, false);
        want(f.waves == DEC_WIDE_WAVES && f.rows == l.per_group, "sixteen waves", l.head_dim, l.rows);
        several += l.splits == 0 && s > 1;
    }
    want(several == 2, "several splits", 0, several);
    if (ok) printf("OK\n");
    return ok ? 0 : 1;
}
