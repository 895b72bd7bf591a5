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
            for (int dump = 0; dump < 2; ++dump)
                for (int e4m3 = 0; e4m3 < 2; ++e4m3)
                    for (int append = 0; append < 2; ++append) {
                        const DecodeKind kind = decode_kind(e4m3, append, far ? (int64_t)1 << 24 : ((int64_t)1 << 24) - 16, dump);
                        want((kind == DECODE_GENERAL) == (far || dump), "general", d, 0);
                        const int group = 64 / (d / 16); // rows of a wave's load
                        for (int64_t rows = 0; rows < 6000; ++rows)
                            for (int64_t groups = 1; groups < 2000; groups = groups * 4 + 1) {
                                const DecodeForm f = decode_form(rows, d, groups, kind);
                                want(f.general == (kind == DECODE_GENERAL), "general kernel", d, rows);
                                want(f.waves == DEC_WAVES || (f.waves == DEC_WIDE_WAVES && !f.general && groups <= 256), "waves", d, rows);
                                want((f.rows == DEC_SHORT) == (rows <= f.waves * DEC_SHORT * group), "short steps", d, rows);
                                want(f.rows == DEC_SHORT || f.rows == (f.waves == DEC_WAVES ? DEC_LONG : DEC_WIDE_LONG), "long steps", d, rows);
                                if (rows <= 64) want(f.waves == DEC_WAVES && f.rows == DEC_SHORT, "a window of 64", d, rows);
                            }
                    }
    // what tests/test_gpu_decode_wide.py and tests/test_gpu_token_step.py are about takes the forms they name
    const struct { DecodeKind kind; int pairs, head_dim, rows, splits, per_group; } SIXTEEN[] = { // splits 0: chosen
        {DECODE_I8, 12, 64, 513, 1, DEC_WIDE_LONG}, {DECODE_I8, 12, 64, 1023, 1, DEC_WIDE_LONG}, {DECODE_E4M3, 12, 64, 1025, 2, DEC_WIDE_LONG},
        {DECODE_E4M3, 12, 64, 2100, 2, DEC_WIDE_LONG}, {DECODE_I8, 12, 128, 257, 1, DEC_WIDE_LONG}, {DECODE_E4M3, 12, 128, 511, 1, DEC_WIDE_LONG},
        {DECODE_I8, 12, 128, 513, 2, DEC_WIDE_LONG}, {DECODE_I8, 12, 128, 1100, 2, DEC_WIDE_LONG}, {DECODE_E4M3, 12, 64, 129, 1, DEC_SHORT},
        {DECODE_E4M3, 12, 64, 256, 1, DEC_SHORT}, {DECODE_E4M3, 12, 128, 65, 1, DEC_SHORT}, {DECODE_E4M3, 12, 128, 128, 1, DEC_SHORT},
        {DECODE_I8_APPEND, 6, 64, 200, 0, DEC_SHORT}, {DECODE_I8_APPEND, 6, 128, 100, 0, DEC_SHORT}, {DECODE_I8_APPEND, 6, 64, 700, 0, DEC_WIDE_LONG},
        {DECODE_I8_APPEND, 6, 128, 400, 0, DEC_WIDE_LONG}, {DECODE_I8_APPEND, 156, 64, 1025, 0, DEC_WIDE_LONG}, {DECODE_I8_APPEND, 6, 64, 4500, 0, DEC_WIDE_LONG},
        {DECODE_I8_APPEND, 6, 128, 2300, 0, DEC_WIDE_LONG}};
    int several = 0;
    for (const auto &l : SIXTEEN) {
        const int s = l.splits ? l.splits : decode_choose_splits(l.rows, l.head_dim, l.pairs, 32, l.kind);
        const DecodeForm f = decode_form((l.rows + s - 1) / s, l.head_dim, (int64_t)l.pairs * s, l.kind);
        want(f.waves == DEC_WIDE_WAVES && f.rows == l.per_group, "sixteen waves", l.head_dim, l.rows);
        several += l.splits == 0 && s > 1;
    }
    want(several == 2, "several splits", 0, several);
    if (ok) printf("OK\n");
    return ok ? 0 : 1;
}
