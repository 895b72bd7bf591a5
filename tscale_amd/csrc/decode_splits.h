// How many workgroups share a (sequence, head) pair's cache rows in a decode launch, and in which form they walk them.  Plain C++: no
// device code, so that the rules can be tested without a GPU.
#pragma once

#include <stdint.h>

namespace tsattn {

constexpr int DEC_WAVES = 4, DEC_WIDE_WAVES = 16; // waves per workgroup (wide: few workgroups, which then have a compute unit each)
constexpr int DEC_LONG = 8, DEC_SHORT = 2; // cache rows per lane group and step (short: ranges of one step of the waves)
constexpr int DEC_WIDE_LONG = 4;           // the same with sixteen waves

// cache rows that a workgroup of four waves takes per step of DEC_LONG: head_dim / 16 lanes per row
constexpr int decode_step_rows(int head_dim) { return DEC_WAVES * DEC_LONG * (64 / (head_dim / 16)); }

constexpr int DECODE_WIDE_GROUPS = 256; // compute units

// Whether a launch takes the general kernels, which exist with four waves: any stride of the cache's tokens (the others multiply it in 24 bits)
// and the dump of raw dot products.
constexpr int64_t DECODE_NEAR = 1 << 24;
constexpr bool decode_general(int64_t tok_stride, bool dump) { return dump || tok_stride >= DECODE_NEAR; }

// Whether a launch of `groups` workgroups with `rows` cache rows each takes sixteen waves per workgroup (decode_wide_kernel)
// instead of four.  Where a workgroup has a compute unit to itself, four waves are one per SIMD, which issues an instruction every
// 7.6 cycles where two and more get one in every 3.8, and have a quarter of the requests on their way; sixteen cost 0.3 to 0.4 us
// more to start and to merge.  The step of the four decides: below it sixteen only shorten a wave's share of it, from one row on past
// it the four begin another.  Microseconds by which sixteen are faster (a minus: slower), averages of launches of 8 to 256 workgroups in
// one to twelve splits in a replayed graph, by rows per workgroup in steps of the four, each launch on a cache of its own / all on one:
//                   1/4 - 1/2      1/2 - 3/4       3/4 - 1      1 - 1 1/2    1 1/2 - 2      2 - 3        more
//   int8          -0.01 / -0.16   -0.22 / -0.47   -1.0 / -1.1   0.8 / 0.5   0.04 / -0.1   0.9 / 0.3    2.5 / 1.6
//   e4m3           0.15 / -0.02   -0.24 / -0.68   -1.0 / -1.2   0.9 / 0.4   0.12 / 0.0    1.1 / 0.4    3.0 / 2.4
//   with a front   0.31            0.22            0.03         0.7        -0.04          0.7          2.6
// (up to a quarter of a step the four take short steps and are 0.4 us faster throughout).  A cache of its own is what a model's layer has; one
// cache for all launches stays in the L2s.  With sixteen waves the other fifteen ask for their rows while the first makes the front, so
// that a front gains at shorter ranges, too; the rule is one for all, so that an append in the launch, one before it and a layer's one
// call add up in the same order.  With more workgroups than compute units the four are the better share: 288 of width 64, 1500 rows 12.9
// and 15.7 us; 96 pairs of 1024 rows in three splits 9.5 and 11.9.
inline bool decode_wide(int64_t rows, int head_dim, int64_t groups, bool general = false)
{
    const int step = decode_step_rows(head_dim);
    return !general && groups <= DECODE_WIDE_GROUPS && (rows > step || (rows > step / 4 && rows <= step / 2));
}

// The form of a launch of `groups` workgroups with `rows` cache rows each.  A range that the waves cover in one step of two rows per lane
// group (a 64-key window) is shared out in such steps, whatever the stride: with steps of eight the first wave alone would compute
// all of it (window 64, width 128: 1.8 us of its instructions).
struct DecodeForm {
    int waves, rows; // per workgroup; per lane group and step
    bool general;
};

inline DecodeForm decode_form(int64_t rows, int head_dim, int64_t groups, bool general)
{
    const bool wide = decode_wide(rows, head_dim, groups, general);
    const int waves = wide ? DEC_WIDE_WAVES : DEC_WAVES;
    const bool one = rows <= waves * DEC_SHORT * (64 / (head_dim / 16));
    return {waves, one ? DEC_SHORT : wide ? DEC_WIDE_LONG : DEC_LONG, general};
}

constexpr double DECODE_START_NS = 3550.0, DECODE_MERGE_NS = 2000.0, DECODE_SPLIT_NS = 305.0;

// Nanoseconds of a decode launch with `splits` workgroups per pair, by a fit of the present kernels in both forms to some 6000 launches of 8
// to 768 pairs, 64 to 4096 rows, in 1 to 16 splits, int8 and e4m3, each on a cache of its own in a replayed graph (and of 144 on one):
//   four waves walk a workgroup's rows at 45 bytes per nanosecond in steps, of which the last is at least 0.53 of a whole one;
//   sixteen walk them at 47.5 in halves of such a step (four of the waves);
//   several workgroups on a compute unit walk all their rows at 41 at most;
//   no launch is faster than memory delivers the rows, 8000 bytes per nanosecond;
//   more than one split costs the merge launch, 2.0 us, 0.3 us per split and 1.7 ns per workgroup, and 0.15 us more where the number is no
//   power of two.
inline double decode_time(int64_t rows, int head_dim, int64_t pairs, int splits, bool general)
{
    const int step = decode_step_rows(head_dim), row_bytes = 2 * head_dim + 8;
    const int64_t per = (rows + splits - 1) / splits, groups = pairs * splits, shared = (groups + DECODE_WIDE_GROUPS - 1) / DECODE_WIDE_GROUPS;
    double ns;
    if (4 * per <= step) {
        ns = DECODE_START_NS;
    } else if (decode_wide(per, head_dim, groups, general)) {
        const int half = step / 2;
        ns = 3780.0 + (double)((per + half - 1) / half * half) * row_bytes / 47.5;
    } else {
        const int64_t last = per % step;
        const double least = 0.53 * step;
        ns = DECODE_START_NS + ((double)(per - last) + (last == 0 ? 0.0 : last > least ? (double)last : least)) * row_bytes / 45.0;
    }
    const double memory = 2400.0 + (double)rows * row_bytes * (double)pairs / 8000.0;
    if (ns < memory) ns = memory;
    if (shared > 1) {
        const double all = DECODE_START_NS + (double)(per * shared) * row_bytes / 41.0;
        if (ns < all) ns = all;
    }
    return splits > 1 ? ns + DECODE_MERGE_NS + DECODE_SPLIT_NS * splits + 1.7 * (double)groups + ((splits & (splits - 1)) == 0 ? 0.0 : 150.0) : ns;
}

// The number of splits (1, 2, 3, 4, 6, 8, 12 and so on; at most max_splits, and at most 1024 workgroups) with the least such time.  Together
// with the form that decode_wide gives it it is 0.2 % off the best of both forms and all numbers on average, 6.5 % at worst (on one cache
// 0.6 % and 8 %).  Chosen by a fit of the four waves alone and the form after it, it was 0.8 and 13 %: 64 pairs of width 64, 1500 rows on one cache in 3
// splits and two launches 8.2 us where one launch of sixteen waves takes 7.4 to 7.9; 156 pairs of width 128, 2500 rows in 3 splits 23.6, in one
// launch of sixteen 21.4.
inline int decode_choose_splits(int64_t rows, int head_dim, int64_t pairs, int max_splits, bool general = false)
{
    int best = 1;
    double best_ns = decode_time(rows, head_dim, pairs, 1, general);
    for (int s = 1; (rows + s - 1) / s * 4 > decode_step_rows(head_dim);) { // (more splits shorten no workgroup's walk)
        s = s == 1 ? 2 : (s & (s - 1)) == 0 ? s + s / 2 : s / 3 * 4;
        if (s > max_splits || s * pairs > 1024 || DECODE_START_NS + DECODE_MERGE_NS + DECODE_SPLIT_NS * s >= best_ns) break; // (nor can more be less)
        const double ns = decode_time(rows, head_dim, pairs, s, general);
        if (ns < best_ns) { best_ns = ns; best = s; }
    }
    return best;
}

} // namespace tsattn
