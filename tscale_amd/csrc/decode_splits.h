// How many workgroups share a (sequence, head) pair's cache rows in a decode launch.  Plain C++: no device code, so that the
// rule can be tested without a GPU.
#pragma once

#include <stdint.h>

namespace tsattn {

// cache rows that a workgroup of decode_split_kernel takes per step: four waves, eight rows per lane group, head_dim / 16 lanes
// per row
constexpr int decode_step_rows(int head_dim) { return 4 * 8 * (64 / (head_dim / 16)); }

// The number of splits (at most max_splits, and at most 1024 workgroups) with the least time, in nanoseconds, by a fit of
// launches of 8 to 768 pairs, 512 to 4096 rows and 1 to 16 splits:
//   a compute unit walks a workgroup's rows at 33 bytes per nanosecond in steps, of which the last is at least a third of a whole one;
//   of several workgroups it walks all the rows;
//   no launch is faster than memory delivers the rows, 6800 bytes per nanosecond;
//   more than one split costs the merge launch, 2.0 us, 0.28 us per split and 3 ns per workgroup, and 0.2 us more where the number is no
//   power of two (8 pairs of width 128 and 3100 rows: 12.6, 12.9, 11.8 us with 5, 6 and 8 splits).
// What it chooses is within 0.7 % of the best number on average and 11 % at worst.  (Times of the kernel before its merge by halving
// exchanges and 24-bit offsets; the present one walks at 54 to 66 bytes per nanosecond, a launch takes 1 to 2 us less, and the choice is 1.0 % off
// the best number on average.)  Without the steps (a workgroup's rows at 37 bytes
// per nanosecond or its share of the memory's rate, the merge 3.5 us and 0.04 us per split) it was 2.2 % and 21 % up to 240 pairs: one
// sequence of 12 heads of width 64 and 4096 rows in 15 splits 12.8 us, in 8 (one step each) 10.3; 4 of 16 heads of width 128 and
// 4096 rows in 3 splits 20.5 us, in 4 18.4; 8 of them with 1500 rows in one 16.5 us, in 2 15.2; 17 with 4096 rows in one 63 us, in
// 3 55 (a few compute units have two workgroups); 24 of 12 heads of width 64 and 1064 rows in one 13.8 us, in 3 15.1.
inline int decode_choose_splits(int64_t rows, int head_dim, int64_t pairs, int max_splits)
{
    const int step = decode_step_rows(head_dim), row_bytes = 2 * head_dim + 8;
    const double memory = (double)rows * row_bytes * (double)pairs / 6800.0;
    int best = 1;
    double best_ns = 0.0;
    for (int s = 1; s <= max_splits && (s == 1 || s * pairs <= 1024); ++s) {
        const bool power = (s & (s - 1)) == 0;
        const int64_t per = (rows + s - 1) / s, last = per % step, shared = (pairs * s + 255) / 256;
        double walked = (double)(per - last) + (last ? (last > 0.3 * step ? (double)last : 0.3 * step) : 0.0);
        if (walked < (double)(per * shared)) walked = (double)(per * shared);
        const double walk = walked * row_bytes / 33.0;
        const double ns = (walk > memory ? walk : memory) + (s > 1 ? 2000.0 + 280.0 * s + 3.0 * (double)(pairs * s) + (power ? 0.0 : 200.0) : 0.0);
        if (s == 1 || ns < best_ns) { best_ns = ns; best = s; }
        if (per <= step && power) break; // (more splits shorten no workgroup's walk)
    }
    return best;
}

// What a decode launch has to do.  An int8 launch that also adds the new row is one kind whether its rows come from a launch before it or from
// its own front: a layer's one call and the chain of calls that it stands for add up in the same order.
enum DecodeKind { DECODE_I8, DECODE_E4M3, DECODE_I8_APPEND };

constexpr int DECODE_WIDE_GROUPS = 256; // compute units

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
// (up to a quarter of a step both take the four's short steps).  With sixteen waves the other fifteen ask for their rows while the first makes
// the front, so that shorter ranges gain, too; above half a step an appending launch without one loses more than it gains.  With more
// workgroups than compute units the four are the better share: 288 of width 64, 1500 rows 12.9 and 15.7 us; 96 pairs of 1024 rows in
// three splits 9.5 and 11.9.
inline bool decode_wide(int64_t rows, int head_dim, int64_t groups, DecodeKind kind = DECODE_I8)
{
    const int step = decode_step_rows(head_dim);
    return groups <= DECODE_WIDE_GROUPS && (rows > step || (kind != DECODE_I8 && rows <= step / 2));
}

} // namespace tsattn
