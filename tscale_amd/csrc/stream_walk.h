// The order in which a wave of gemm_stream_kernel asks for its share of the matrix: plain C++, so that it can be tested without a
// GPU.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define TSATTN_HD __host__ __device__
#else
#define TSATTN_HD
#endif

namespace tsattn {

// One stage: 16 rows x 128 bytes at byte 128 * stage of the rows from row 16 * block on.  A stage of nothing (past the wave's share,
// so that one count of requests holds for every step) has no bytes and begins at byte 0: a range check never meets an offset beyond
// the size.
struct StreamStage {
    int block;
    int size;       // bytes from the block's first row to the end of its last row; 0: nothing
    int scalar_off; // where in the rows the stage begins
};

struct StreamWalk {
    int block, stage, left, stages; // next stage, stages left in the share, stages per block
};

TSATTN_HD inline StreamWalk stream_walk(int first_block, int begin, int end, int stages)
{
    return StreamWalk{first_block + begin / stages, begin % stages, end - begin, stages};
}

// the next stage of the walk (n rows of k bytes, w_pitch apart)
TSATTN_HD inline StreamStage stream_next(StreamWalk &w, int n, int k, int w_pitch)
{
    if (w.left <= 0) return StreamStage{0, 0, 0};
    const int rows = n - w.block * 16 < 16 ? n - w.block * 16 : 16;
    const StreamStage s = {w.block, (rows - 1) * w_pitch + k, w.stage * 128};
    --w.left;
    if (++w.stage == w.stages) { w.stage = 0; ++w.block; }
    return s;
}

} // namespace tsattn
