// Device side of the few-row int8 product (gemm_few.hip): one kernel body, four sources of the activations.
//
//   out[part][m][n] = sum over part's K of a[m][k] * w[n][k],   m up to 128 rows
//
// Bound by the time to bring the weights in once, and below a few megabytes by latencies.  A wave takes 16 weight rows and
// a stretch of K straight from memory into the registers v_mfma_i32_16x16x64_i8 multiplies from (16 bytes per lane: 16 rows
// times 64 consecutive bytes per request, eight requests on their way before the first is used): the weights cross neither
// LDS nor a barrier.  The activations of the workgroup's part of K stand in LDS.  Waves that share weight rows add up in
// LDS; parts of K that go to different workgroups become planes of the result.
//
// A launch of a few microseconds is mostly the instructions before its first load: about one per 3 ns and wave.  So the start has
// no division (runs of blocks and reciprocals come from the host; the two 64-bit divisions that gave a workgroup its run and the
// eight that placed a thread's pieces were 700 instructions) and 32-bit offsets from scalar bases, and no weight request is behind a
// branch, which would make the activations wait for the weights.  768 x 3072 under one row: activations in LDS 2.6 us after the
// start, now 1.4; its normalising forms end after 4.1 instead of 5.6 us.
//
// The activations are int8 rows in memory, or they are made here: the rows a normalisation of the layer would have written
// (state and the planes of the product before it in, RMS normalisation per group, int8 out), for the part of K this
// workgroup multiplies.  Every workgroup repeats that for its columns, which costs it their bytes from L2, and a launch and
// its memory round trip are gone from the chain that a token step is.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace tsattn {

constexpr int GF_U = 8;                 // requests of 64 bytes of K per weight row and round
constexpr int GF_LDS_MAX = 160 << 10;
typedef int v4i_u __attribute__((ext_vector_type(4), aligned(4)));

// LDS: int8 rows [16 MT][kc + 16], values and their squares [pairs][group + 4] and a multiplier per pair where they are normalised here
inline int gf_lds_bytes(int waves, int mt, int64_t m, int64_t kc, int group)
{
    int64_t b = (int64_t)16 * mt * (kc + 16);
    if (group) b += m * (kc / group) * (2 * (group + 4) + 1) * 4;
    const int64_t sums = (int64_t)waves * mt * WAVE * 16;
    return (int)(b > sums ? b : sums);
}

template <int N>
using Pieces = std::integral_constant<int, N>;

// a barrier for LDS traffic only: requests to memory stay on their way over it
__device__ __forceinline__ void gf_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// SRC -1: int8 rows.  SRC >= 0: that many int32 planes (RESID: added to the state), or the state alone (SRC 0).
// NT: the weights are asked for as data that will not be used again soon.
//
// Where the source is planes alone (the feed-forward block's second product), the launch also carries a residual update
// that the launch before it has read past: state += planes * scale, spread over the grid, one group of four per thread.
template <int GF_THREADS, int MODE, int MT, int SRC, bool RESID, bool NT>
__global__ __launch_bounds__(GF_THREADS) void gemm_few_kernel(FewParams p)
{
#pragma clang fp contract(off)
    extern __shared__ __attribute__((aligned(16))) uint8_t gf_lds[];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wn = wave & (p.wn - 1), wk = wave >> p.wn_log;
    const int r16 = lane & 15, g = lane >> 4;
    const int k_begin = (int)blockIdx.y * p.k_part, k_end = min((int)p.k, k_begin + p.k_part);
    // This wave's blocks of 16 weight rows: every wn-th of the workgroup's run of them (one, unless there are so many that
    // workgroups which stage the activations once and walk several blocks are the better cut).
    const int begin = (int)blockIdx.x * p.blk_per + min((int)blockIdx.x, p.blk_more);
    const int blk0 = begin + wn, blk_end = begin + p.blk_per + ((int)blockIdx.x < p.blk_more ? 1 : 0);
    const int w_off = r16 * (int)p.w_pitch + g * 16;

    const int pitch = p.k_chunk + 16;
    uint8_t *const a_lds = gf_lds;
    float *const vals = (float *)(gf_lds + 16 * MT * pitch);
    v4i acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = v4i{0, 0, 0, 0};
    constexpr bool UPDATES = SRC > 0 && !RESID;
    ResidUpdate update;
    if constexpr (UPDATES) update.request(p.upd, ((int)blockIdx.y * gridDim.x + blockIdx.x) * GF_THREADS + tid, (int)(gridDim.x * gridDim.y) * GF_THREADS);

    // acc[t][i]: activation row 16 t + lane % 16, weight row 16 blk + 4 (lane / 16) + i
    auto store = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            if ((t & (p.wk - 1)) != wk) continue; // (the waves of a row group store a share each; all of it where there is one)
            const int m = 16 * t + r16, n = blk * 16 + 4 * g;
            if (m >= p.m || n >= p.n) continue;
            const int64_t at = (int64_t)m * p.out_pitch + n;
            if (MODE == TSATTN_MM_I32) {
                int32_t *const o = (int32_t *)p.out + (int64_t)blockIdx.y * p.out_stride + at;
                if (n + 4 <= p.n) *(v4i_u *)o = acc[t];
                else
                    for (int i = 0; i < 4; ++i)
                        if (n + i < p.n) o[i] = acc[t][i];
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (n + i >= p.n) continue;
                    float *const o = (float *)p.out + at + i;
                    const float y = (float)acc[t][i] * p.scale;
                    *o = MODE == TSATTN_MM_F32 ? y : *o + y;
                }
            }
        }
    };

    for (int kc = k_begin; kc < k_end; kc += p.k_chunk) { // (one round unless the rows of this part do not fit into LDS)
        const int len = min(p.k_chunk, k_end - kc);
        // this wave's stretch of the chunk, in steps of 64 bytes
        const int steps = len / 64, per = (steps + p.wk - 1) >> p.wk_log;
        const int s0 = wk * per, s1 = min(steps, s0 + per);
        v4i w[2][GF_U];
        // a round of requests: a block of rows and where in K it starts
        struct Round {
            int blk, s;
        };
        auto after = [&](const Round &r) __attribute__((always_inline)) { return r.s + GF_U < s1 ? Round{r.blk, r.s + GF_U} : Round{r.blk + p.wn, s0}; };
        auto request = [&](v4i(&dst)[GF_U], const Round &r) __attribute__((always_inline)) {
            // (rows past n, and a round that is not there: zero bytes)
            const int blk = r.blk < blk_end ? r.blk : blk_end - 1, n0 = blk * 16, rows = min(16, (int)p.n - n0);
            const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.w + (int64_t)n0 * p.w_pitch), 0,
                                                                                r.blk < blk_end ? (rows - 1) * (int)p.w_pitch + (int)p.k : 0, 0x00020000);
#pragma unroll
            for (int u = 0; u < GF_U; ++u)
                dst[u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wr, w_off + kc + (r.s + u) * 64, 0, NT ? 2 : 0));
        };
        Round r0 = Round{s0 < s1 ? blk0 : blk_end, s0}, r1 = after(r0);
        auto first_requests = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            request(w[0], r0);
            request(w[1], r1);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (kc != k_begin) gf_barrier(); // the chunk before has been multiplied

        // The activations' requests go out first: what is requested first arrives first, and they have the longer way
        // to the multiplication.  The weights' requests follow in the last round whatever there is to ask for: behind a branch they
        // would have to be waited for together with the activations.
        if constexpr (SRC < 0) {
            const int per_row = len / 16, total = (int)p.m * per_row;
            const WgDiv by_row = len == p.k_chunk ? p.by_row : wg_make_div((uint32_t)per_row);
            auto stage = [&](auto pieces, auto last, int base) __attribute__((always_inline)) { // pieces of every thread
                constexpr int QB = decltype(pieces)::value;
                v4i q[QB];
                int dst[QB];
#pragma unroll
                for (int i = 0; i < QB; ++i) {
                    const int j = base + i * GF_THREADS + tid, jc = j < total ? j : total - 1;
                    const int row = (int)wg_div_small((uint32_t)jc, by_row), c = jc - row * per_row;
                    dst[i] = row * pitch + c * 16;
                    q[i] = *(const v4i *)(p.a + kc + (uint32_t)(row * (int)p.a_pitch + c * 16));
                }
                if constexpr (decltype(last)::value) first_requests();
#pragma unroll
                for (int i = 0; i < QB; ++i) {
                    *(v4i *)(a_lds + dst[i]) = q[i];
                }
            };
            if (total <= GF_THREADS) { // (one row: the rest of a round would be instructions for nothing)
                stage(Pieces<1>(), std::true_type(), 0);
            } else {
                constexpr int QB = 8;
                int base = 0;
                for (; base + QB * GF_THREADS < total; base += QB * GF_THREADS) stage(Pieces<QB>(), std::false_type(), base);
                stage(Pieces<QB>(), std::true_type(), base);
            }
            gf_barrier();
        } else {
            const int G = p.group, per_row = len / 4, total = (int)p.m * per_row, groups = len / G, pairs = (int)p.m * groups;
            float *const squares = vals + pairs * (G + 4), *const mults = squares + pairs * (G + 4);
            const WgDiv by_row = len == p.k_chunk ? p.by_row : wg_make_div((uint32_t)per_row);
            auto stage = [&](auto pieces, auto last, int base) __attribute__((always_inline)) {
                constexpr int QB = decltype(pieces)::value;
                v4i sum[QB][SRC > 0 ? SRC : 1];
                v4f st[QB];
                int at[QB];
#pragma unroll
                for (int i = 0; i < QB; ++i) {
                    const int j = base + i * GF_THREADS + tid, jc = j < total ? j : total - 1;
                    const int row = (int)wg_div_small((uint32_t)jc, by_row), x = (jc - row * per_row) * 4;
                    at[i] = (row * groups + (x >> p.group_log)) * (G + 4) + (x & (G - 1));
#pragma unroll
                    for (int s = 0; s < SRC; ++s) sum[i][s] = *(const v4i *)((const char *)(p.src + s * p.src_stride + kc) + (uint32_t)(row * (int)p.k + x) * 4u);
                    if (RESID) st[i] = *(const v4f *)((const char *)(p.state + kc) + (uint32_t)(row * (int)p.state_pitch + x) * 4u);
                }
                if constexpr (decltype(last)::value) first_requests();
#pragma unroll
                for (int i = 0; i < QB; ++i) {
                    v4f v;
                    if (SRC > 0) {
                        v4i a = sum[i][0];
#pragma unroll
                        for (int s = 1; s < SRC; ++s) a += sum[i][s];
                        v = v4f{(float)a.x, (float)a.y, (float)a.z, (float)a.w};
                        if (RESID) { // the state as the residual update leaves it (delta * scale rounded before it is added)
                            v = v4f{v.x * p.resid_scale, v.y * p.resid_scale, v.z * p.resid_scale, v.w * p.resid_scale};
                            v = v4f{st[i].x + v.x, st[i].y + v.y, st[i].z + v.z, st[i].w + v.w};
                        }
                    } else {
                        v = st[i];
                    }
                    *(v4f *)(vals + at[i]) = v;
                    *(v4f *)(squares + at[i]) = v4f{v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w};
                }
            };
            if (total <= GF_THREADS) { // (one row: the rest of a round would be instructions for nothing)
                stage(Pieces<1>(), std::true_type(), 0);
            } else {
                constexpr int QB = SRC + (RESID ? 1 : 0) <= 3 ? 8 : 4;
                int base = 0;
                for (; base + QB * GF_THREADS < total; base += QB * GF_THREADS) stage(Pieces<QB>(), std::false_type(), base);
                stage(Pieces<QB>(), std::true_type(), base);
            }
            if constexpr (UPDATES) {
                if (kc == k_begin) update.finish(p.upd);
            }
            gf_barrier();
            for (int pr = tid; pr < pairs; pr += GF_THREADS) { // squares added in index order, as the producer does
                const float *const v = squares + pr * (G + 4);
                float sum2 = 0.0f;
                v4f q0[4], q1[4]; // (sixteen on their way while sixteen are added)
                auto read = [&](v4f(&q)[4], int x) __attribute__((always_inline)) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) q[c] = *(const v4f *)(v + x + 4 * c);
                };
                auto add = [&](const v4f(&q)[4]) __attribute__((always_inline)) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        sum2 = sum2 + q[c].x;
                        sum2 = sum2 + q[c].y;
                        sum2 = sum2 + q[c].z;
                        sum2 = sum2 + q[c].w;
                    }
                };
                read(q0, 0);
#pragma unroll 1
                for (int x = 0; x < G; x += 32) {
                    read(q1, x + 16);
                    add(q0);
                    read(q0, x + 32 < G ? x + 32 : 0);
                    add(q1);
                }
                float mult = 0.0f;
                if (sum2 != 0.0f) mult = 1.0f / (sqrt_rounded(sum2 / (float)G) * p.vec_scale);
                mults[pr] = mult;
            }
            gf_barrier();
            const float low = p.relu ? 0.0f : -127.0f;
            for (int j = tid; j < total; j += GF_THREADS) {
                const int row = (int)wg_div_small((uint32_t)j, by_row), x = (j - row * per_row) * 4, pr = row * groups + (x >> p.group_log);
                const v4f v = *(const v4f *)(vals + pr * (G + 4) + (x & (G - 1)));
                const float mult = mults[pr]; // a group of zeros has 0: zero bytes
                *(uint32_t *)(a_lds + row * pitch + x) = pack_i8x4(v.x * mult, v.y * mult, v.z * mult, v.w * mult, low);
            }
            gf_barrier();
        }

        // rows past m hold whatever LDS held: their sums are not stored
        const uint8_t *const ab = a_lds + r16 * pitch + g * 16;
        auto multiply = [&](const v4i(&x)[GF_U], const Round &r) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < GF_U; ++u) {
                if (r.s + u < s1) { // uniform
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        const v4i y = *(const v4i *)(ab + t * 16 * pitch + (r.s + u) * 64);
                        acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[u], y, acc[t], 0, 0, 0);
                    }
                }
            }
        };
        auto step = [&](v4i(&x)[GF_U], Round &r, const Round &other) __attribute__((always_inline)) {
            multiply(x, r);
            const int done = r.s + GF_U >= s1 ? r.blk : -1; // this block's last round
            r = after(other);
            if (r.blk < blk_end) request(x, r);
            if (done >= 0 && p.walk) {
                store(done);
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] = v4i{0, 0, 0, 0};
            }
        };
        while (r0.blk < blk_end) {
            step(w[0], r0, r1);
            if (r1.blk < blk_end) step(w[1], r1, r0);
        }
    }
    if (p.walk) return;

    if (p.wk > 1) {
        gf_barrier();
        v4i *const red = (v4i *)gf_lds;
#pragma unroll
        for (int t = 0; t < MT; ++t) red[(wave * MT + t) * WAVE + lane] = acc[t];
        gf_barrier();
        // the waves of a row group share its blocks of 16 activation rows out
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            if ((t & (p.wk - 1)) != wk) continue;
            for (int i = 0; i < p.wk; ++i)
                if (i != wk) acc[t] += red[((wn + (i << p.wn_log)) * MT + t) * WAVE + lane];
        }
    }
    if (blk0 < blk_end) store(blk0);
}

} // namespace tsattn
