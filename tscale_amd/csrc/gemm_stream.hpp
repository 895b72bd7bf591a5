// The int8 product with few activation rows and a matrix of tens of megabytes (the final layer: one row per label).
//
//   out[m][n] = sum over k of a[m][k] * w[n][k],   m up to 32 rows
//
// Bound by the rate at which memory delivers the matrix.  One workgroup of eight waves per compute unit holds the activations in
// LDS and walks a run of the matrix in stages of 16 rows x 128 bytes, a wave an equal number of consecutive stages: memory
// writes them straight into the wave's own ring in LDS, GS_STAGES - 1 stages (64 KiB per compute unit) on their way at any time
// and no barrier in the loop.  A request covers 8 rows x 128 bytes, whole lines; requests into registers in the operand's layout
// touch 16 rows x 64 bytes each and end at 4.4 TB/s (50257 x 2048 under one row: 26.3 us that way, 20.4 us = 5.0 TB/s this way,
// start and end of the launch included).  A block of 16 rows that begins in one wave's share and ends in the next's
// is added up through LDS at the end.
#pragma once

#include "gemm_few.hpp"
#include "stream_walk.h"

namespace tsattn {

constexpr int GS_THREADS = 512, GS_WAVES = GS_THREADS / WAVE, GS_STAGES = 5, GS_STAGE_BYTES = 2048;
typedef __attribute__((address_space(3))) void *gs_lds_ptr;

// LDS: int8 rows [16 MT][k + 16] (the sums of shared blocks at the end), the waves' rings
inline int64_t gs_rows_bytes(int mt, int64_t k)
{
    const int64_t rows = (int64_t)16 * mt * (k + 16), sums = (int64_t)GS_WAVES * mt * WAVE * 16;
    return ((rows > sums ? rows : sums) + 127) & ~(int64_t)127;
}
inline int64_t gs_lds_bytes(int mt, int64_t k) { return gs_rows_bytes(mt, k) + GS_WAVES * GS_STAGES * GS_STAGE_BYTES; }

// (functions of their own, and not templates: inside the kernel the host pass of the compiler drops the kernel)
__device__ __forceinline__ void gs_request(__amdgpu_buffer_rsrc_t r, uint8_t *dst, int off, int scalar_off)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (gs_lds_ptr)dst, 16, off, scalar_off, 0, 2); // (data that is not used again soon)
}
__device__ __forceinline__ void gs_wait_stage() { asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); } // all but the newest GS_STAGES - 1 stages have landed

template <int MODE, int MT>
__global__ __launch_bounds__(GS_THREADS) void gemm_stream_kernel(FewParams p)
{
#pragma clang fp contract(off)
    static_assert(GS_STAGES == 5, "two requests per stage, counted in gs_wait_stage");
    extern __shared__ __attribute__((aligned(128))) uint8_t gs_lds[];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int r16 = lane & 15, g = lane >> 4;
    const int k = (int)p.k, pitch = k + 16, ns = (k + 127) / 128; // (the last stage may hold only half of its bytes)
    const int b0 = (int)blockIdx.x * p.blk_per + min((int)blockIdx.x, p.blk_more), b1 = b0 + p.blk_per + ((int)blockIdx.x < p.blk_more ? 1 : 0);
    const int total = (b1 - b0) * ns;
    auto share = [&](int w) { return (int)((int64_t)w * total / GS_WAVES); }; // where wave w's stages begin
    const int t0 = share(wave), t1 = share(wave + 1);
    uint8_t *const a_lds = gs_lds;
    uint8_t *const ring = gs_lds + p.k_chunk + wave * (GS_STAGES * GS_STAGE_BYTES); // (k_chunk: bytes of the rows)

    // ---- requests: lane L of one fills position L % 8 of row L / 8 (+ 8), which holds chunk (L % 8) ^ (row / 2) % 8 of the stage's
    // row: row-per-lane reads then touch every bank once
    const int row = lane >> 3, chunk = (lane & 7) ^ (row >> 1);
    const int off0 = row * (int)p.w_pitch + chunk * 16, off1 = (row + 8) * (int)p.w_pitch + (chunk ^ 4) * 16;
    StreamWalk walk = stream_walk(b0, t0, t1, ns);
    int ask_slot = 0;
    auto ask = [&]() __attribute__((always_inline)) {
        const StreamStage st = stream_next(walk, (int)p.n, k, (int)p.w_pitch);
        const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.w + (int64_t)st.block * 16 * p.w_pitch), 0, st.size, 0x00020000);
        uint8_t *const d = ring + ask_slot * GS_STAGE_BYTES;
        gs_request(wr, d, off0, st.scalar_off);
        gs_request(wr, d + 1024, off1, st.scalar_off);
        ask_slot = ask_slot == GS_STAGES - 1 ? 0 : ask_slot + 1;
    };

    // ---- the activations; what is asked for first arrives first, and they have the longer way
    {
        constexpr int QB = 8;
        const int per_row = k / 16, pieces = (int)p.m * per_row;
        for (int base = 0; base < pieces; base += QB * GS_THREADS) {
            v4i q[QB];
            int dst[QB];
#pragma unroll
            for (int i = 0; i < QB; ++i) {
                const int j = base + i * GS_THREADS + tid, jc = j < pieces ? j : pieces - 1;
                const int m = (int)wg_div_small((uint32_t)jc, p.by_row), c = jc - m * per_row;
                dst[i] = m * pitch + c * 16;
                q[i] = *(const v4i *)(p.a + (uint32_t)(m * (int)p.a_pitch + c * 16));
            }
            if (base + QB * GS_THREADS >= pieces) {
                __builtin_amdgcn_sched_barrier(0);
                for (int i = 0; i < GS_STAGES; ++i) ask();
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < QB; ++i) *(v4i *)(a_lds + dst[i]) = q[i];
        }
    }
    gf_barrier();

    // acc[t][i]: activation row 16 t + lane % 16, weight row 16 blk + 4 (lane / 16) + i
    auto store = [&](int blk, const v4i(&acc)[MT]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const int m = 16 * t + r16, n = blk * 16 + 4 * g;
            if (m >= p.m || n >= p.n) continue;
            const int64_t at = (int64_t)m * p.out_pitch + n;
            if (MODE == TSATTN_MM_I32) {
                int32_t *const o = (int32_t *)p.out + at;
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
    v4i acc[MT], head[MT]; // head: the end of a block that began in an earlier wave's share
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = head[t] = v4i{0, 0, 0, 0};
    const uint8_t *const a_row = a_lds + r16 * pitch + g * 16;
    const int w_at = r16 * 128 + ((g ^ (r16 >> 1)) << 4); // (chunk 4 + g of the stage: bit 6 the other way round)
    int blk = b0 + t0 / ns, s = t0 % ns, slot = 0;
    bool begun_before = s != 0;
    for (int i = t0; i < t1; ++i) {
        gs_wait_stage();
        const uint8_t *const st = ring + slot * GS_STAGE_BYTES;
        slot = slot == GS_STAGES - 1 ? 0 : slot + 1;
        const v4i x0 = *(const v4i *)(st + w_at), x1 = *(const v4i *)(st + (w_at ^ 64));
        v4i y0[MT], y1[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            y0[t] = *(const v4i *)(a_row + t * 16 * pitch + s * 128);
            y1[t] = *(const v4i *)(a_row + t * 16 * pitch + s * 128 + 64);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the stage has been read: its place may be written again
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x0, y0[t], acc[t], 0, 0, 0);
        if (s * 128 + 64 < k) {
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x1, y1[t], acc[t], 0, 0, 0);
        }
        ask();
        if (++s == ns) {
            if (begun_before) {
#pragma unroll
                for (int t = 0; t < MT; ++t) head[t] = acc[t];
            } else {
                store(blk, acc);
            }
            begun_before = false;
            s = 0;
            ++blk;
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = v4i{0, 0, 0, 0};
        }
    }
    if (begun_before) { // the whole share lies inside one block, and neither begins nor ends it
#pragma unroll
        for (int t = 0; t < MT; ++t) head[t] = acc[t];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // nothing may still be on its way into LDS when the workgroup ends
    gf_barrier();
    v4i *const heads = (v4i *)gs_lds;
#pragma unroll
    for (int t = 0; t < MT; ++t) heads[(wave * MT + t) * WAVE + lane] = head[t];
    gf_barrier();
    if (begun_before || s == 0) return; // no block that begins here and ends later
    for (int w = wave + 1; w < GS_WAVES; ++w) {
        const int at = share(w);
        if (at >= (blk - b0 + 1) * ns) break;
        if (at == share(w + 1)) continue;
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] += heads[(w * MT + t) * WAVE + lane];
    }
    store(blk, acc);
}

} // namespace tsattn
