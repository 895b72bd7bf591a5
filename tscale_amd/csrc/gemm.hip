// int8 x int8 -> int32 matrix product with the epilogues of the reference's int8 inference path:
//   out[m][n] = sum_k a[m][k] * w[n][k]
// MulForward (gpt/train/cpu_infer.cpp:294-305: one weight row per output, exact int32 sums, result as int32 or
// converted to float) and AddScaled (:308-316: state += delta * scale).
//
// Here the largest products (256 x 256 output tiles; bound by the matrix cores) and the choice between the kernels; a few
// hundred to a few thousand rows: gemm_mid.hip, few rows (one token per sequence): gemm_few.hpp.
// Integer sums are exact, so every decomposition gives the same bits.
#include <algorithm>
#include <type_traits>
#include "common.hpp"
#include "kernels.hpp"

namespace tsattn {

namespace {

__device__ inline __amdgpu_buffer_rsrc_t rows_rsrc(const void *base, int64_t rows, int64_t pitch, int64_t row_bytes)
{
    // the last row ends after row_bytes, not after a whole pitch
    int64_t bytes = rows <= 0 ? 0 : (rows - 1) * pitch + row_bytes;
    const uint32_t n = bytes > 0xffffffffll ? 0xffffffffu : (uint32_t)bytes;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)n, 0x00020000);
}

template <int MODE>
__device__ inline void store_out(const GemmParams &p, int64_t m, int64_t n, int acc)
{
#pragma clang fp contract(off) // delta * scale is rounded before it is added, as in the reference's two statements
    if (MODE == TSATTN_MM_I32) {
        ((int32_t *)p.out)[m * p.out_pitch + n] = acc;
    } else if (MODE == TSATTN_MM_F32) {
        ((float *)p.out)[m * p.out_pitch + n] = (float)acc * p.scale;
    } else {
        float *o = (float *)p.out + m * p.out_pitch + n;
        *o += (float)acc * p.scale; // (*pRes)[k] += delta[k] * scale
    }
}

// Wide tiles for the largest products: 256 x 256 outputs by eight waves, K in steps of 64 bytes, one
// workgroup per compute unit; per MFMA cycle this moves a third less through LDS and the caches than 256 x 128 tiles.
// Each SIMD holds two of the waves, one from each half of the workgroup, and the halves run half a step apart: while
// one half issues the 16 MFMAs of its step, the other does its memory work (requests its share of the tile three
// steps on, which memory writes straight into LDS, and reads its operands of the next step from LDS), then they swap
// at a barrier.  The MFMA pipe always has a wave feeding it and no wave waits for memory while it feeds.  Four LDS
// buffers of 32 KiB: one being read, three tiles on their way (a request has two whole steps to land).
// LDS rows are 64 bytes without padding; the 16-byte chunks of a row are permuted by (row / 4) % 4, which keeps the
// row-per-lane operand reads free of bank conflicts; a memory-to-LDS request writes the 64 lanes' 16 bytes one after
// the other, so the permutation is applied to the addresses the lanes request.  K must be a multiple of 64.
constexpr int GW_THREADS = 512, GW_BM = 256, GW_BN = 256, GW_BK = 64, GW_NBUF = 4;
constexpr int GW_BUF = (GW_BM + GW_BN) * GW_BK;
constexpr int GW_LDS_BYTES = GW_NBUF * GW_BUF;
typedef int v4i_w __attribute__((ext_vector_type(4), aligned(4)));
typedef float v4f_w __attribute__((ext_vector_type(4), aligned(4)));

// four values of lanes 16..31 and 48..63 of lo change places with those of lanes 0..15 and 32..47 of hi
__device__ __forceinline__ void swap16(float *lo, float *hi)
{
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const auto y = __builtin_amdgcn_permlane16_swap(__float_as_uint(lo[c]), __float_as_uint(hi[c]), false, false);
        lo[c] = __uint_as_float(y[0]);
        hi[c] = __uint_as_float(y[1]);
    }
}

template <int MODE, int EP_D>
__global__ __launch_bounds__(GW_THREADS, 1) void gemm_wide_kernel(GemmParams p)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t gw_lds[];
    typedef __attribute__((address_space(3))) void *lds_ptr;
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int half = wave >> 2; // waves 0-3 and 4-7 land on SIMDs 0-3 each
    // A wave's share is four blocks of 32 of the matrix instructions' first operand by two of the second.  For a plain result the
    // activations come first: 128 rows x 64 columns, columns over lanes, so that it leaves in whole lines.  With the producer
    // as epilogue the weights come first: 64 rows x 128 columns; lane li of acc[j][i] has row 32 i + li of the wave's rows and, four
    // after four, the columns 32 j + 8 (r / 4) + 4 g + r % 4 -- a row's values lie in two lanes instead of over all of them.
    // (The result of 65536 x 2048 -> 8192 as int32: 1240 us, 1328 with a row per lane.)
    constexpr bool ROWS = EP_D != 0;
    const int wm = ROWS ? wave & 3 : wave >> 2, wn = ROWS ? wave >> 2 : wave & 3;
    const int li = lane & 31, g = lane >> 5;

    // Which output tile.  The 8 XCDs take workgroups round-robin and each has its own L2; the workgroups an XCD runs at a
    // time walk through K at about the same pace, so its L2 only has to hold the current slices of the rows they use.  8 x 8
    // blocks of tiles per XCD where the shape allows: 8 tiles of activations and 8 of weights cross the fabric per 64
    // output tiles instead of up to 64 + 8.  Shapes that do not divide that way walk along rows of tiles.
    const int64_t tiles_n = (p.n + GW_BN - 1) / GW_BN, tiles_m = (p.m + GW_BM - 1) / GW_BM;
    int64_t tile_m, tile_n;
    if (tiles_n % 8 == 0 && tiles_m % 8 == 0 && ((tiles_n >> 3) * (tiles_m >> 3)) % 8 == 0) {
        const int64_t x = blockIdx.x & 7, l = blockIdx.x >> 3;
        const int64_t sb = (l >> 6) * 8 + x, within = l & 63;
        const int64_t sb_per_row = tiles_n >> 3;
        tile_m = (sb / sb_per_row) * 8 + (within >> 3);
        tile_n = (sb % sb_per_row) * 8 + (within & 7);
    } else {
        tile_m = blockIdx.x / tiles_n;
        tile_n = blockIdx.x % tiles_n;
    }
    const int64_t m0 = tile_m * GW_BM, n0 = tile_n * GW_BN;
    const __amdgpu_buffer_rsrc_t ar = rows_rsrc(p.a + m0 * p.a_pitch, p.m - m0 < GW_BM ? p.m - m0 : GW_BM, p.a_pitch, p.k);
    const __amdgpu_buffer_rsrc_t wr = rows_rsrc(p.w + n0 * p.w_pitch, p.n - n0 < GW_BN ? p.n - n0 : GW_BN, p.w_pitch, p.k);
    // A buffer holds 256 rows of A, then 256 rows of W.  A wave's request fills 16 rows (1 KiB): lane L writes the
    // chunk at position L % 4 of row L / 4, which is chunk (L % 4) ^ perm(row) of the matrix row.  Rows
    // wave * 16 + 128 i: perm depends on the lane only.
    const int sr = wave * 16 + (lane >> 2), sc = (lane & 3) ^ ((lane >> 4) & 3);
    const int a_off0 = sr * (int)p.a_pitch + sc * 16, a_off1 = a_off0 + 128 * (int)p.a_pitch;
    const int w_off0 = sr * (int)p.w_pitch + sc * 16, w_off1 = w_off0 + 128 * (int)p.w_pitch;
    auto request = [&](int kb, uint8_t *buf) __attribute__((always_inline)) { // tile at K offset kb -> buf
        uint8_t *const d = buf + wave * 16 * GW_BK;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (lds_ptr)(d), 16, a_off0, kb, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (lds_ptr)(d + 128 * GW_BK), 16, a_off1, kb, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr)(d + 256 * GW_BK), 16, w_off0, kb, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr)(d + 384 * GW_BK), 16, w_off1, kb, 0, 0);
    };
    // operands: row li of each 32-row block, chunk 2 * h + g of its 64 bytes (h: which 32 bytes of the step)
    const int f_perm = (li >> 2) & 3;
    const int row_a = wm * (ROWS ? 64 : 128) + li, row_w = GW_BM + wn * (ROWS ? 128 : 64) + li;
    const int at4 = (ROWS ? row_w : row_a) * GW_BK + ((g ^ f_perm) << 4), at2 = (ROWS ? row_a : row_w) * GW_BK + ((g ^ f_perm) << 4);
    v4i f4[2][4], f2[2][2];
    v16i acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = v16i{0};

    // A barrier that waits for this wave's LDS reads only: __syncthreads() would also wait for every tile still on its
    // way into LDS, which is exactly what must stay in flight.  What has to have landed is waited for by count.
#define GW_BARRIER                                              \
    do {                                                        \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      \
        __builtin_amdgcn_s_barrier();                           \
        asm volatile("" ::: "memory");                          \
    } while (0)
    const int n_steps = (int)(p.k / GW_BK);
    // (with the producer as epilogue: the positions of this lane's rows, asked for now, so that the epilogue's rope rows do not
    // wait for them)
    int row_pos[2] = {0, 0};
    if constexpr (EP_D != 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int64_t m = m0 + wm * 64 + i * 32 + li;
            if (p.ep.pos && m < p.m) row_pos[i] = p.ep.pos[m];
        }
    }
    const int k_bytes = (int)p.k;
    request(0, gw_lds);
    request(wide_k_offset(1, GW_BK, k_bytes), gw_lds + GW_BUF);
    request(wide_k_offset(2, GW_BK, k_bytes), gw_lds + 2 * GW_BUF);
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); // this wave's share of the first tile has landed
    GW_BARRIER;
    if (half == 1) GW_BARRIER; // the second half of the workgroup runs half a step behind the first
#define GW_FENCE __builtin_amdgcn_sched_barrier(0)
    for (int s = 0; s < n_steps; ++s) {
        uint8_t *const cur = gw_lds + (s & 3) * GW_BUF;
        // memory half: request the tile of step s + 3 into the buffer step s - 1 was read from, read this step's
        // operands, make sure this wave's share of the tile of step s + 1 has landed before the barrier
        GW_FENCE;
        request(wide_k_offset(s + 3, GW_BK, k_bytes), gw_lds + ((s + 3) & 3) * GW_BUF);
        GW_FENCE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int j = 0; j < 4; ++j) f4[h][j] = *(const v4i *)(cur + ((at4 + j * 32 * GW_BK) ^ (h * 32)));
#pragma unroll
            for (int i = 0; i < 2; ++i) f2[h][i] = *(const v4i *)(cur + ((at2 + i * 32 * GW_BK) ^ (h * 32)));
        }
        GW_FENCE;
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        GW_BARRIER;
        // MFMA half
        GW_FENCE;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f4[h][j], f2[h][i], acc[j][i], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        GW_FENCE;
        GW_BARRIER;
    }
#undef GW_FENCE
    if (half == 0) GW_BARRIER;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // nothing may still be on its way into LDS when the workgroup ends
#undef GW_BARRIER
    if constexpr (EP_D != 0) {
        // The producer as the product's epilogue (the reference's projection kernels end the same way,
        // TStoreRowTileNormalizeRope, gpt/compute/gpt_rope.cuh:4-66): the int32 sums never go to memory.  A wave's 128
        // columns are whole heads.  Residual update and rotation are lane-local (x in acc[2 b][.] and x + 32 in
        // acc[2 b + 1][.]); then one exchange between the wave's halves per two values gives every lane one row's 128
        // values, whose squares it adds up in index order, as the producer kernel and the CPU path do, and converts them:
        // no barrier, and only the bytes go through LDS (to leave as whole lines).  Every float operation as written there.
        // A residual update and a rotation in one call are left to the producer kernel by the launcher.
        // (With the waves' sums in the other layout, columns over lanes, the floats went through LDS 128 rows at a time for
        // the ordered sums, three barriers each: 17.7 of a projection tile's 67 thousand cycles.  65536 rows, bytes alone /
        // with a residual update: 2048 -> 8192 1179 / 1940 us, now 1120 / 1873; 2048 -> 2048 274 / 500, now 256 / 471.)
#pragma clang fp contract(off)
        const ProduceParams &e = p.ep;
        const int rows_here = (int)(p.m - m0 < GW_BM ? p.m - m0 : GW_BM);
        constexpr int HEADS_W = 128 / EP_D; // heads per wave
        const int head0 = (int)(n0 / EP_D) + wn * HEADS_W;
        // Addresses inside the tile are 32-bit offsets from a base that is the same for the whole wave (the launcher
        // checks that the pitches allow it): one add per access instead of a 64-bit multiply.
        char *const resid_base = (char *)(e.resid + m0 * e.resid_pitch + (n0 + wn * 128));
        const uint32_t resid_pitch_bytes = (uint32_t)e.resid_pitch * 4u;
        float val[4][2][16];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) val[j][i][r] = (float)acc[j][i][r];
        // Step s = (i, b): rows of block i, columns 64 b + ..63; what it needs from memory is requested two steps ahead.  State
        // is read and written sixteen rows by 64 bytes at a time: the values of two groups of columns change places between
        // the 16 lanes of the block's upper and lower rows (and back).
        v4f x[2][8];
        const int r16 = lane & 15, c16 = 8 * ((lane >> 4) & 1) + 4 * g;
        auto resid_at = [&](int s, int k) __attribute__((always_inline)) { // k = (column half, 16 of its columns, 16 rows)
            const int row = wm * 64 + (s >> 1) * 32 + (k & 1) * 16 + r16, col = (s & 1) * 64 + (k >> 1) * 16 + c16;
            return resid_base + ((uint32_t)row * resid_pitch_bytes + (uint32_t)col * 4u);
        };
        auto resid_ok = [&](int s, int k) __attribute__((always_inline)) {
            return wm * 64 + (s >> 1) * 32 + (k & 1) * 16 + r16 < rows_here && head0 + (s & 1) * 64 / EP_D < e.n_heads;
        };
        auto request = [&](int s) __attribute__((always_inline)) {
            if (e.resid) {
#pragma unroll
                for (int k = 0; k < 8; ++k) x[s & 1][k] = resid_ok(s, k) ? *(const v4f_w *)resid_at(s, k) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
            } else if (e.pos) {
                const int i = s >> 1, t = row_pos[i] < 0 ? 0 : (row_pos[i] >= e.rope_len ? (int)e.rope_len - 1 : row_pos[i]);
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    x[s & 1][k] = *(const v4f_w *)((const char *)e.rope + ((uint32_t)t * (uint32_t)(EP_D * 4) + (uint32_t)((s & 1) * 64 % EP_D + 8 * k + 4 * g) * 4u));
            }
        };
        request(0);
        request(1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int i = s >> 1, b = s & 1;
            float *const v0 = val[2 * b][i], *const v1 = val[2 * b + 1][i];
            if (e.resid) { // state += delta * scale, written back; the updated state is what gets normalised
#pragma unroll
                for (int k = 0; k < 8; k += 2) {
                    float *const lo = (k < 4 ? v0 : v1) + (k & 2) * 4, *const hi = lo + 4;
                    swap16(lo, hi);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        lo[c] = x[b][k][c] + lo[c] * e.resid_scale;
                        hi[c] = x[b][k + 1][c] + hi[c] * e.resid_scale;
                    }
                    if (resid_ok(s, k)) *(v4f_w *)resid_at(s, k) = v4f{lo[0], lo[1], lo[2], lo[3]};
                    if (resid_ok(s, k + 1)) *(v4f_w *)resid_at(s, k + 1) = v4f{hi[0], hi[1], hi[2], hi[3]};
                    swap16(lo, hi);
                }
            } else if (e.pos && head0 + b * 64 / EP_D < e.rope_heads) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float cos_value = x[b][r / 4][r & 3], sin_value = x[b][4 + r / 4][r & 3] * e.rotate_dir;
                    const float r0 = v0[r] * cos_value - v1[r] * sin_value;
                    const float r1 = v0[r] * sin_value + v1[r] * cos_value;
                    v0[r] = r0;
                    v1[r] = r1;
                }
            }
            if (s < 2) request(s + 2);
        }
        // lane L gets row L of the wave's 64: [j][0] its columns 32 j + 8 q + ..3, [j][1] those 4 further on
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(val[j][0][r]), __float_as_uint(val[j][1][r]), false, false);
                val[j][0][r] = __uint_as_float(y[0]);
                val[j][1][r] = __uint_as_float(y[1]);
            }
        const int row = wm * 64 + lane;
        float mult[HEADS_W];
#pragma unroll
        for (int h = 0; h < HEADS_W; ++h) { // sum of squares in index order, scale
            float sum2 = 0.0f;
#pragma unroll
            for (int j = h * EP_D / 32; j < (h + 1) * EP_D / 32; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const float y = val[j][c >> 2][4 * q + (c & 3)];
                        sum2 = sum2 + y * y;
                    }
            float discr = 0.0f;
            mult[h] = 0.0f;
            if (sum2 != 0.0f) {
                const float sko = (float)sqrt((double)(sum2 / (float)EP_D)); // correctly rounded (see the producer kernel)
                discr = sko * e.vec_scale;
                mult[h] = 1.0f / discr;
            }
            const int hd = head0 + h, sh = hd - e.scale_head_begin;
            if (e.scale && row < rows_here && hd < e.n_heads && sh >= 0 && sh < e.scale_head_count)
                e.scale[sh * e.scale_pitch + (m0 + row) * e.scale_row_stride] = discr * e.scale_mult;
        }
        // Convert; the wave's bytes go through 8 KiB of LDS of its own (16-byte chunk c of row r at c ^ r % 8) and leave as
        // whole lines, eight rows per store.  A head of zeros has mult 0: zero bytes.
        const float low = e.relu ? 0.0f : -127.0f;
        __syncthreads(); // every wave is done with the operand buffers
        uint8_t *const bytes = gw_lds + wave * 64 * 128;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float m = mult[c * 16 / EP_D];
            v4i w;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float *const y = &val[c >> 1][k & 1][4 * ((c & 1) * 2 + (k >> 1))];
                w[k] = (int)pack_i8x4(y[0] * m, y[1] * m, y[2] * m, y[3] * m, low);
            }
            *(v4i *)(bytes + lane * 128 + ((c ^ (lane & 7)) << 4)) = w;
        }
        asm volatile("" ::: "memory"); // (a wave's own bytes: LDS keeps its accesses in order)
        uint8_t *const dst_base = e.dst + m0 * e.dst_pitch + n0 + wn * 128;
        const int c = lane & 7;
        const bool head_ok = head0 + c * 16 / EP_D < e.n_heads;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int r = k * 8 + (lane >> 3);
            const v4i w = *(const v4i *)(bytes + r * 128 + ((c ^ (r & 7)) << 4));
            if (wm * 64 + r < rows_here && head_ok) *(v4i *)(dst_base + ((uint32_t)(wm * 64 + r) * (uint32_t)e.dst_pitch + (uint32_t)c * 16u)) = w;
        }
    } else if constexpr (MODE == TSATTN_MM_ADD_SCALED) {
        // state += sum * scale: the 32 old values of a block of rows are requested together, then updated and stored
        // (element by element every store would have to be waited for before the next load, which it might overlap;
        // with one workgroup per compute unit nothing else runs under those waits)
#pragma clang fp contract(off)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float old[2][16];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int64_t n = n0 + wn * 64 + j * 32 + li;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int64_t m = m0 + wm * 128 + i * 32 + 8 * (r / 4) + 4 * g + (r & 3);
                    old[j][r] = (n < p.n && m < p.m) ? ((const float *)p.out)[m * p.out_pitch + n] : 0.0f;
                }
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int64_t n = n0 + wn * 64 + j * 32 + li;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int64_t m = m0 + wm * 128 + i * 32 + 8 * (r / 4) + 4 * g + (r & 3);
                    if (n < p.n && m < p.m) ((float *)p.out)[m * p.out_pitch + n] = old[j][r] + (float)acc[i][j][r] * p.scale;
                }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int64_t n = n0 + wn * 64 + j * 32 + li;
                if (n >= p.n) continue;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int64_t m = m0 + wm * 128 + i * 32 + 8 * (r / 4) + 4 * g + (r & 3);
                    if (m < p.m) store_out<MODE>(p, m, n, acc[i][j][r]);
                }
            }
    }
}

// sums the planes of the workspace and applies the epilogue: one thread per output element
template <int MODE>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmParams p, const int32_t *ws, int n_split)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= p.m * p.n) return;
    int sum = 0;
    for (int s = 0; s < n_split; ++s) sum += ws[s * p.split_stride + i];
    store_out<MODE>(p, i / p.n, i % p.n, sum);
}

// Which kernel, by about what each would take (microseconds): rounds of one workgroup per compute unit, each a fixed part --
// launch, first stages, the last steps -- and a part per 128 bytes of K, both as measured on products of 40 to 8192 rows, 768 to
// 8192 columns, K of 768 to 8192; with every compute unit at work the wide tiles' rounds take up to 1.6 times as long (the
// clock), the others' 1.1 times.  Examples: 2048 x 8192 x 2048 wide 37, 128 rows 51, 64 rows 69; 550 x 8192 x 2048: 25, 25, 32;
// 400 x 2048 x 2048: 24, 13, 10; 100 x 2048 x 8192 with the normalisation: 65, 32, 21, few-row kernel and its launch 20.
enum class Tiles { WIDE, ROWS128, ROWS64, FEW };

double rounds_us(int64_t tiles, double fixed, double per_stage, double full, int64_t k)
{
    const double rounds = (double)((tiles + 255) / 256);
    return rounds * (fixed + per_stage * ((double)k / 128)) * (1.0 + full * (double)tiles / (256.0 * rounds));
}

FewParams few_params(const GemmParams &p);

// Parts of K through the caller's workspace and a second launch that adds them up, for results that cannot be left as planes: how
// many (1: no room, or K cannot be cut) and about how many nanoseconds.  Rows and K beyond what a compute unit's LDS holds go in
// parts (matrices from memory): 8192 -> 2048 under 32, 64 and 128 rows 12.0, 15.7 and 21.1 us, 16.3, 27.5 and 30.3 in one launch by
// the better kernel; 3072 -> 768 under 64 rows 10.2 and 15.0.  Short products lose to the second launch: 1024 -> 256 under 8 rows
// 7.2 and 5.4, 2048 -> 2048 under 32 rows 8.6 and 7.2.
int workspace_parts(const GemmParams &p, double *ns)
{
    const int64_t room = p.workspace ? p.workspace_bytes / (p.m * p.n * 4) : 0;
    int parts = 1;
    if (room >= 2 && p.m <= FEW_ROWS) *ns = few_split(few_params(p), room >= 16 ? 16 : room >= 8 ? 8 : room >= 4 ? 4 : 2, &parts);
    return parts;
}

// (*parts: of K through the workspace, 1 = one launch)
Tiles choose_tiles(const GemmParams &p, bool wide_ok, bool normalised, int *parts)
{
    *parts = 1;
    const int64_t n256 = (p.n + 255) / 256, n128 = (p.n + 127) / 128;
    // no tiles faster than memory brings them the matrix (32 x 50257 x 2048: 26.5 us, 3.9 TB/s)
    const double memory = 4.0 + (double)p.n * p.k * 1e-6 / 4.6;
    double best = std::max(memory, rounds_us(n128 * ((p.m + 127) / 128), 6.7, 0.40, 0.1, p.k));
    Tiles tiles = Tiles::ROWS128;
    const auto consider = [&](Tiles t, double us) {
        if (us < best) { best = us; tiles = t; }
    };
    consider(Tiles::ROWS64, std::max(memory, rounds_us(n128 * ((p.m + 63) / 64), 5.8, 0.25, 0.1, p.k)));
    if (wide_ok) consider(Tiles::WIDE, rounds_us(n256 * ((p.m + 255) / 256), 10.0, 0.87, 0.6, p.k));
    if (p.m <= FEW_ROWS) {
        consider(Tiles::FEW, few_ns(few_params(p), p.mode == TSATTN_MM_I32_PLANES ? 16 : 1) * 1e-3 + (normalised ? 5.0 : 0.0));
        if (p.mode != TSATTN_MM_I32_PLANES) {
            double ns = 0.0;
            *parts = workspace_parts(p, &ns);
            if (*parts > 1 && ns * 1e-3 < best) tiles = Tiles::FEW;
            else *parts = 1;
        }
    }
    return tiles;
}

template <int MODE>
hipError_t launch_tiles(const GemmParams &p, Tiles tiles, int ep_d, hipStream_t st)
{
    if (tiles != Tiles::WIDE) {
        GemmParams q = p;
        q.mode = MODE;
        return launch_gemm_mid(q, tiles == Tiles::ROWS64 ? 64 : 128, ep_d, st);
    }
    const dim3 grid((unsigned)(((p.m + GW_BM - 1) / GW_BM) * ((p.n + GW_BN - 1) / GW_BN)));
    if (ep_d == 128) hipLaunchKernelGGL((gemm_wide_kernel<TSATTN_MM_I32, 128>), grid, dim3(GW_THREADS), GW_LDS_BYTES, st, p);
    else if (ep_d == 64) hipLaunchKernelGGL((gemm_wide_kernel<TSATTN_MM_I32, 64>), grid, dim3(GW_THREADS), GW_LDS_BYTES, st, p);
    else hipLaunchKernelGGL((gemm_wide_kernel<MODE, 0>), grid, dim3(GW_THREADS), GW_LDS_BYTES, st, p);
    return hipGetLastError();
}

FewParams few_params(const GemmParams &p)
{
    FewParams f = {};
    f.w = p.w; f.w_pitch = p.w_pitch; f.m = p.m; f.n = p.n; f.k = p.k; f.a = p.a; f.a_pitch = p.a_pitch;
    f.mode = p.mode == TSATTN_MM_I32_PLANES ? TSATTN_MM_I32 : p.mode;
    f.scale = p.scale; f.out = p.out; f.out_pitch = p.out_pitch; f.parts = 1;
    return f;
}

} // namespace

// Once per device, before the first product: the wide-tile kernels use more LDS than a launch may ask for by default.
hipError_t prepare_matmul_i8()
{
    const struct {
        const void *kernel;
        int lds;
    } kernels[] = {{(const void *)gemm_wide_kernel<TSATTN_MM_I32, 0>, GW_LDS_BYTES},
                   {(const void *)gemm_wide_kernel<TSATTN_MM_F32, 0>, GW_LDS_BYTES},
                   {(const void *)gemm_wide_kernel<TSATTN_MM_ADD_SCALED, 0>, GW_LDS_BYTES},
                   {(const void *)gemm_wide_kernel<TSATTN_MM_I32, 64>, GW_LDS_BYTES},
                   {(const void *)gemm_wide_kernel<TSATTN_MM_I32, 128>, GW_LDS_BYTES}};
    for (const auto &k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, k.lds);
        if (e != hipSuccess) return e;
    }
    const hipError_t e = prepare_gemm_few();
    return e != hipSuccess ? e : prepare_gemm_mid();
}

hipError_t launch_matmul_i8(const GemmParams &p, hipStream_t st, int *planes_out)
{
    if (p.m <= 0 || p.n <= 0) {
        if (planes_out) *planes_out = 1;
        return hipSuccess;
    }
    if (p.mode == TSATTN_MM_I32_PLANES) {
        GemmParams q = p;
        bool fused = false, offsets_fit = true;
        if (p.ep_head_dim) {
            // the producer on the result: in the product's own kernel, or after it
            q.ep.src = p.out; q.ep.src_pitch = p.n; q.ep.n_rows = p.m; q.ep.n_heads = (int)(p.n / p.ep_head_dim);
            q.ep.src_planes = 1; q.ep.src_plane_stride = p.m * p.n;
            // (the wide kernel's epilogue addresses a tile's rows with 32-bit offsets)
            offsets_fit = q.ep.dst_pitch < (1 << 23) && (!q.ep.resid || q.ep.resid_pitch < (1 << 21)) &&
                          (!q.ep.pos || q.ep.rope_len * p.ep_head_dim * 4 < ((int64_t)1 << 31));
            // one operand besides the product: the old state, or cos and sin; wider groups than a head have a launch of their own
            fused = p.ep_dst_dtype == TSATTN_I8 && !(q.ep.resid && q.ep.pos) && (p.ep_head_dim == 64 || p.ep_head_dim == 128);
        }
        int parts;
        const Tiles tiles = choose_tiles(p, offsets_fit || !fused, p.ep_head_dim != 0, &parts);
        *planes_out = 1;
        if (tiles != Tiles::FEW && fused) return launch_tiles<TSATTN_MM_I32>(q, tiles, p.ep_head_dim, st);
        hipError_t e;
        if (tiles == Tiles::FEW) {
            // the parts' sums straight into the caller's planes (with few rows 16 * m * n ints of room by contract)
            FewParams f = few_params(p);
            f.parts = few_parts(f, 16);
            f.out_stride = p.m * p.n;
            *planes_out = q.ep.src_planes = f.parts;
            e = launch_gemm_few(f, st);
        } else {
            e = launch_tiles<TSATTN_MM_I32>(q, tiles, 0, st);
        }
        if (e != hipSuccess || !p.ep_head_dim) return e;
        return launch_rope_normalize(q.ep, p.ep_dst_dtype, p.ep_head_dim, true, st);
    }
    int parts;
    const Tiles tiles = choose_tiles(p, true, false, &parts);
    if (tiles == Tiles::FEW) {
        FewParams f = few_params(p);
        if (parts == 1) return launch_gemm_few(f, st);
        f.mode = TSATTN_MM_I32;
        f.parts = parts;
        f.out = p.workspace; f.out_pitch = p.n; f.out_stride = p.m * p.n;
        const hipError_t e = launch_gemm_few(f, st);
        if (e != hipSuccess) return e;
        GemmParams r = p;
        r.split_stride = p.m * p.n;
        const dim3 grid((unsigned)((p.m * p.n + 255) / 256));
        if (p.mode == TSATTN_MM_I32) hipLaunchKernelGGL((gemm_reduce_kernel<TSATTN_MM_I32>), grid, dim3(256), 0, st, r, (const int32_t *)p.workspace, f.parts);
        else if (p.mode == TSATTN_MM_F32) hipLaunchKernelGGL((gemm_reduce_kernel<TSATTN_MM_F32>), grid, dim3(256), 0, st, r, (const int32_t *)p.workspace, f.parts);
        else hipLaunchKernelGGL((gemm_reduce_kernel<TSATTN_MM_ADD_SCALED>), grid, dim3(256), 0, st, r, (const int32_t *)p.workspace, f.parts);
        return hipGetLastError();
    }
    if (p.mode == TSATTN_MM_I32) return launch_tiles<TSATTN_MM_I32>(p, tiles, 0, st);
    if (p.mode == TSATTN_MM_F32) return launch_tiles<TSATTN_MM_F32>(p, tiles, 0, st);
    if (p.mode == TSATTN_MM_ADD_SCALED) return launch_tiles<TSATTN_MM_ADD_SCALED>(p, tiles, 0, st);
    return hipErrorInvalidValue;
}

} // namespace tsattn
