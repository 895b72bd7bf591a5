// Producer of the attention operands: RoPE, per-head RMS normalisation and 8-bit conversion of a projection
// result, with the per-(row, head) scale the attention kernels consume.  Follows the reference's CPU inference
// (ApplyRope + NormalizeState, gpt/train/cpu_infer.cpp:486-499, :358-391; gpt/att/rope.cpp:28-46) operation by
// operation: the same float products, the sum of squares taken in index order, no fused multiply-adds, so the
// bytes and scales are identical to a CPU evaluation in that order.
//
// One wave takes 64 / (D / 8) pairs: a lane holds eight values (four couples x, x + 32), squares go through the wave's LDS to
// the lane that adds its pair's up in index order -- additions only, one instruction per value -- and the multiplier comes back
// through a lane exchange: no barrier, no second pass over the values.  Bound by memory for large launches (65536 x 16 x 128 f32 ->
// int8, no rotation: 124 us, 5.7 TB/s, as with workgroups of 32 pairs, 256 threads and three barriers), by its chain of waits for small
// ones (531 x 16 x 128: 4.8 against 6.3 us; 32 x 16, two planes and the residual update: 4.5 against 5.6 us).
#include <math.h>

#include "common.hpp"
#include "kernels.hpp"

namespace tsattn {

// every float operation below is meant as written: no fused multiply-adds
#pragma clang fp contract(off)

// ROPE: with positions (a kernel of its own: without, their registers would cost the others 2 to 10 % of a large launch)
template <int D, int DST, bool SRC_I32, bool ROPE>
__global__ __launch_bounds__(WAVE) void rope_normalize_kernel(ProduceParams p)
{
    constexpr int LPP = D / 8, PAIRS = WAVE / LPP; // lanes per pair, pairs per wave
    constexpr int PITCH = D + 4;
    __shared__ __attribute__((aligned(16))) float squares[PAIRS * PITCH];
    const int lane = threadIdx.x;
    const int pr = lane / LPP, c = lane % LPP;
    const uint32_t pair = blockIdx.x * PAIRS + pr, n_pairs = (uint32_t)p.n_rows * (uint32_t)p.n_heads;
    const bool mine = pr < PAIRS && pair < n_pairs;
    const uint32_t pc = mine ? pair : n_pairs - 1;
    const int64_t row = pc / (uint32_t)p.n_heads;
    const int head = (int)(pc % (uint32_t)p.n_heads);
    const int x0 = (c / 8) * 64 + (c % 8) * 4;
    v4f v0, v1;
    v4f u0, u1, cs, sn;
    const int64_t e = row * p.src_pitch + (int64_t)head * D + x0;
    float *const resid = p.resid + row * p.resid_pitch + (int64_t)head * D + x0;
    // The position is asked for first and the table's row as soon as it is there, behind the requests of the values: what is asked for
    // first arrives first, and one wait covers both (33000 x 12 x 64, one int32 plane: 35.7 us with the position behind the values).
    int t = ROPE ? p.pos[row] : 0;
    const auto ask_rope = [&]() __attribute__((always_inline)) {
        if (!ROPE) return;
        t = t < 0 ? 0 : (t >= p.rope_len ? (int)p.rope_len - 1 : t);
        const float *const rr = p.rope + (int64_t)t * D + x0;
        cs = *(const v4f *)rr;
        sn = *(const v4f *)(rr + 32);
    };
    if (SRC_I32) {
        constexpr int PL = 4; // planes asked for together (those that are not there: the last one again)
        const int32_t *const src = (const int32_t *)p.src + e;
        v4i a = v4i{0, 0, 0, 0}, b = v4i{0, 0, 0, 0};
        if (p.src_planes == 1) {
            a = *(const v4i *)src;
            b = *(const v4i *)(src + 32);
            if (p.resid) {
                u0 = *(const v4f *)resid;
                u1 = *(const v4f *)(resid + 32);
            }
            ask_rope();
        }
        for (int p0 = 0; p0 < p.src_planes && p.src_planes > 1; p0 += PL) {
            v4i qa[PL], qb[PL];
#pragma unroll
            for (int i = 0; i < PL; ++i) {
                const int32_t *const q = src + (p0 + i < p.src_planes ? p0 + i : p.src_planes - 1) * p.src_plane_stride;
                qa[i] = *(const v4i *)q;
                qb[i] = *(const v4i *)(q + 32);
            }
            if (p0 == 0 && p.resid) {
                u0 = *(const v4f *)resid;
                u1 = *(const v4f *)(resid + 32);
            }
            if (p0 == 0) ask_rope();
#pragma unroll
            for (int i = 0; i < PL; ++i)
                if (p0 + i < p.src_planes) { a += qa[i]; b += qb[i]; }
        }
        v0 = v4f{(float)a.x, (float)a.y, (float)a.z, (float)a.w};
        v1 = v4f{(float)b.x, (float)b.y, (float)b.z, (float)b.w};
    } else {
        v0 = *(const v4f *)((const float *)p.src + e);
        v1 = *(const v4f *)((const float *)p.src + e + 32);
        if (p.resid) {
            u0 = *(const v4f *)resid;
            u1 = *(const v4f *)(resid + 32);
        }
        ask_rope();
    }
    if (p.resid) {
        v0 = u0 + v0 * p.resid_scale;
        v1 = u1 + v1 * p.resid_scale;
        if (mine) {
            *(v4f *)resid = v0;
            *(v4f *)(resid + 32) = v1;
        }
    }
    if (ROPE) {
        const bool turn = head < p.rope_heads; // (the other heads turn by the identity)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float cos_value = turn ? cs[i] : 1.0f;
            const float sin_value = turn ? sn[i] * p.rotate_dir : 0.0f;
            const float r0 = v0[i] * cos_value - v1[i] * sin_value;
            const float r1 = v0[i] * sin_value + v1[i] * cos_value;
            v0[i] = r0;
            v1[i] = r1;
        }
    }
    if (pr < PAIRS) {
        *(v4f *)(squares + pr * PITCH + x0) = v0 * v0;
        *(v4f *)(squares + pr * PITCH + x0 + 32) = v1 * v1;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (one wave: its LDS accesses are in order)
    float mult = 0.0f;
    if (lane < PAIRS) {
        const float *const v = squares + lane * PITCH;
        float sum2 = 0.0f;
#pragma unroll 4
        for (int x = 0; x < D; x += 32) {
            v4f q[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) q[i] = *(const v4f *)(v + x + 4 * i);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sum2 = sum2 + q[i].x;
                sum2 = sum2 + q[i].y;
                sum2 = sum2 + q[i].z;
                sum2 = sum2 + q[i].w;
            }
        }
        float discr = 0.0f;
        if (sum2 != 0.0f) {
            // the single-precision square root instruction is one ulp off now and then; the double-precision routine
            // is exact to well below a float ulp, and rounding its result to float gives the correctly rounded root
            discr = (float)sqrt((double)(sum2 / (float)D)) * p.vec_scale;
            mult = 1.0f / discr;
        }
        const uint32_t q = blockIdx.x * PAIRS + lane;
        if (p.scale && q < n_pairs) {
            const int sh = (int)(q % (uint32_t)p.n_heads) - p.scale_head_begin;
            if (sh >= 0 && sh < p.scale_head_count) p.scale[sh * p.scale_pitch + (int64_t)(q / (uint32_t)p.n_heads) * p.scale_row_stride] = discr * p.scale_mult;
        }
    }
    mult = __shfl(mult, pr < PAIRS ? pr : 0, WAVE);
    if (!mine) return;
    uint32_t w0, w1;
    if (DST == TSATTN_I8) {
        const float low = p.relu ? 0.0f : -127.0f;
        w0 = pack_i8x4(v0.x * mult, v0.y * mult, v0.z * mult, v0.w * mult, low);
        w1 = pack_i8x4(v1.x * mult, v1.y * mult, v1.z * mult, v1.w * mult, low);
    } else {
        w0 = w1 = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) { // (a head of zeros is zero bytes whatever the signs of its zeros)
            w0 |= (mult == 0.0f ? 0u : (uint32_t)float_to_e4m3(v0[i] * mult)) << (8 * i);
            w1 |= (mult == 0.0f ? 0u : (uint32_t)float_to_e4m3(v1[i] * mult)) << (8 * i);
        }
    }
    uint8_t *const dst = p.dst + row * p.dst_pitch + (int64_t)head * D + x0;
    *(uint32_t *)dst = w0;
    *(uint32_t *)(dst + 32) = w1;
}

hipError_t launch_rope_normalize(const ProduceParams &p, int dst_dtype, int head_dim, bool src_i32, hipStream_t st)
{
    const int64_t n_pairs = p.n_rows * p.n_heads;
    if (n_pairs == 0) return hipSuccess;
    if (p.n_rows > 0xffffffffll / p.n_heads) return hipErrorInvalidValue; // (pairs are counted in 32 bits: 1 TB of values)
    const int per_wave = WAVE / (head_dim / 8); // (one group of 384 or 512 values)
    dim3 grid((unsigned)((n_pairs + per_wave - 1) / per_wave)), block(WAVE);
#define TSATTN_PR(D_, DST_, I32_, ROPE_)                                                             \
    if (head_dim == D_ && dst_dtype == DST_ && src_i32 == I32_ && (p.pos != nullptr) == ROPE_) {          \
        hipLaunchKernelGGL((rope_normalize_kernel<D_, DST_, I32_, ROPE_>), grid, block, 0, st, p);        \
        return hipGetLastError();                                                                         \
    }
#define TSATTN_PR_HEAD(D_, DST_) \
    TSATTN_PR(D_, DST_, false, false) TSATTN_PR(D_, DST_, false, true) TSATTN_PR(D_, DST_, true, false) TSATTN_PR(D_, DST_, true, true)
#define TSATTN_PR_WIDE(D_) TSATTN_PR(D_, TSATTN_I8, false, false) TSATTN_PR(D_, TSATTN_I8, true, false)
    TSATTN_PR_HEAD(64, TSATTN_I8)
    TSATTN_PR_HEAD(64, TSATTN_E4M3)
    TSATTN_PR_HEAD(128, TSATTN_I8)
    TSATTN_PR_HEAD(128, TSATTN_E4M3)
    TSATTN_PR_WIDE(256)
    TSATTN_PR_WIDE(384)
    TSATTN_PR_WIDE(512)
#undef TSATTN_PR_WIDE
#undef TSATTN_PR_HEAD
#undef TSATTN_PR
    return hipErrorInvalidValue;
}

// KVProduct, gpt/train/cpu_infer.cpp:320-337 (GPU form compute/gpt_combiner.cuh:13-37): the step after attention,
// kv[head][blk][z] = int8(k[head][z ^ blk] * value[head][z] * mult) for blk < 4.  One thread per 16 consecutive z of a
// (row, head): z ^ blk stays inside an aligned group of four, so a thread needs only its own 16 key bytes.
template <bool VAL_F16>
__global__ __launch_bounds__(256) void kv_product_kernel(KvProductParams p)
{
    const int chunks = p.head_dim / 16;
    const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t total = p.n_rows * p.n_heads * chunks;
    if (id >= total) return;
    const int c = (int)(id % chunks);
    const int head = (int)((id / chunks) % p.n_heads);
    const int64_t row = id / ((int64_t)chunks * p.n_heads);
    const int64_t e = (int64_t)head * p.head_dim + c * 16;
    const v4i kw = *(const v4i *)(p.k + row * p.k_pitch + e);
    const int kws[4] = {kw.x, kw.y, kw.z, kw.w};
    float key[16], val[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) key[i] = (float)(int8_t)((kws[i / 4] >> (8 * (i % 4))) & 0xff);
    if (VAL_F16) {
        const v8h a = *(const v8h *)((const _Float16 *)p.val + row * p.val_pitch + e);
        const v8h b = *(const v8h *)((const _Float16 *)p.val + row * p.val_pitch + e + 8);
#pragma unroll
        for (int i = 0; i < 8; ++i) { val[i] = (float)a[i]; val[8 + i] = (float)b[i]; }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const v4f a = *(const v4f *)((const float *)p.val + row * p.val_pitch + e + 4 * i);
            val[4 * i] = a.x; val[4 * i + 1] = a.y; val[4 * i + 2] = a.z; val[4 * i + 3] = a.w;
        }
    }
#pragma unroll
    for (int blk = 0; blk < 4; ++blk) {
        if (blk >= p.rep) break;
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (int z = 0; z < 16; ++z) {
            const float y = (key[z ^ blk] * val[z]) * p.mult;
            w[z / 4] |= (uint32_t)(uint8_t)float_to_i8(y) << (8 * (z % 4));
        }
        *(v4i *)(p.kv + row * p.kv_pitch + ((int64_t)head * p.rep + blk) * p.head_dim + c * 16) = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
}

hipError_t launch_kv_product(const KvProductParams &p, bool val_f16, hipStream_t st)
{
    const int64_t total = p.n_rows * p.n_heads * (p.head_dim / 16);
    if (total == 0) return hipSuccess;
    dim3 grid((unsigned)((total + 255) / 256)), block(256);
    if (val_f16) hipLaunchKernelGGL((kv_product_kernel<true>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((kv_product_kernel<false>), grid, block, 0, st, p);
    return hipGetLastError();
}

// FillRopeBuf, gpt/att/rope.cpp:4-24 (host): table[t][base + k] = cos(t f), table[t][base + k + 32] = sin(t f),
// f = theta^-(2 (base/2 + k) / width), theta = 500000.  The float/double mix follows the reference's C++ overloads.
void fill_rope_table(int width, int64_t max_len, float *table)
{
    const float theta = 500000;
    for (int64_t t = 0; t < max_len; ++t) {
        for (int base = 0; base < width; base += 64) {
            for (int k = 0; k < 32; ++k) {
                const float freq = (float)exp((double)(-logf(theta)) * ((base / 2 + k) * 2. / width));
                const float angle = t * freq;
                table[t * width + base + k] = cosf(angle);
                table[t * width + base + k + 32] = sinf(angle);
            }
        }
    }
}

} // namespace tsattn
