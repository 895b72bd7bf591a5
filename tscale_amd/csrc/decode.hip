// Single-token attention over a planar int8 / e4m3 KV cache: bandwidth-bound split-KV kernel plus
// the cross-split merge.
//
// Work decomposition.  grid = (n_splits, n_heads, n_seqs), four or sixteen waves (decode_form in decode_splits.h).  A (sequence, head) pair owns
// two contiguous planes, K[L][d] and V[L][d]; a split owns a contiguous run of cache rows.  Inside
// a wave, d/16 neighbouring lanes share one cache row and each lane reads 16 B of it, so one wave
// load instruction covers 1 KiB of consecutive memory (8 rows at d=128, 16 rows at d=64).  Each lane
// group keeps its own online-softmax state (running max, sum, 16 value accumulators) across all the
// rows it visits; states are merged only once, at the end: across lane groups by lane exchanges,
// across the waves through LDS, across splits by merge_kernel.
//
// Semantics follow ComputeValLookup of gpt/train/cpu_infer.cpp:413-460: keys cur-1 ... cur-min(cur,W)
// (cur itself when W == 0), a leading logit 0 of value zero (:444), logit =
// dot * key_scale * attDotScale * q_scale - slope * (cur - to) (:448), value weight times the value
// scale (:454).  The running max starts at 0 in every split, which is what the zero logit makes it
// in the reference anyway, so no split ever needs a -inf state.
#include "common.hpp"
#include "kernels.hpp"

namespace tsattn {

template <int DTYPE>
struct QFrag;

template <>
struct QFrag<TSATTN_I8> {
    int w[4];
    __device__ void set(const uint8_t *b)
    {
        const int *p = (const int *)b;
        w[0] = p[0]; w[1] = p[1]; w[2] = p[2]; w[3] = p[3];
    }
    // exact int32 dot product of 16 bytes of the row with this lane's slice of q
    __device__ float dot_partial_as_bits(v4i kv) const
    {
        int acc = 0;
        acc = __builtin_amdgcn_sdot4(kv.x, w[0], acc, false);
        acc = __builtin_amdgcn_sdot4(kv.y, w[1], acc, false);
        acc = __builtin_amdgcn_sdot4(kv.z, w[2], acc, false);
        acc = __builtin_amdgcn_sdot4(kv.w, w[3], acc, false);
        return __int_as_float(acc);
    }
};

template <>
struct QFrag<TSATTN_E4M3> {
    float f[16];
    __device__ void set(const uint8_t *b)
    {
        const int *p = (const int *)b;
        for (int i = 0; i < 4; ++i) {
            v2f lo = e4m3x2_to_float(p[i], false);
            v2f hi = e4m3x2_to_float(p[i], true);
            f[4 * i + 0] = lo.x; f[4 * i + 1] = lo.y; f[4 * i + 2] = hi.x; f[4 * i + 3] = hi.y;
        }
    }
    __device__ float dot_partial_as_bits(v4i kv) const
    {
        float acc = 0;
        int kw[4] = {kv.x, kv.y, kv.z, kv.w};
        for (int i = 0; i < 4; ++i) {
            v2f lo = e4m3x2_to_float(kw[i], false);
            v2f hi = e4m3x2_to_float(kw[i], true);
            acc = fmaf(lo.x, f[4 * i + 0], acc);
            acc = fmaf(lo.y, f[4 * i + 1], acc);
            acc = fmaf(hi.x, f[4 * i + 2], acc);
            acc = fmaf(hi.y, f[4 * i + 3], acc);
        }
        return acc;
    }
};

// sum over the LPK lanes that share a cache row; every one of them ends with the total
template <int DTYPE, int LPK>
__device__ inline float group_sum_bits(float bits)
{
    if (DTYPE == TSATTN_I8) {
        int a = __float_as_int(bits);
        a += dpp_xor1(a);
        a += dpp_xor2(a);
        if (LPK == 8) {
            a += dpp_half_mirror(a);
        }
        return __int_as_float(a);
    } else {
        float a = bits;
        a += __int_as_float(dpp_xor1(__float_as_int(a)));
        a += __int_as_float(dpp_xor2(__float_as_int(a)));
        if (LPK == 8) {
            a += __int_as_float(dpp_half_mirror(__float_as_int(a)));
        }
        return a;
    }
}

template <int DTYPE>
__device__ inline void accumulate_values(float w, v4i vv, float *acc)
{
    int vw[4] = {vv.x, vv.y, vv.z, vv.w};
    if (DTYPE == TSATTN_I8) {
        for (int i = 0; i < 4; ++i) {
            int x = vw[i];
            acc[4 * i + 0] = fmaf(w, (float)(int8_t)(x & 0xff), acc[4 * i + 0]);
            acc[4 * i + 1] = fmaf(w, (float)(int8_t)((x >> 8) & 0xff), acc[4 * i + 1]);
            acc[4 * i + 2] = fmaf(w, (float)(int8_t)((x >> 16) & 0xff), acc[4 * i + 2]);
            acc[4 * i + 3] = fmaf(w, (float)(x >> 24), acc[4 * i + 3]);
        }
    } else {
        for (int i = 0; i < 4; ++i) {
            v2f lo = e4m3x2_to_float(vw[i], false);
            v2f hi = e4m3x2_to_float(vw[i], true);
            acc[4 * i + 0] = fmaf(w, lo.x, acc[4 * i + 0]);
            acc[4 * i + 1] = fmaf(w, lo.y, acc[4 * i + 1]);
            acc[4 * i + 2] = fmaf(w, hi.x, acc[4 * i + 2]);
            acc[4 * i + 3] = fmaf(w, hi.y, acc[4 * i + 3]);
        }
    }
}

// KVProduct of a finished output element (gpt/train/cpu_infer.cpp:320-337): kv[head][blk][x] = int8((k[head][x ^ blk] *
// value) * mult) for blk < rep; x ^ blk stays inside x's aligned group of four key bytes.  The same arithmetic as
// kv_product_kernel on the stored output.
template <int D>
__device__ inline void kv_product_store(const uint8_t *kv_k, int64_t kv_k_pitch, uint8_t *kv_out, int64_t kv_out_pitch, int rep, float mult,
                                        int64_t seq, int head, int x, float value)
{
    const uint32_t kw = *(const uint32_t *)(kv_k + seq * kv_k_pitch + (int64_t)head * D + (x & ~3));
    for (int blk = 0; blk < rep; ++blk) {
        const float key = (float)(int8_t)((kw >> (8 * ((x ^ blk) & 3))) & 0xff);
        const float y = (key * value) * mult;
        kv_out[seq * kv_out_pitch + ((int64_t)head * rep + blk) * D + x] = (uint8_t)float_to_i8(y);
    }
}

// FRONT: what the launch before would have made -- q, the new key and value rows, the key of KVProduct, RoPE and
// normalisation included -- is made by the first wave of every workgroup from the projections' planes of its own head, while
// the other waves ask for their first cache rows (nothing is made twice but q by the splits of a head).  It saves a launch
// of 5.7 us for 1.5 us; the bytes are those of rope_normalize_kernel, the same float operations in the same order.
// GENERAL: any stride of the cache's tokens, and the raw dot products on request; the others address a step's rows with 24-bit
// products from a scalar base (the launcher checks the stride): two 64-bit products per row were a third of the loop's instructions.
template <int DTYPE, int D, bool QBF16, bool GENERAL, bool FRONT, int WAVES, int DEC_U>
__device__ __forceinline__ void decode_split(const DecodeParams &p)
{
    constexpr int DEC_THREADS = WAVES * WAVE;
    constexpr int LPK = D / 16;      // lanes per cache row
    constexpr int KPL = WAVE / LPK;  // rows per wave load
    constexpr int ROWS_PER_STEP = DEC_U * KPL;

    const int split = blockIdx.x;
    const int head = blockIdx.y;
    const int seq = blockIdx.z;
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int c = lane % LPK;        // which 16-byte slice of the row
    const int g = lane / LPK;        // which row of a wave load

    __shared__ float sm_m[WAVES];
    __shared__ float sm_l[WAVES];
    __shared__ float sm_acc[WAVES][D];
    __shared__ __attribute__((aligned(16))) float f_square[FRONT ? 4 * (D + 4) : 4];
    __shared__ __attribute__((aligned(16))) uint8_t f_row[FRONT ? 4 * D : 16]; // q, new key, key of KVProduct, new value
    __shared__ float f_key_scale;

    ResidUpdate update;
    v4i fa[FRONT ? 4 : 1], fb[FRONT ? 4 : 1];
    v4f f_cos, f_sin;
    const int f_part = lane / (D / 8), f_x = ((lane % (D / 8)) / 8) * 64 + (lane % 8) * 4; // values f_x.. and f_x + 32.. of a row
    const bool f_mine = FRONT && wave == 0 && lane < D / 2;
    if constexpr (FRONT) {
        if (f_mine) {
            const int32_t *const src = p.front.src + ((int64_t)seq * 4 + f_part) * p.n_heads * D + head * D + f_x;
#pragma unroll
            for (int i = 0; i < 4; ++i) { // (planes that are not there: the last one again)
                const int32_t *const q = src + (i < p.front.planes ? i : p.front.planes - 1) * p.front.src_stride;
                fa[i] = *(const v4i *)q;
                fb[i] = *(const v4i *)(q + 32);
            }
            int t = p.front.pos[seq];
            t = t < 0 ? 0 : (t >= p.front.rope_len ? (int)p.front.rope_len - 1 : t);
            const float *const rr = p.front.rope + (int64_t)t * D + f_x;
            f_cos = *(const v4f *)rr;
            f_sin = *(const v4f *)(rr + 32);
        } else if (wave != 0) {
            const int wg = (seq * p.n_heads + head) * p.n_splits + split;
            update.request(p.front.upd, wg * (DEC_THREADS - WAVE) + tid - WAVE, (int)(gridDim.x * gridDim.y * gridDim.z) * (DEC_THREADS - WAVE));
        }
    }

    // ---- key range of this block --------------------------------------------------------------
    // With a fused append the cache holds cache_len rows and the new token's row is being added as row cache_len
    // by the first split's workgroup of each head (a full cache drops it, as the separate append does).
    int cur = p.cache_len[seq] - 1;
    const bool append = FRONT || p.k_new != nullptr;
    const bool new_row = append && cur + 1 < p.max_len;
    if (new_row) {
        cur += 1;
        if (!FRONT && split == 0 && tid < 2 * LPK) {
            const int pl = tid / LPK, ch = tid % LPK; // plane (K or V), 16-byte chunk
            const int64_t src = (int64_t)seq * p.new_pitch + head * D + ch * 16;
            const int64_t dst = (int64_t)seq * p.seq_stride + (int64_t)head * p.head_stride + (int64_t)cur * p.tok_stride + ch * 16;
            if (pl == 0) *(v4i *)(const_cast<uint8_t *>(p.k) + dst) = *(const v4i *)(p.k_new + src);
            else *(v4i *)(const_cast<uint8_t *>(p.v) + dst) = *(const v4i *)(p.v_new + src);
            if (ch == 0) {
                const int64_t sd = (int64_t)seq * p.s_seq_stride + (int64_t)head * p.s_head_stride + cur;
                if (pl == 0 && p.ks_new) const_cast<float *>(p.ks)[sd] = p.ks_new[seq * p.n_heads + head];
                if (pl == 1 && p.vs_new) const_cast<float *>(p.vs)[sd] = p.vs_new[seq * p.n_heads + head];
            }
        }
    }
    const bool direct = p.n_splits == 1; // no merge kernel follows: this workgroup writes the output
    // A single-split launch with a fused append has no merge kernel to count the new row either: every workgroup
    // of a sequence (one per head) reports when it is done with the old length, and the last to report adds one.
    // (The counter is back at zero when the launch ends; launches that share a handle must not overlap.)
    auto report_done = [&]() {
        if (tid == 0) {
            const int done = atomicAdd(&p.seq_done[seq], 1);
            if (done == p.n_heads - 1) {
                p.seq_done[seq] = 0;
                const int len = p.cache_len_rw[seq];
                if (len >= 0 && len < p.max_len) p.cache_len_rw[seq] = len + 1;
            }
        }
    };
    const bool count_row = direct && append;
    int lo, n;
    if (cur < 0) {
        lo = 0; n = 0;
    } else if (p.window == 0) {
        lo = cur; n = 1;
    } else {
        n = (int)((p.window < (int64_t)cur) ? p.window : (int64_t)cur);
        lo = cur - n;
    }
    int per = (n + p.n_splits - 1) / p.n_splits;
    per = ((per + KPL - 1) / KPL) * KPL;
    const int s0 = lo + split * per;
    int s1 = s0 + per;
    if (s1 > lo + n) s1 = lo + n;

    const int64_t part = ((int64_t)seq * p.n_heads + head) * p.n_splits + split;
    if (!FRONT && s0 >= s1) { // nothing to do: neutral partial (max 0, sum 0, zeros)
        if (direct) {
            if (tid < D) {
                p.out[((int64_t)seq * p.n_heads + head) * D + tid] = 0.0f;
                if (p.kv_out) kv_product_store<D>(p.kv_k, p.kv_k_pitch, p.kv_out, p.kv_out_pitch, p.kv_rep, p.kv_mult, seq, head, tid, 0.0f);
            }
            if (count_row) {
                __syncthreads(); // every thread has read the old length
                report_done();
            }
            return;
        }
        if (tid < D) p.part_acc[part * D + tid] = 0.0f;
        if (tid == 0) { p.part_ml[part * 2] = 0.0f; p.part_ml[part * 2 + 1] = 0.0f; }
        return;
    }

    const uint8_t *const kbase = p.k + (int64_t)seq * p.seq_stride + (int64_t)head * p.head_stride;
    const uint8_t *const vbase = p.v + (int64_t)seq * p.seq_stride + (int64_t)head * p.head_stride;
    const float *const ksb = p.ks ? p.ks + (int64_t)seq * p.s_seq_stride + (int64_t)head * p.s_head_stride : nullptr;
    const float *const vsb = p.vs ? p.vs + (int64_t)seq * p.s_seq_stride + (int64_t)head * p.s_head_stride : nullptr;
    v4i kreg[DEC_U], vreg[DEC_U];
    float ksr[DEC_U], vsr[DEC_U];
    auto request = [&](int base) __attribute__((always_inline)) {
        const uint8_t *const kb = kbase + (int64_t)base * p.tok_stride, *const vb = vbase + (int64_t)base * p.tok_stride;
        const int last = s1 - 1 - base; // clamp the address, mask the logit below
        uint32_t row[DEC_U];
        uint64_t at[DEC_U];
#pragma unroll
        for (int u = 0; u < DEC_U; ++u) {
            row[u] = (uint32_t)min(u * KPL + g, last);
            at[u] = GENERAL ? (uint64_t)row[u] * (uint64_t)p.tok_stride + c * 16 : __umul24(row[u], (uint32_t)p.tok_stride) + c * 16;
            kreg[u] = __builtin_nontemporal_load((const v4i *)(kb + at[u]));
            ksr[u] = ksb ? (ksb + base)[row[u]] : p.ks_const;
        }
#pragma unroll
        for (int u = 0; u < DEC_U; ++u) {
            vreg[u] = __builtin_nontemporal_load((const v4i *)(vb + at[u]));
            vsr[u] = vsb ? (vsb + base)[row[u]] : p.vs_const;
        }
    };
    int base = s0 + wave * ROWS_PER_STEP;
    if (FRONT && base < s1) request(base);

    // ---- query slice of this lane ----------------------------------------------------------------
    QFrag<DTYPE> qf;
    float qs;
    if constexpr (FRONT) {
#pragma clang fp contract(off)
        if (wave == 0) {
            float mult = 0.0f;
            v4f v0, v1;
            if (f_mine) {
                v4i a = fa[0], b = fb[0];
#pragma unroll
                for (int i = 1; i < 4; ++i)
                    if (i < p.front.planes) { a += fa[i]; b += fb[i]; }
                v0 = v4f{(float)a.x, (float)a.y, (float)a.z, (float)a.w};
                v1 = v4f{(float)b.x, (float)b.y, (float)b.z, (float)b.w};
                const bool turn = f_part < 2; // (k and v turn by the identity, as in the producer)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float cos_value = turn ? f_cos[i] : 1.0f, sin_value = turn ? f_sin[i] : 0.0f;
                    const float r0 = v0[i] * cos_value - v1[i] * sin_value;
                    const float r1 = v0[i] * sin_value + v1[i] * cos_value;
                    v0[i] = r0;
                    v1[i] = r1;
                }
                *(v4f *)(f_square + f_part * (D + 4) + f_x) = v4f{v0.x * v0.x, v0.y * v0.y, v0.z * v0.z, v0.w * v0.w};
                *(v4f *)(f_square + f_part * (D + 4) + f_x + 32) = v4f{v1.x * v1.x, v1.y * v1.y, v1.z * v1.z, v1.w * v1.w};
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (one wave: its LDS accesses are in order)
            float discr = 0.0f;
            if (lane < 4) { // squares added in index order
                const float *const v = f_square + lane * (D + 4);
                float sum2 = 0.0f;
#pragma unroll
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
                if (sum2 != 0.0f) {
                    discr = sqrt_rounded(sum2 / (float)D) * p.front.vec_scale;
                    mult = 1.0f / discr;
                }
                if (lane == 1) f_key_scale = discr * p.front.key_mult;
            }
            mult = __shfl(mult, f_part & 3, WAVE);
            if (f_mine) {
                *(uint32_t *)(f_row + f_part * D + f_x) = pack_i8x4(v0.x * mult, v0.y * mult, v0.z * mult, v0.w * mult, -127.0f);
                *(uint32_t *)(f_row + f_part * D + f_x + 32) = pack_i8x4(v1.x * mult, v1.y * mult, v1.z * mult, v1.w * mult, -127.0f);
            }
        } else {
            update.finish(p.front.upd);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // (cache rows stay on their way over the barrier)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        qf.set(f_row + c * 16);
        qs = p.q_scale_const;
        if (split == 0) {
            if (new_row && tid < 2 * LPK) {
                const int pl = tid / LPK, ch = tid % LPK; // plane (K or V), 16-byte chunk
                const int64_t dst = (int64_t)seq * p.seq_stride + (int64_t)head * p.head_stride + (int64_t)cur * p.tok_stride + ch * 16;
                *(v4i *)(const_cast<uint8_t *>(pl == 0 ? p.k : p.v) + dst) = *(const v4i *)(f_row + (pl == 0 ? 1 : 3) * D + ch * 16);
                if (ch == 0) {
                    const int64_t sd = (int64_t)seq * p.s_seq_stride + (int64_t)head * p.s_head_stride + cur;
                    if (pl == 0 && p.ks) const_cast<float *>(p.ks)[sd] = f_key_scale;
                    if (pl == 1 && p.vs) const_cast<float *>(p.vs)[sd] = p.front.vec_scale;
                }
            }
            if (!direct && tid < LPK) *(v4i *)(p.front.k_row + ((int64_t)seq * p.n_heads + head) * D + tid * 16) = *(const v4i *)(f_row + 2 * D + tid * 16);
        }
    } else {
        __attribute__((aligned(16))) uint8_t qb[16];
        if (QBF16) {
            const uint16_t *src = (const uint16_t *)(p.q + (int64_t)seq * p.q_pitch) + head * D + c * 16;
            float x[16];
            float amax = 0;
            for (int i = 0; i < 16; ++i) {
                x[i] = bf16_to_float(src[i]);
                amax = fmaxf(amax, fabsf(x[i]));
            }
            for (int o = 1; o < LPK; o <<= 1) {
                amax = fmaxf(amax, __shfl_xor(amax, o, WAVE));
            }
            // absmax rule of lib/cuda/cuda_matmul.cuh:237-249
            float discr = 0, mult = 0;
            if (amax > 0) {
                discr = (DTYPE == TSATTN_I8) ? amax / 127.0f : amax / 256.0f;
                mult = 1.0f / discr;
            }
            for (int i = 0; i < 16; ++i) {
                float y = x[i] * mult;
                qb[i] = (DTYPE == TSATTN_I8) ? (uint8_t)float_to_i8(y) : float_to_e4m3(y);
            }
            qs = discr;
        } else {
            const v4i *src = (const v4i *)(p.q + (int64_t)seq * p.q_pitch + head * D + c * 16);
            *(v4i *)qb = *src;
            qs = p.q_scale ? p.q_scale[seq * p.n_heads + head] : p.q_scale_const;
        }
        qf.set(qb);
    }

    const float scale = att_dot_scale(D) * qs;

    float m = 0.0f, l = 0.0f;
    float acc[16];
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;

    for (; base < s1; base += WAVES * ROWS_PER_STEP) {
        if constexpr (!FRONT) { // (with nothing to wait for but the query a second copy of the requests only makes the code longer: 4 % of a short launch)
            request(base);
            // Every request of the step before the first sum: left to itself the compiler moves the last value row's request
            // behind the waits for the keys, and where one workgroup per compute unit is all there is nothing hides that row's
            // latency (e4m3, width 128: 8 x 16 pairs of 1024 rows 13.2 us that way, 12.6 this way; 16 x 16 16.4 and 15.9; width 64,
            // 13 x 12 pairs of 1500 rows 11.6 and 11.2).  With two workgroups per unit it can be the other way round (int8,
            // width 128: 32 x 16 pairs of 512 rows 14.2 and 14.6 us, 24 x 16 of 2048 36.5 and 37.6), from three on they are equal.
            __builtin_amdgcn_sched_barrier(0);
        }
        float s[DEC_U];
        float m_new = m;
#pragma unroll
        for (int u = 0; u < DEC_U; ++u) {
            float bits = group_sum_bits<DTYPE, LPK>(qf.dot_partial_as_bits(kreg[u]));
            float accf = (DTYPE == TSATTN_I8) ? (float)__float_as_int(bits) : bits;
            const int row = base + u * KPL + g;
            if (GENERAL) {
                if (p.dbg && c == 0 && row < s1) {
                    ((float *)p.dbg)[((int64_t)seq * p.n_heads + head) * p.dbg_pitch + row] = bits;
                }
            }
            float dp = accf * ksr[u] * scale - p.slope * (float)(cur - row);
            s[u] = row < s1 ? dp : -INFINITY;
            m_new = fmaxf(m_new, s[u]);
        }
        float alpha = fast_exp2(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] *= alpha;
#pragma unroll
        for (int u = 0; u < DEC_U; ++u) {
            float pu = fast_exp2(s[u] - m_new);
            l += pu;
            accumulate_values<DTYPE>(pu * vsr[u], vreg[u], acc);
        }
        if (FRONT && base + WAVES * ROWS_PER_STEP < s1) request(base + WAVES * ROWS_PER_STEP);
    }

    // ---- merge the lane groups of this wave ---------------------------------------------------
    // One maximum for all of them, then every exchange halves what a lane still adds up: 15 sums per lane instead of 64 (with all
    // of them in every lane, through LDS, the merge took 1.1 of a short launch's 6 us).  A lane ends with the columns
    // 16 c + e .. of its c, e the bits of its group number from the top.
    const auto largest = [](float x, float y) __attribute__((always_inline)) { return fmaxf(x, y); };
    const auto sum = [](float x, float y) __attribute__((always_inline)) { return x + y; };
    const float m_wave = lane_reduce<LPK, 32>(m, largest), f_lane = fast_exp2(m - m_wave);
    l = lane_reduce<LPK, 32>(l * f_lane, sum);
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] *= f_lane;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        lane_swap32(acc[i], acc[i + 8]);
        acc[i] += acc[i + 8];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        lane_swap16(acc[i], acc[i + 4]);
        acc[i] += acc[i + 4];
    }
    const bool high8 = lane & 8, high4 = lane & 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float keep = high8 ? acc[i + 2] : acc[i], give = high8 ? acc[i] : acc[i + 2];
        acc[i] = keep + lane_xor8(give);
    }
    const int e = (lane >> 5) * 8 + ((lane >> 4) & 1) * 4 + (high8 ? 2 : 0);
    if (LPK == 4) {
        const float keep = high4 ? acc[1] : acc[0], give = high4 ? acc[0] : acc[1];
        sm_acc[wave][c * 16 + e + (high4 ? 1 : 0)] = keep + lane_xor4(give);
    } else {
        *(v2f *)&sm_acc[wave][c * 16 + e] = v2f{acc[0], acc[1]};
    }
    if (lane == 0) { sm_m[wave] = m_wave; sm_l[wave] = l; }
    __syncthreads();
    // ---- merge the waves, write this split's partial --------------------------------------------
    if (tid < D) {
        const float m_w = sm_m[lane % WAVES], M = lane_reduce<1, WAVES / 2>(m_w, largest); // (lane i: wave i % WAVES)
        const float f_w = fast_exp2(m_w - M), L = lane_reduce<1, WAVES / 2>(sm_l[lane % WAVES] * f_w, sum);
        float o = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) o += sm_acc[w][tid] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f_w), w));
        if (direct) {
            // the only split: add the zero vector's weight 2^-M (M >= 0 by construction) and normalise here
            const float res = o / (L + fast_exp2(-M));
            p.out[((int64_t)seq * p.n_heads + head) * D + tid] = res;
            if (FRONT) kv_product_store<D>(f_row + 2 * D - (int64_t)head * D, 0, p.kv_out, p.kv_out_pitch, p.kv_rep, p.kv_mult, seq, head, tid, res);
            else if (p.kv_out) kv_product_store<D>(p.kv_k, p.kv_k_pitch, p.kv_out, p.kv_out_pitch, p.kv_rep, p.kv_mult, seq, head, tid, res);
        } else {
            p.part_acc[part * D + tid] = o;
            if (tid == 0) { p.part_ml[part * 2] = M; p.part_ml[part * 2 + 1] = L; }
        }
    }
    if (count_row) report_done(); // after the barrier above: every thread has read the old length
}

template <int DTYPE, int D, bool QBF16, bool GENERAL, bool FRONT, int DEC_U>
__global__ __launch_bounds__(DEC_WAVES * WAVE) void decode_split_kernel(DecodeParams p)
{
    decode_split<DTYPE, D, QBF16, GENERAL, FRONT, DEC_WAVES, DEC_U>(p);
}

// Sixteen waves per workgroup
template <int DTYPE, int D, bool QBF16, bool FRONT, int DEC_U>
__global__ __launch_bounds__(DEC_WIDE_WAVES * WAVE) void decode_wide_kernel(DecodeParams p)
{
    decode_split<DTYPE, D, QBF16, false, FRONT, DEC_WIDE_WAVES, DEC_U>(p);
}

// out = sum_s acc_s 2^(m_s - M) / (2^-M + sum_s l_s 2^(m_s - M)),  M = max(0, max_s m_s)
template <int D>
__global__ __launch_bounds__(D) void decode_merge_kernel(const float *part_acc, const float *part_ml, int n_splits, float *out,
                                                         int32_t *bump_len, int n_heads, int max_len, const uint8_t *kv_k,
                                                         int64_t kv_k_pitch, uint8_t *kv_out, int64_t kv_out_pitch, int kv_rep, float kv_mult)
{
    const int64_t sh = blockIdx.x; // seq * n_heads + head
    const int x = threadIdx.x;
    // after a fused append: every split kernel has finished with the old length, count the new row
    if (bump_len && x == 0 && sh % n_heads == 0) {
        const int64_t seq = sh / n_heads;
        const int len = bump_len[seq];
        if (len >= 0 && len < max_len) bump_len[seq] = len + 1;
    }
    float M = 0.0f;
    for (int s = 0; s < n_splits; ++s) M = fmaxf(M, part_ml[(sh * n_splits + s) * 2]);
    float L = fast_exp2(-M); // the zero vector of weight 1 (cpu_infer.cpp:444)
    float o = 0;
    for (int s = 0; s < n_splits; ++s) {
        float f = fast_exp2(part_ml[(sh * n_splits + s) * 2] - M);
        L += part_ml[(sh * n_splits + s) * 2 + 1] * f;
        o += part_acc[(sh * n_splits + s) * D + x] * f;
    }
    const float res = o / L;
    out[sh * D + x] = res;
    if (kv_out) kv_product_store<D>(kv_k, kv_k_pitch, kv_out, kv_out_pitch, kv_rep, kv_mult, sh / n_heads, (int)(sh % n_heads), x, res);
}

template <int DTYPE, int D, int U>
static hipError_t launch_decode_u(const DecodeParams &p, bool qbf16, dim3 grid, hipStream_t st)
{
    const dim3 block(DEC_WAVES * WAVE);
    const bool general = p.form.general;
    if (p.front.src) {
        if constexpr (DTYPE == TSATTN_I8) {
            if (qbf16 || p.dbg || !p.kv_out) return hipErrorInvalidValue;
            if (general) hipLaunchKernelGGL((decode_split_kernel<TSATTN_I8, D, false, true, true, U>), grid, block, 0, st, p);
            else hipLaunchKernelGGL((decode_split_kernel<TSATTN_I8, D, false, false, true, U>), grid, block, 0, st, p);
        } else {
            return hipErrorInvalidValue;
        }
    } else if (qbf16) {
        if (general) hipLaunchKernelGGL((decode_split_kernel<DTYPE, D, true, true, false, U>), grid, block, 0, st, p);
        else hipLaunchKernelGGL((decode_split_kernel<DTYPE, D, true, false, false, U>), grid, block, 0, st, p);
    } else {
        if (general) hipLaunchKernelGGL((decode_split_kernel<DTYPE, D, false, true, false, U>), grid, block, 0, st, p);
        else hipLaunchKernelGGL((decode_split_kernel<DTYPE, D, false, false, false, U>), grid, block, 0, st, p);
    }
    return hipGetLastError();
}

template <int DTYPE, int D, int U>
static hipError_t launch_decode_wide(const DecodeParams &p, bool qbf16, dim3 grid, hipStream_t st)
{
    const dim3 block(DEC_WIDE_WAVES * WAVE);
    if (p.front.src) {
        if constexpr (DTYPE == TSATTN_I8) {
            if (qbf16 || !p.kv_out) return hipErrorInvalidValue;
            hipLaunchKernelGGL((decode_wide_kernel<TSATTN_I8, D, false, true, U>), grid, block, 0, st, p);
        } else {
            return hipErrorInvalidValue;
        }
    } else if (qbf16) {
        hipLaunchKernelGGL((decode_wide_kernel<DTYPE, D, true, false, U>), grid, block, 0, st, p);
    } else {
        hipLaunchKernelGGL((decode_wide_kernel<DTYPE, D, false, false, U>), grid, block, 0, st, p);
    }
    return hipGetLastError();
}

template <int DTYPE, int D>
static hipError_t launch_decode_dd(const DecodeParams &p, bool qbf16, dim3 grid, hipStream_t st)
{
    if (p.form.waves == DEC_WIDE_WAVES) {
        return p.form.rows == DEC_SHORT ? launch_decode_wide<DTYPE, D, DEC_SHORT>(p, qbf16, grid, st) : launch_decode_wide<DTYPE, D, DEC_WIDE_LONG>(p, qbf16, grid, st);
    }
    return p.form.rows == DEC_SHORT ? launch_decode_u<DTYPE, D, DEC_SHORT>(p, qbf16, grid, st) : launch_decode_u<DTYPE, D, DEC_LONG>(p, qbf16, grid, st);
}

hipError_t launch_decode(const DecodeParams &p, int dtype, int head_dim, bool qbf16, int n_seqs, float *out, hipStream_t st)
{
    if (p.form.general ? p.form.waves != DEC_WAVES : p.dbg != nullptr || p.tok_stride >= DECODE_NEAR) return hipErrorInvalidValue;
    dim3 grid(p.n_splits, p.n_heads, n_seqs);
    hipError_t e;
    if (dtype == TSATTN_I8 && head_dim == 128) e = launch_decode_dd<TSATTN_I8, 128>(p, qbf16, grid, st);
    else if (dtype == TSATTN_I8 && head_dim == 64) e = launch_decode_dd<TSATTN_I8, 64>(p, qbf16, grid, st);
    else if (dtype == TSATTN_E4M3 && head_dim == 128) e = launch_decode_dd<TSATTN_E4M3, 128>(p, qbf16, grid, st);
    else if (dtype == TSATTN_E4M3 && head_dim == 64) e = launch_decode_dd<TSATTN_E4M3, 64>(p, qbf16, grid, st);
    else return hipErrorInvalidValue;
    if (e != hipSuccess) return e;
    if (p.n_splits == 1) return hipSuccess; // the split kernel wrote the output (and counted a fused append's row) itself
    dim3 mgrid((unsigned)(n_seqs * p.n_heads));
    int32_t *bump = p.k_new || p.front.src ? p.cache_len_rw : nullptr;
    if (head_dim == 128) hipLaunchKernelGGL((decode_merge_kernel<128>), mgrid, dim3(128), 0, st, p.part_acc, p.part_ml, p.n_splits, out, bump, p.n_heads, p.max_len, p.kv_k, p.kv_k_pitch, p.kv_out, p.kv_out_pitch, p.kv_rep, p.kv_mult);
    else hipLaunchKernelGGL((decode_merge_kernel<64>), mgrid, dim3(64), 0, st, p.part_acc, p.part_ml, p.n_splits, out, bump, p.n_heads, p.max_len, p.kv_k, p.kv_k_pitch, p.kv_out, p.kv_out_pitch, p.kv_rep, p.kv_mult);
    return hipGetLastError();
}

} // namespace tsattn
