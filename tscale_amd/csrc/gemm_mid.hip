// The int8 product with more rows than a token step has and fewer outputs than fill the chip with 256 x 256 tiles (a few
// short prompts): tiles of 64 or 128 rows by 128 columns, the whole of K in one workgroup, so that the producer (RoPE,
// residual update, normalisation, int8 rows) can be the product's last step here too.
//
// What bounds it is what a compute unit gets from its L2 (64 bytes a cycle) and moves in and out of LDS (128), then latency.
// The 128 x 128 kernel this replaces waited for all its requests at every __syncthreads(), a memory round trip per 64 bytes of
// K (531 x 8192 -> 2048: 53 us; now 25 us with the producer's steps).  Here
// * K goes by in stages of 128 bytes that memory writes straight into LDS (buffer_load ... lds), several stages ahead, and the
//   one barrier per stage waits by count for the stage that is due.  (Weights asked for in the layout of the matrix
//   instructions instead, a row per lane, come in at a quarter of the rate: neighbouring lanes have to share a line.);
// * eight waves of 64 x 64: the two or four groups of waves that cover the tile once each take 64 or 32 of a stage's 128 bytes,
//   so that an operand read from LDS is used twice over and a SIMD has two waves; the groups' sums meet in LDS at the end;
// * the operands of a stage are read from LDS while the matrix instructions of the stage before run;
// * LDS rows are 128 bytes, the 16-byte chunk c of row r at position c ^ (r % 8) (applied to the addresses the lanes ask memory
//   for): operand reads free of bank conflicts;
// * an XCD's workgroups take neighbouring tiles, eight tile rows at a time, so that its L2 holds what they share.
#include "common.hpp"
#include "kernels.hpp"

namespace tsattn {

namespace {

constexpr int GM_THREADS = 512, GM_BN = 128, GM_BK = 128;
constexpr int GM_PITCH = GM_BN + 4; // result rows in LDS, in words
constexpr int gm_groups(int bm) { return bm == 64 ? 4 : 2; } // groups of waves that share K
// the stages; after them two planes of sums (then the values and their squares), a multiplier per (row, head)
constexpr int gm_stages(int bm) { return bm == 64 ? 6 : 5; }
constexpr int gm_lds_bytes(int bm)
{
    const int staged = gm_stages(bm) * (bm + GM_BN) * GM_BK, result = (2 * bm * GM_PITCH + 2 * bm) * 4;
    return staged > result ? staged : result;
}
typedef int v4i_w __attribute__((ext_vector_type(4), aligned(4)));
typedef float v4f_w __attribute__((ext_vector_type(4), aligned(4)));

__device__ inline __amdgpu_buffer_rsrc_t gm_rows(const uint8_t *base, int rows, int64_t pitch, int64_t row_bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, (int)((rows - 1) * pitch + row_bytes), 0x00020000);
}

// 64 lanes' 16 bytes from memory to 1 KiB of LDS
__device__ __forceinline__ void gm_request(__amdgpu_buffer_rsrc_t rows, uint8_t *lds, int offset)
{
    typedef __attribute__((address_space(3))) void *lds_ptr;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (lds_ptr)lds, 16, offset, 0, 0, 0);
}

__device__ __forceinline__ void gm_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int BM, int MODE, int EP_D>
__global__ __launch_bounds__(GM_THREADS, 2) void gemm_mid_kernel(GemmParams p)
{
#pragma clang fp contract(off)
    extern __shared__ __attribute__((aligned(16))) uint8_t gm_lds[];
    constexpr int NS = gm_stages(BM), STAGE = (BM + GM_BN) * GM_BK, A_REQ = BM / 64, LPS = A_REQ + 2; // requests of a stage per wave
    constexpr int KG = gm_groups(BM), KS = 4 / KG; // groups, 32-byte steps of K per group and stage
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int kg = wave / (8 / KG), wm = BM == 64 ? 0 : (wave >> 1) & 1, wn = wave & 1; // waves 0-3 and 4-7 sit on SIMDs 0-3 each
    const int li = lane & 31, g = lane >> 5;

    // which tile: runs of neighbouring tiles per XCD (workgroups go to them round-robin), columns walked under groups of
    // eight tile rows
    const int tiles_n = (int)((p.n + GM_BN - 1) / GM_BN), tiles_m = (int)((p.m + BM - 1) / BM);
    const int total = tiles_n * tiles_m, xcd = blockIdx.x & 7, per = total >> 3, more = total & 7;
    const int t = xcd * per + min(xcd, more) + (int)(blockIdx.x >> 3);
    const int group = t / (8 * tiles_n), rows_in = min(8, tiles_m - group * 8), within = t - group * 8 * tiles_n;
    const int64_t m0 = (int64_t)(group * 8 + within % rows_in) * BM, n0 = (int64_t)(within / rows_in) * GM_BN;
    const int rows_here = (int)(p.m - m0 < BM ? p.m - m0 : BM), cols_here = (int)(p.n - n0 < GM_BN ? p.n - n0 : GM_BN);

    // (what is asked for past a tile's last row comes back as zeros)
    const __amdgpu_buffer_rsrc_t ar = gm_rows(p.a + m0 * p.a_pitch, rows_here, p.a_pitch, p.k);
    const __amdgpu_buffer_rsrc_t wr = gm_rows(p.w + n0 * p.w_pitch, cols_here, p.w_pitch, p.k);
    // a wave's request fills eight rows; lane L writes position L % 8 of row L / 8
    const int r8 = lane >> 3, c8 = ((lane & 7) ^ r8) * 16;
    int a_off[A_REQ], w_off[2];
#pragma unroll
    for (int i = 0; i < A_REQ; ++i) a_off[i] = ((wave + 8 * i) * 8 + r8) * (int)p.a_pitch + c8;
#pragma unroll
    for (int i = 0; i < 2; ++i) w_off[i] = ((wave + 8 * i) * 8 + r8) * (int)p.w_pitch + c8;
    auto request = [&](int kb, uint8_t *buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < A_REQ; ++i) gm_request(ar, buf + (wave + 8 * i) * 1024, a_off[i] + kb);
#pragma unroll
        for (int i = 0; i < 2; ++i) gm_request(wr, buf + BM * GM_BK + (wave + 8 * i) * 1024, w_off[i] + kb);
    };
    int f[KS]; // this lane's chunks of a row
#pragma unroll
    for (int h = 0; h < KS; ++h) f[h] = li * GM_BK + ((((kg * KS + h) * 2 + g) ^ (li & 7)) << 4);

    v16i acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = v16i{0};

    const int n_stages = (int)((p.k + GM_BK - 1) / GM_BK), k_bytes = (int)p.k;
    struct Operands {
        v4i a[KS][2], w[KS][2];
    } op[2];
    auto read = [&](Operands &o, int stage) __attribute__((always_inline)) {
        const uint8_t *const cur = gm_lds + stage * STAGE;
#pragma unroll
        for (int h = 0; h < KS; ++h) {
#pragma unroll
            for (int i = 0; i < 2; ++i) o.a[h][i] = *(const v4i *)(cur + (wm * 64 + i * 32) * GM_BK + f[h]);
#pragma unroll
            for (int j = 0; j < 2; ++j) o.w[h][j] = *(const v4i *)(cur + (BM + wn * 64 + j * 32) * GM_BK + f[h]);
        }
    };
    auto next = [](int stage) __attribute__((always_inline)) { return stage + 1 == NS ? 0 : stage + 1; };
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) request(s * GM_BK, gm_lds + s * STAGE);
    // at step s: stage s is in registers; stage s + 1 has landed, for this wave by count and behind the barrier for all;
    // nobody reads stage s - 1 any more, whose place stage s + NS - 1 takes
    static_assert((NS - 2) * LPS == 12 && (NS - 3) * LPS == (BM == 64 ? 9 : 8), "the counts below");
    int due = 1, free_ = NS - 1;
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    gm_barrier();
    read(op[0], 0);
    auto step = [&](Operands &mine, Operands &coming, int s) __attribute__((always_inline)) {
        if constexpr (BM == 64) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        gm_barrier();
        request((s + NS - 1) * GM_BK, gm_lds + free_ * STAGE);
        __builtin_amdgcn_sched_barrier(0);
        read(coming, due);
        __builtin_amdgcn_sched_barrier(0);
        due = next(due);
        free_ = next(free_);
#pragma unroll
        for (int h = 0; h < KS; ++h) {
            if (s * GM_BK + (kg * KS + h) * 32 < k_bytes) { // (K may end in the middle of a stage)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(mine.a[h][i], mine.w[h][j], acc[i][j], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int s = 0; s < n_stages; s += 2) {
        step(op[0], op[1], s);
        if (s + 1 < n_stages) step(op[1], op[0], s + 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // nothing may still be on its way into LDS
    __syncthreads();

    // The groups' sums in two planes in LDS, row r of the tile at words r * GM_PITCH; whoever uses an element adds them up.
    int *const sums = (int *)gm_lds;
    constexpr int PLANE = BM * GM_PITCH;
    auto place = [&](int i, int j, int r) __attribute__((always_inline)) {
        return (kg & 1) * PLANE + (wm * 64 + i * 32 + 8 * (r / 4) + 4 * g + (r & 3)) * GM_PITCH + wn * 64 + j * 32 + li;
    };
    if (kg < 2) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) sums[place(i, j, r)] = acc[i][j][r];
    }
    __syncthreads();
    if constexpr (KG == 4) {
        if (kg >= 2) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sums[place(i, j, r)] += acc[i][j][r];
        }
        __syncthreads();
    }
    auto sum4 = [&](int row, int x) __attribute__((always_inline)) {
        return *(const v4i *)(sums + row * GM_PITCH + x) + *(const v4i *)(sums + PLANE + row * GM_PITCH + x);
    };

    if constexpr (EP_D == 0) {
        constexpr int ITER = BM * 32 / GM_THREADS; // four columns per thread and step
        if constexpr (MODE == TSATTN_MM_ADD_SCALED) {
            v4f old[ITER];
#pragma unroll
            for (int it = 0; it < ITER; ++it) { // all old values requested before the first is updated and stored
                const int row = (it * GM_THREADS + tid) >> 5, x = ((it * GM_THREADS + tid) & 31) * 4;
                const float *const o = (const float *)p.out + (m0 + row) * p.out_pitch + n0 + x;
                old[it] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
                if (row < rows_here) {
                    if (x + 4 <= cols_here) old[it] = *(const v4f_w *)o;
                    else
                        for (int c = 0; c < 4; ++c)
                            if (x + c < cols_here) old[it][c] = o[c];
                }
            }
#pragma unroll
            for (int it = 0; it < ITER; ++it) {
                const int row = (it * GM_THREADS + tid) >> 5, x = ((it * GM_THREADS + tid) & 31) * 4;
                const v4i v = sum4(row, x);
                float *const o = (float *)p.out + (m0 + row) * p.out_pitch + n0 + x;
                v4f d = v4f{(float)v.x, (float)v.y, (float)v.z, (float)v.w};
                d = v4f{d.x * p.scale, d.y * p.scale, d.z * p.scale, d.w * p.scale}; // delta * scale is rounded before it is added
                d = v4f{old[it].x + d.x, old[it].y + d.y, old[it].z + d.z, old[it].w + d.w};
                if (row < rows_here) {
                    if (x + 4 <= cols_here) *(v4f_w *)o = d;
                    else
                        for (int c = 0; c < 4; ++c)
                            if (x + c < cols_here) o[c] = d[c];
                }
            }
        } else {
#pragma unroll
            for (int it = 0; it < ITER; ++it) {
                const int row = (it * GM_THREADS + tid) >> 5, x = ((it * GM_THREADS + tid) & 31) * 4;
                if (row >= rows_here) continue;
                v4i v = sum4(row, x);
                if (MODE == TSATTN_MM_F32) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) v[c] = __float_as_int((float)v[c] * p.scale);
                }
                int32_t *const o = (int32_t *)p.out + (m0 + row) * p.out_pitch + n0 + x;
                if (x + 4 <= cols_here) *(v4i_w *)o = v;
                else
                    for (int c = 0; c < 4; ++c)
                        if (x + c < cols_here) o[c] = v[c];
            }
        }
        return;
    } else {
        // The producer (see rope_normalize_kernel): a thread takes four couples (x, x + 32) of a row, consecutive lanes
        // consecutive couples, so that state and rope rows are read and written in whole lines.
        constexpr int HEADS_T = GM_BN / EP_D, PAIRS = BM * HEADS_T, ITER = BM * 16 / GM_THREADS;
        float *const vals = (float *)gm_lds, *const squares = vals + PLANE, *const mults = vals + 2 * PLANE; // (over the planes of sums)
        const ProduceParams &e = p.ep;
        const int head0 = (int)(n0 / EP_D);
        v4f u0[ITER], u1[ITER];
        if (e.resid || e.pos) {
#pragma unroll
            for (int it = 0; it < ITER; ++it) {
                const int j = it * GM_THREADS + tid, c = j & 15, x = (c / 8) * 64 + (c % 8) * 4;
                const int row = min(j >> 4, rows_here - 1), xc = x < cols_here ? x : 0;
                const float *q;
                if (e.resid) {
                    q = e.resid + (m0 + row) * e.resid_pitch + n0 + xc;
                } else {
                    int at = e.pos[m0 + row];
                    at = at < 0 ? 0 : (at >= e.rope_len ? (int)e.rope_len - 1 : at);
                    q = e.rope + (int64_t)at * EP_D + xc % EP_D;
                }
                u0[it] = *(const v4f *)q;
                u1[it] = *(const v4f *)(q + 32);
            }
        }
#pragma unroll
        for (int it = 0; it < ITER; ++it) {
            const int j = it * GM_THREADS + tid, row = j >> 4, c = j & 15, x = (c / 8) * 64 + (c % 8) * 4;
            const v4i a = sum4(row, x), b = sum4(row, x + 32);
            v4f v0 = v4f{(float)a.x, (float)a.y, (float)a.z, (float)a.w}, v1 = v4f{(float)b.x, (float)b.y, (float)b.z, (float)b.w};
            if (e.resid) { // state += delta * scale, written back; the updated state is what gets normalised
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    v0[i] = u0[it][i] + v0[i] * e.resid_scale;
                    v1[i] = u1[it][i] + v1[i] * e.resid_scale;
                }
                if (row < rows_here && x < cols_here) {
                    float *const q = e.resid + (m0 + row) * e.resid_pitch + n0 + x;
                    *(v4f *)q = v0;
                    *(v4f *)(q + 32) = v1;
                }
            } else if (e.pos) {
                const bool turn = head0 + x / EP_D < e.rope_heads; // (the other heads turn by the identity)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float cos_value = turn ? u0[it][i] : 1.0f, sin_value = turn ? u1[it][i] * e.rotate_dir : 0.0f;
                    const float r0 = v0[i] * cos_value - v1[i] * sin_value;
                    const float r1 = v0[i] * sin_value + v1[i] * cos_value;
                    v0[i] = r0;
                    v1[i] = r1;
                }
            }
            *(v4f *)(vals + row * GM_PITCH + x) = v0;
            *(v4f *)(vals + row * GM_PITCH + x + 32) = v1;
            *(v4f *)(squares + row * GM_PITCH + x) = v4f{v0.x * v0.x, v0.y * v0.y, v0.z * v0.z, v0.w * v0.w};
            *(v4f *)(squares + row * GM_PITCH + x + 32) = v4f{v1.x * v1.x, v1.y * v1.y, v1.z * v1.z, v1.w * v1.w};
        }
        __syncthreads();
        if (tid < PAIRS) { // squares added in index order, scale
            const int row = tid / HEADS_T, ht = tid % HEADS_T;
            const float *const v = squares + row * GM_PITCH + ht * EP_D;
            float sum2 = 0.0f;
#pragma unroll
            for (int x = 0; x < EP_D; x += 32) {
                v4f q[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) q[c] = *(const v4f *)(v + x + 4 * c);
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    sum2 = sum2 + q[c].x;
                    sum2 = sum2 + q[c].y;
                    sum2 = sum2 + q[c].z;
                    sum2 = sum2 + q[c].w;
                }
            }
            float discr = 0.0f, mult = 0.0f;
            if (sum2 != 0.0f) {
                discr = (float)sqrt((double)(sum2 / (float)EP_D)) * e.vec_scale;
                mult = 1.0f / discr;
            }
            mults[tid] = mult;
            const int sh = head0 + ht - e.scale_head_begin;
            if (e.scale && row < rows_here && head0 + ht < e.n_heads && sh >= 0 && sh < e.scale_head_count)
                e.scale[sh * e.scale_pitch + (m0 + row) * e.scale_row_stride] = discr * e.scale_mult;
        }
        __syncthreads();
        const float low = e.relu ? 0.0f : -127.0f;
#pragma unroll
        for (int it = 0; it < BM * 8 / GM_THREADS; ++it) { // sixteen bytes per thread and step
            const int j = it * GM_THREADS + tid, row = j >> 3, x = (j & 7) * 16;
            const float mult = mults[row * HEADS_T + x / EP_D]; // a head of zeros has 0: zero bytes
            v4i w;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const v4f q = *(const v4f *)(vals + row * GM_PITCH + x + 4 * k);
                w[k] = (int)pack_i8x4(q.x * mult, q.y * mult, q.z * mult, q.w * mult, low);
            }
            if (row < rows_here && x < cols_here) *(v4i *)(e.dst + (m0 + row) * e.dst_pitch + n0 + x) = w;
        }
    }
}

template <int BM, int MODE, int EP_D>
hipError_t launch_one(const GemmParams &p, hipStream_t st, bool prepare)
{
    if (prepare) return hipFuncSetAttribute((const void *)gemm_mid_kernel<BM, MODE, EP_D>, hipFuncAttributeMaxDynamicSharedMemorySize, gm_lds_bytes(BM));
    const int64_t tiles = ((p.m + BM - 1) / BM) * ((p.n + GM_BN - 1) / GM_BN);
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_mid_kernel<BM, MODE, EP_D>), dim3((unsigned)tiles), dim3(GM_THREADS), gm_lds_bytes(BM), st, p);
    return hipGetLastError();
}

template <int BM>
hipError_t launch_bm(const GemmParams &p, int mode, int ep_d, hipStream_t st, bool prepare)
{
    if (ep_d == 128) return launch_one<BM, TSATTN_MM_I32, 128>(p, st, prepare);
    if (ep_d == 64) return launch_one<BM, TSATTN_MM_I32, 64>(p, st, prepare);
    if (mode == TSATTN_MM_F32) return launch_one<BM, TSATTN_MM_F32, 0>(p, st, prepare);
    if (mode == TSATTN_MM_ADD_SCALED) return launch_one<BM, TSATTN_MM_ADD_SCALED, 0>(p, st, prepare);
    return launch_one<BM, TSATTN_MM_I32, 0>(p, st, prepare);
}

} // namespace

hipError_t launch_gemm_mid(const GemmParams &p, int rows, int ep_d, hipStream_t st)
{
    return rows == 64 ? launch_bm<64>(p, p.mode, ep_d, st, false) : launch_bm<128>(p, p.mode, ep_d, st, false);
}

hipError_t prepare_gemm_mid()
{
    const GemmParams p = {};
    hipError_t e = hipSuccess;
    for (int ep_d = 0; ep_d <= 128 && e == hipSuccess; ep_d += 64)
        for (int mode : {TSATTN_MM_I32, TSATTN_MM_F32, TSATTN_MM_ADD_SCALED}) {
            if (ep_d && mode != TSATTN_MM_I32) continue;
            if (e == hipSuccess) e = launch_bm<64>(p, mode, ep_d, nullptr, true);
            if (e == hipSuccess) e = launch_bm<128>(p, mode, ep_d, nullptr, true);
        }
    return e;
}

} // namespace tsattn
