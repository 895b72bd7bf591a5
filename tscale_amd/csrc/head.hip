// The two ends of the int8 inference path around the layers (ComputePrediction, gpt/train/cpu_infer.cpp:552-582):
// the embedding sum that makes the first state, and the softmax over the final layer's products with the greedy
// choice of the next token; and the sampled choice (SampleFromDistr, :585-599).
#include "../../include/tsattn.h"
#include "common.hpp"
#include "kernels.hpp"

namespace tsattn {

#pragma clang fp contract(off)

// state[row][x] = sum over the row's labels of embed[label][x] * scale, added in label order starting from 0
// (cpu_infer.cpp:559-565).  One thread per four consecutive x, so that a wave stores 1 KiB of consecutive floats (bound by
// those stores: 65536 rows of 2048, 184 us with sixteen x per thread, whose stores leave 64-byte gaps).
__global__ __launch_bounds__(256) void embed_rows_kernel(HeadParams p)
{
    const unsigned blocks_per_row = (p.dim / 4 + 255) / 256;
    const int64_t row = blockIdx.x / blocks_per_row;
    const int x0 = (int)((blockIdx.x % blocks_per_row) * 256 + threadIdx.x) * 4;
    if (x0 >= p.dim) return;
    v4f acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (int l = 0; l < p.labels_per_row; ++l) {
        const int label = p.labels[row * p.labels_per_row + l];
        if (label < 0 || label >= p.n_labels) continue; // an empty slot
        const int w = *(const int *)(p.embed + (int64_t)label * p.embed_pitch + x0);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] = acc[j] + (float)(int8_t)((w >> (8 * j)) & 0xff) * p.embed_scale;
    }
    *(v4f *)(p.state + row * p.state_pitch + x0) = acc;
}

// w[k] = vec[k] * scale + bias[k]; M = max(0, max w) (the buffer's maximum starts at 0, cpu_infer.cpp:226-244);
// p[k] = 2^(w[k] - M) / sum (base 2: the scale carries 1/ln 2).  The choice is the first k of the largest w.
//
// A row is cut into chunks, one workgroup each, so that few rows still fill the chip: a vocabulary row of 200 KB for one
// compute unit is bound by what that unit can have in flight.  Two launches: every chunk's largest value, where it is
// first reached and the sum of its weights, then every chunk merges all of its row's records and writes its probabilities.
// 32 x 50257: 25.6 us with one workgroup per row walking it three times, 11.8 us like this.
// Rows of one chunk: both steps in one launch (32 x 1000 8.7 -> 5.8 us).
//
// Calls on one handle may be on several streams at once, so the records between the two launches cannot stand in the handle.
// They stand in scratch that the caller lends; without it, in the probabilities' own place until those are written (every chunk
// puts its record at the front of every chunk of its row, and the second launch reads the ones at the front of its own chunk
// only: 32 x 50257 0.4 us more).  A choice without probabilities has no such place: without scratch the chunks exchange the
// choice itself (32 x 50257: greedy choice 15 us, sampling 19 us; with scratch 6.8 and 10.3).
constexpr int SM_THREADS = 256, SM_ROW_THREADS = 1024;
constexpr int SM_U = 4;
constexpr int SM_CHUNK = 4 * SM_U * SM_THREADS; // values a workgroup of a chunk takes per round
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(4)));
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));
constexpr int NO_INDEX = 0x7fffffff;

__device__ inline float softmax_logit(const HeadParams &p, int64_t row, int64_t k)
{
    int v = p.src[row * p.src_pitch + k];
    for (int pl = 1; pl < p.src_planes; ++pl) v += p.src[pl * p.src_plane_stride + row * p.src_pitch + k];
    const float w = (float)v * p.scale;
    return p.bias ? w + p.bias[k] : w;
}

// the same for k .. k + 3
__device__ inline v4f softmax_logit4(const HeadParams &p, int64_t row, int64_t k)
{
    v4i v = *(const v4i_any *)(p.src + row * p.src_pitch + k);
    for (int pl = 1; pl < p.src_planes; ++pl) v += *(const v4i_any *)(p.src + pl * p.src_plane_stride + row * p.src_pitch + k);
    v4f w = v4f{(float)v.x * p.scale, (float)v.y * p.scale, (float)v.z * p.scale, (float)v.w * p.scale};
    if (p.bias) {
        const v4f b = *(const v4f_any *)(p.bias + k);
        w = v4f{w.x + b.x, w.y + b.y, w.z + b.z, w.w + b.w};
    }
    return w;
}

// Walks the values [begin, end) of a row (begin a multiple of 4): groups of four from the front, SM_U requests per thread
// out before the first is used (none under a branch: a group past the end asks for the last whole group again), then the
// up to three values that are left.  A thread sees its k in ascending order.
template <int THREADS, typename F>
__device__ inline void softmax_walk(const HeadParams &p, int64_t row, int64_t begin, int64_t end, int tid, F &&f)
{
    const int64_t n4 = begin + ((end - begin) & ~(int64_t)3);
    for (int64_t base = begin; base < n4; base += 4 * SM_U * THREADS) {
        v4f w[SM_U];
#pragma unroll
        for (int u = 0; u < SM_U; ++u) {
            const int64_t k = base + 4 * (tid + u * THREADS);
            w[u] = softmax_logit4(p, row, k < n4 ? k : n4 - 4);
        }
#pragma unroll
        for (int u = 0; u < SM_U; ++u) {
            const int64_t k = base + 4 * (tid + u * THREADS);
            if (k < n4) f(k, w[u], 4);
        }
    }
    if (n4 + tid < end) {
        const float w = softmax_logit(p, row, n4 + tid);
        f(n4 + tid, v4f{w, w, w, w}, 1);
    }
}

// largest value and the first index of it over the workgroup; every thread gets both
template <int THREADS>
__device__ inline void first_max(float &best, int &arg, float *s_max, int *s_arg, int tid)
{
    for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o, WAVE);
        const int oa = __shfl_xor(arg, o, WAVE);
        if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
    }
    if ((tid & (WAVE - 1)) == 0) { s_max[tid / WAVE] = best; s_arg[tid / WAVE] = arg; }
    __syncthreads();
    best = s_max[0]; arg = s_arg[0];
    for (int w = 1; w < THREADS / WAVE; ++w) {
        if (s_max[w] > best || (s_max[w] == best && s_arg[w] < arg)) { best = s_max[w]; arg = s_arg[w]; }
    }
}

// The largest value of [begin, end) and where it is first reached, to every thread.
template <int THREADS>
__device__ inline void softmax_best(const HeadParams &p, int64_t row, int64_t begin, int64_t end, int tid, float &best, int &arg)
{
    __shared__ float s_max[THREADS / WAVE];
    __shared__ int s_arg[THREADS / WAVE];
    best = -INFINITY;
    arg = NO_INDEX;
    softmax_walk<THREADS>(p, row, begin, end, tid, [&](int64_t k, v4f w, int) { // (a single value four times changes nothing)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (w[j] > best) { best = w[j]; arg = (int)k + j; }
    });
    first_max<THREADS>(best, arg, s_max, s_arg, tid);
}

// the sum of the weights of [begin, end) against M, to every thread
template <int THREADS>
__device__ inline float softmax_sum(const HeadParams &p, int64_t row, int64_t begin, int64_t end, int tid, float M)
{
    __shared__ float s_sum[THREADS / WAVE];
    float sum = 0.0f;
    softmax_walk<THREADS>(p, row, begin, end, tid, [&](int64_t, v4f w, int count) {
        sum += fast_exp2(fmaxf(w.x - M, -127.0f));
        if (count == 4) sum += fast_exp2(fmaxf(w.y - M, -127.0f)) + fast_exp2(fmaxf(w.z - M, -127.0f)) + fast_exp2(fmaxf(w.w - M, -127.0f));
    });
    sum = wave_sum(sum);
    if ((tid & (WAVE - 1)) == 0) s_sum[tid / WAVE] = sum;
    __syncthreads();
    sum = 0.0f;
    for (int w = 0; w < THREADS / WAVE; ++w) sum += s_sum[w];
    return sum;
}

// (a thread writes only what it has read itself: the probabilities may take the products' place)
template <int THREADS>
__device__ inline void softmax_store(const HeadParams &p, int64_t row, int64_t begin, int64_t end, int tid, float M, float sum)
{
    const float inv = 1.0f / sum;
    float *const prob = p.prob + row * p.prob_pitch;
    softmax_walk<THREADS>(p, row, begin, end, tid, [&](int64_t k, v4f w, int count) {
        v4f q;
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = fast_exp2(fmaxf(w[j] - M, -127.0f)) * inv;
        if (count == 4) *(v4f_any *)(prob + k) = q;
        else prob[k] = q.x;
    });
}

// one workgroup per row
template <int THREADS>
__global__ __launch_bounds__(THREADS) void softmax_rows_kernel(HeadParams p)
{
    const int64_t row = p.row0 + blockIdx.x;
    const int tid = threadIdx.x;
    float best;
    int arg;
    softmax_best<THREADS>(p, row, 0, p.n, tid, best, arg);
    if (tid == 0 && p.argmax) p.argmax[row] = arg;
    if (!p.prob) return;
    const float M = fmaxf(0.0f, best), sum = softmax_sum<THREADS>(p, row, 0, p.n, tid, M);
    softmax_store<THREADS>(p, row, 0, p.n, tid, M, sum);
}

// a chunk's record in lent scratch
__device__ inline v4f_any *head_record(const HeadParams &p, int64_t row, int n_chunks, int chunk)
{
    return (v4f_any *)p.scratch + row * n_chunks + chunk;
}

__global__ __launch_bounds__(256) void head_fill_kernel(int32_t *dst, int64_t n, int32_t value)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = value;
}

// A chunk's best value into the row's choice, which workgroups of the row share: the index of the best one so far, whose value is
// computed again from the inputs, so that the 32 bits of the output are all the memory it takes.  The result does not
// depend on the order of the workgroups; every failed exchange is another's success.  Called by one thread.
template <typename F>
__device__ inline void offer_choice(int32_t *choice, float best, int arg, F &&value_of)
{
    int have = __hip_atomic_load(choice, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    do {
        if (have != NO_INDEX) {
            const float v = value_of(have);
            if (v > best || (v == best && have <= arg)) return;
        }
    } while (!__hip_atomic_compare_exchange_strong(choice, &have, arg, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// The chunks' records {best, its index, sum of the weights against max(0, best)} -- the floor of 0 in it, so that a row whose values
// are all far below adds up the clamped weights as one pass over it would -- or without probabilities the choice alone.
template <bool PROB>
__global__ __launch_bounds__(SM_THREADS) void softmax_stats_kernel(HeadParams p)
{
    const int64_t row = blockIdx.y;
    const int tid = threadIdx.x;
    const int64_t begin = (int64_t)blockIdx.x * p.chunk, end = begin + p.chunk < p.n ? begin + p.chunk : p.n;
    float best;
    int arg;
    softmax_best<SM_THREADS>(p, row, begin, end, tid, best, arg);
    if constexpr (PROB) {
        const float sum = softmax_sum<SM_THREADS>(p, row, begin, end, tid, fmaxf(0.0f, best)); // the chunk again, from the nearest cache
        const v4f record = v4f{best, __int_as_float(arg), sum, 0.0f};
        if (p.scratch) {
            if (tid == 0) *head_record(p, row, gridDim.x, blockIdx.x) = record;
        } else if (tid < (int)gridDim.x) {
            *(v4f_any *)(p.prob + row * p.prob_pitch + tid * p.chunk + 4 * blockIdx.x) = record;
        }
    } else if (tid == 0) {
        if (p.scratch) *head_record(p, row, gridDim.x, blockIdx.x) = v4f{best, __int_as_float(arg), 0.0f, 0.0f};
        else if (arg != NO_INDEX) offer_choice(p.argmax + row, best, arg, [&](int k) { return softmax_logit(p, row, k); });
    }
}

__global__ __launch_bounds__(SM_THREADS) void softmax_write_kernel(HeadParams p)
{
    const int64_t row = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), n_chunks = (int)gridDim.x;
    const int64_t begin = (int64_t)blockIdx.x * p.chunk, end = begin + p.chunk < p.n ? begin + p.chunk : p.n;
    // every wave merges the row's records for itself
    const v4f_any *const rec = p.scratch ? head_record(p, row, n_chunks, 0) : (const v4f_any *)(p.prob + row * p.prob_pitch + begin);
    float best = -INFINITY, top = 0.0f, sum = 0.0f;
    int arg = NO_INDEX;
    for (int i = lane; i < n_chunks; i += WAVE) {
        const v4f r = rec[i];
        if (r.x > best) { best = r.x; arg = __float_as_int(r.y); }
        const float m = fmaxf(top, r.x);
        sum = sum * fast_exp2(top - m) + r.z * fast_exp2(fmaxf(0.0f, r.x) - m);
        top = m;
    }
    if (!p.scratch) __syncthreads(); // read by all: the front of the chunk may be written
    for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o, WAVE), ot = __shfl_xor(top, o, WAVE), os = __shfl_xor(sum, o, WAVE);
        const int oa = __shfl_xor(arg, o, WAVE);
        if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
        const float m = fmaxf(top, ot);
        sum = sum * fast_exp2(top - m) + os * fast_exp2(ot - m);
        top = m;
    }
    if (blockIdx.x == 0 && tid == 0 && p.argmax) p.argmax[row] = arg;
    softmax_store<SM_THREADS>(p, row, begin, end, tid, top, sum);
}

// the choice from the chunks' records, one wave per row; `none`: what a row gets that has no value to choose
__global__ __launch_bounds__(WAVE) void head_merge_kernel(HeadParams p, int n_chunks, int32_t none)
{
    const int64_t row = blockIdx.x;
    const int lane = threadIdx.x;
    float best = -INFINITY;
    int arg = NO_INDEX;
    for (int i = lane; i < n_chunks; i += WAVE) {
        const v4f r = *head_record(p, row, n_chunks, i);
        if (r.x > best) { best = r.x; arg = __float_as_int(r.y); }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const float ob = __shfl_xor(best, o, WAVE);
        const int oa = __shfl_xor(arg, o, WAVE);
        if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
    }
    if (lane == 0) p.argmax[row] = arg == NO_INDEX ? none : arg;
}

// SampleFromDistr (cpu_infer.cpp:585-599), the Gumbel-max choice:
// score[k] = (float)(logf(prob[k]) / temperature - log(-log(u))), u = (r + 0.5) / 2^32 in double (GenRandReal3 of the
// reference's 32-bit generator); the first k of the largest score above -1e38, else 0.  r: the caller's words, or a
// 64-bit mix of (seed, offset + row * n + k), the output function of splitmix64 on a counter.
//
// Two logarithms in double per value were 80 us for 32 x 50257 values.  Only values that can win need them: a wave scores
// 1024 values with the single-precision logarithm first, and evaluates exactly those that come within the error of that
// score of the best so far -- one or two of the 1024.  Rows are cut into chunks as for the softmax.
__device__ inline uint32_t mix32(uint64_t seed, uint64_t index)
{
    uint64_t z = seed + (index + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (uint32_t)(z >> 32);
}

// The score to within 1e-3 + 1e-5 |log(prob) / temperature|.  -log(u): from u where u is below 1 - 2^-6 (its rounding to
// float moves log(u) by 4e-6 of itself at most), from the series in 1 - u above (three terms leave 2^-24 of it).
__device__ inline float rough_score(float prob, uint32_t r, float inv_temperature)
{
    const float LN2 = 0.69314718f;
    const float u = ((float)r + 0.5f) * (1.0f / 4294967296.0f), v = ((float)(~r) + 0.5f) * (1.0f / 4294967296.0f);
    const float near_one = v * (1.0f + v * (0.5f + v * 0.33333333f)), far = -LN2 * __builtin_amdgcn_logf(u);
    const float e = v < 0.015625f ? near_one : far;
    // (the logarithm instruction takes a denormal for zero)
    const float lp = prob < 1e-30f ? __builtin_amdgcn_logf(prob * 4294967296.0f) - 32.0f : __builtin_amdgcn_logf(prob);
    return LN2 * (lp * inv_temperature - __builtin_amdgcn_logf(e));
}

__device__ inline float exact_score(const HeadParams &p, int64_t row, int64_t k)
{
    const uint32_t word = p.rnd ? p.rnd[row * p.rnd_pitch + k] : mix32(p.seed, p.offset + (uint64_t)(row * p.n + k));
    const double u = ((double)word + 0.5) * (1.0 / 4294967296.0);
    return (float)((double)(logf(p.prob[row * p.prob_pitch + k]) / p.temperature) - log(-log(u)));
}

// CHUNKS: a chunk of the row; else all of it.  A row without a score above -1e38 gets 0 (what its chunks' choice starts at).
template <bool CHUNKS>
__global__ __launch_bounds__(SM_THREADS) void sample_rows_kernel(HeadParams p)
{
    __shared__ float s_max[SM_THREADS / WAVE];
    __shared__ int s_arg[SM_THREADS / WAVE];
    const int64_t row = CHUNKS ? blockIdx.y : p.row0 + blockIdx.x;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const int64_t begin = CHUNKS ? (int64_t)blockIdx.x * p.chunk : 0, end = CHUNKS && begin + p.chunk < p.n ? begin + p.chunk : p.n;
    const float *const prob = p.prob + row * p.prob_pitch;
    const uint32_t *const rnd = p.rnd ? p.rnd + row * p.rnd_pitch : nullptr;
    const uint64_t counter = p.offset + (uint64_t)(row * p.n);
    const float inv_t = fminf(1.0f / p.temperature, 3e38f);
    float best = -1e38f;
    int arg = NO_INDEX;
    constexpr int PER_WAVE = 16 * WAVE;
    for (int64_t base = begin + wave * PER_WAVE; base < end; base += PER_WAVE * (SM_THREADS / WAVE)) {
        float q[16];
        uint32_t r[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) { // (past the end: the last value again, which changes no maximum)
            const int64_t k = base + j * WAVE + lane, kc = k < end ? k : end - 1;
            q[j] = prob[kc];
            r[j] = rnd ? rnd[kc] : mix32(p.seed, counter + (uint64_t)kc);
        }
        float top = -INFINITY;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            q[j] = rough_score(q[j], r[j], inv_t);
            top = fmaxf(top, q[j]);
        }
        // the best of the wave so far, exact or rough, less the error both may have
        top = wave_max(fmaxf(top, best));
        const float bound = top - (2e-3f + 2e-5f * (fminf(fabsf(top), 1e30f) + 64.0f));
        uint32_t todo = 0;
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (q[j] >= bound && base + j * WAVE + lane < end) todo |= 1u << j;
        while (todo) {
            const int j = __ffs(todo) - 1;
            todo &= todo - 1;
            const int64_t k = base + j * WAVE + lane;
            const float score = exact_score(p, row, k);
            if (score > best) { best = score; arg = (int)k; } // (a thread's k ascend)
        }
    }
    first_max<SM_THREADS>(best, arg, s_max, s_arg, tid);
    if (tid != 0) return;
    if (!CHUNKS) p.argmax[row] = arg == NO_INDEX ? 0 : arg;
    else if (p.scratch) *head_record(p, row, gridDim.x, blockIdx.x) = v4f{best, __int_as_float(arg), 0.0f, 0.0f};
    else if (arg != NO_INDEX) offer_choice(p.argmax + row, best, arg, [&](int k) { return exact_score(p, row, k); });
}

// How many workgroups share each of `rows` rows, and the values each takes: one round's worth each as long as the rows
// are few, at most about four workgroups per compute unit in all, and of a size that the front of each, the last one too, has
// room for the row's records (which also bounds them: 1024 in lent scratch).
static int head_chunks(HeadParams &p)
{
    int64_t chunks = (p.n + SM_CHUNK - 1) / SM_CHUNK;
    const int64_t most = p.n_rows < 1024 ? 1024 / p.n_rows : 1;
    chunks = chunks < most ? chunks : most;
    chunks = chunks < SM_THREADS ? chunks : SM_THREADS; // (a thread per record)
    for (;; --chunks) {
        p.chunk = ((p.n + chunks - 1) / chunks + 3) & ~(int64_t)3;
        const int64_t last = p.n - (chunks - 1) * p.chunk;
        if (chunks == 1 || last >= 4 * chunks) return (int)chunks;
    }
}

static_assert(TSATTN_HEAD_SCRATCH_BYTES >= 1024 * 16 && TSATTN_HEAD_CHUNK == SM_CHUNK, "a record per workgroup; rows of one chunk have none");

hipError_t launch_embed_rows(const HeadParams &p, hipStream_t st)
{
    if (p.n_rows == 0) return hipSuccess;
    const int64_t blocks = p.n_rows * ((p.dim / 4 + 255) / 256);
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(embed_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, st, p);
    return hipGetLastError();
}

// rows in slices that fit a grid
template <typename F>
static void for_row_slices(HeadParams &p, F &&f)
{
    constexpr int64_t MOST = 1 << 30;
    for (p.row0 = 0; p.row0 < p.n_rows; p.row0 += MOST) f(dim3((unsigned)(p.n_rows - p.row0 < MOST ? p.n_rows - p.row0 : MOST)));
}

// the choice of rows in chunks: stats(grid) makes the records in lent scratch, or exchanges the choices, which start at `none`
template <typename F>
static void choose_in_chunks(const HeadParams &p, int chunks, int32_t none, hipStream_t st, F &&stats)
{
    if (!p.scratch) hipLaunchKernelGGL(head_fill_kernel, dim3((unsigned)((p.n_rows + 255) / 256)), dim3(256), 0, st, p.argmax, p.n_rows, none);
    stats(dim3((unsigned)chunks, (unsigned)p.n_rows));
    if (p.scratch) hipLaunchKernelGGL(head_merge_kernel, dim3((unsigned)p.n_rows), dim3(WAVE), 0, st, p, chunks, none);
}

hipError_t launch_softmax_rows(const HeadParams &params, hipStream_t st)
{
    HeadParams p = params;
    if (p.n_rows == 0 || p.n == 0) return hipSuccess;
    const int chunks = head_chunks(p);
    // Probabilities that overlap the inputs leave records no place among them.
    const float *const prob_end = p.prob + (p.n_rows - 1) * p.prob_pitch + p.n;
    const int32_t *const src_end = p.src + (p.src_planes - 1) * p.src_plane_stride + (p.n_rows - 1) * p.src_pitch + p.n;
    const auto overlaps = [&](const void *begin, const void *end) { return (uintptr_t)p.prob < (uintptr_t)end && (uintptr_t)begin < (uintptr_t)prob_end; };
    const bool in_place = p.prob && (overlaps(p.src, src_end) || (p.bias && overlaps(p.bias, p.bias + p.n)));
    if (chunks == 1 || (in_place && !p.scratch)) { // one workgroup per row, and no records
        for_row_slices(p, [&](dim3 grid) {
            if (p.n <= SM_CHUNK) hipLaunchKernelGGL((softmax_rows_kernel<SM_THREADS>), grid, dim3(SM_THREADS), 0, st, p);
            else hipLaunchKernelGGL((softmax_rows_kernel<SM_ROW_THREADS>), grid, dim3(SM_ROW_THREADS), 0, st, p);
        });
    } else if (p.prob) {
        const dim3 grid((unsigned)chunks, (unsigned)p.n_rows);
        hipLaunchKernelGGL((softmax_stats_kernel<true>), grid, dim3(SM_THREADS), 0, st, p);
        hipLaunchKernelGGL(softmax_write_kernel, grid, dim3(SM_THREADS), 0, st, p);
    } else {
        choose_in_chunks(p, chunks, NO_INDEX, st, [&](dim3 grid) { hipLaunchKernelGGL((softmax_stats_kernel<false>), grid, dim3(SM_THREADS), 0, st, p); });
    }
    return hipGetLastError();
}

hipError_t launch_sample_rows(const HeadParams &params, hipStream_t st)
{
    HeadParams p = params;
    const int chunks = head_chunks(p);
    if (chunks > 1) {
        choose_in_chunks(p, chunks, 0, st, [&](dim3 grid) { hipLaunchKernelGGL((sample_rows_kernel<true>), grid, dim3(SM_THREADS), 0, st, p); });
    } else {
        for_row_slices(p, [&](dim3 grid) { hipLaunchKernelGGL((sample_rows_kernel<false>), grid, dim3(SM_THREADS), 0, st, p); });
    }
    return hipGetLastError();
}

} // namespace tsattn
