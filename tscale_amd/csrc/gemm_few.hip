// The int8 product with few activation rows (one token per sequence): plan and launches.  The kernel: gemm_few.hpp.
#include "few_offsets.h"
#include "gemm_stream.hpp"

namespace tsattn {

namespace {

struct FewPlan {
    int waves, parts, wn_log, k_part, k_chunk, groups;
    double ns;
};

int few_mt(int64_t m) { return m <= 16 ? 1 : m <= 32 ? 2 : m <= 64 ? 4 : 8; }

int log2_of(int x)
{
    int l = 0;
    while ((1 << l) < x) ++l;
    return l;
}

// What a launch with this cut would take, in nanoseconds; what matters is the order of the cuts.  From launches of
// 768 x 768 to 8192 x 2048 matrices under 1 and 32 rows, each with every cut (before the kernel's start became 1.2 us shorter, which
// is the same for all of them): 3.3 us for a launch whatever it does, the
// matrix at 6 TB/s, what a wave's steps add one after the other, the activations of a compute unit's workgroups (int8 rows,
// or what they are normalised from) at 45 bytes per nanosecond, and workgroups beyond one or two per compute unit, which
// cost their start: 8192 x 2048 under one row takes 6.3 us with 512 workgroups of four waves, 9.9 us with 1024.
FewPlan few_plan(const FewParams &p, int waves, int parts, int wn_log)
{
    FewPlan f;
    const int wn = 1 << wn_log, wk = waves / wn;
    const int unit = p.a ? 64 : (p.group > 64 ? p.group : 64); // K is cut into whole steps and whole groups
    const int64_t units = p.k / unit;
    f.waves = waves; f.parts = parts; f.wn_log = wn_log;
    f.k_part = (int)((units + parts - 1) / parts) * unit;
    f.k_chunk = f.k_part;
    const int mt = few_mt(p.m), group = p.a ? 0 : p.group;
    while (gf_lds_bytes(waves, mt, p.m, f.k_chunk, group) > GF_LDS_MAX && f.k_chunk > unit) f.k_chunk = ((f.k_chunk / unit + 1) / 2) * unit;
    // workgroups that walk several blocks: with one part, K undivided, and every wave with rows of its own
    f.groups = (int)((p.n + 16 * wn - 1) / (16 * wn));
    const int walkers = 256;
    if (parts == 1 && wk == 1 && f.k_chunk == f.k_part && f.groups > walkers) f.groups = walkers;
    const double words = p.a ? 1.0 : 4.0 * (p.src_planes + (p.state ? 1 : 0));
    const double units4 = (double)f.groups * parts * waves / 4; // workgroups of four waves
    const double steps = (double)f.k_part / 64 / wk * ((p.n + 15) / 16) / ((double)f.groups * wn);
    const double chunks = (f.k_part + f.k_chunk - 1) / f.k_chunk;
    const double a_bytes = words * p.m * f.k_part * (double)(((int64_t)f.groups * parts + 255) / 256);
    f.ns = 3300 + (double)p.n * p.k / 6000 + steps * (60 + 12 * mt) + (units4 > 512 ? 512 + (units4 - 512) * 7 : units4 > 256 ? (units4 - 256) * 2 : 0) +
           (waves == 8 ? 600 : 0) + a_bytes / 45 + (chunks - 1) * (p.a ? 1500 : 4000) + (parts - 1) * (100 + (double)p.m * p.n * 4 / 3000);
    return f;
}

FewPlan few_best(const FewParams &p, int min_parts, int max_parts)
{
    FewPlan best = {};
    for (int parts = min_parts; parts <= max_parts; parts *= 2) {
        if (parts > min_parts && p.k / parts < 128) break;
        for (int waves = 4; waves <= 8; waves += 4)
            for (int wn_log = 0; (1 << wn_log) <= waves; ++wn_log) {
                const FewPlan f = few_plan(p, waves, parts, wn_log);
                // (every part has K to multiply)
                if ((int64_t)(parts - 1) * f.k_part >= p.k) continue;
                if (best.parts == 0 || f.ns < best.ns) best = f;
            }
    }
    return best;
}

template <int THREADS, int MODE, int MT, int SRC, bool RESID>
hipError_t launch_threads(const FewParams &p, hipStream_t st, bool prepare)
{
    // Matrices of 8 MB and more as data that is not used again soon: 10 % faster at 50257 x 2048 (103 MB); smaller ones
    // (a whole small model stays in the caches from one token to the next) are up to 10 % slower that way.
    constexpr bool HAS_NT = SRC < 0 && MODE == TSATTN_MM_I32;
    const bool nt = HAS_NT && p.n * p.k >= (8 << 20);
    if (prepare) {
        const hipError_t e = hipFuncSetAttribute((const void *)gemm_few_kernel<THREADS, MODE, MT, SRC, RESID, false>, hipFuncAttributeMaxDynamicSharedMemorySize, GF_LDS_MAX);
        return e != hipSuccess ? e : hipFuncSetAttribute((const void *)gemm_few_kernel<THREADS, MODE, MT, SRC, RESID, HAS_NT>, hipFuncAttributeMaxDynamicSharedMemorySize, GF_LDS_MAX);
    }
    const int lds = gf_lds_bytes(THREADS / WAVE, MT, p.m, p.k_chunk, SRC < 0 ? 0 : p.group);
    const dim3 grid((unsigned)p.groups, (unsigned)p.parts);
    if (nt) hipLaunchKernelGGL((gemm_few_kernel<THREADS, MODE, MT, SRC, RESID, HAS_NT>), grid, dim3(THREADS), (unsigned)lds, st, p);
    else hipLaunchKernelGGL((gemm_few_kernel<THREADS, MODE, MT, SRC, RESID, false>), grid, dim3(THREADS), (unsigned)lds, st, p);
    return hipGetLastError();
}

template <int MODE, int MT, int SRC, bool RESID>
hipError_t launch_one(const FewParams &p, hipStream_t st, bool prepare)
{
    if (prepare) {
        const hipError_t e = launch_threads<256, MODE, MT, SRC, RESID>(p, st, true);
        return e != hipSuccess ? e : launch_threads<512, MODE, MT, SRC, RESID>(p, st, true);
    }
    return p.wn * p.wk == 4 ? launch_threads<256, MODE, MT, SRC, RESID>(p, st, false) : launch_threads<512, MODE, MT, SRC, RESID>(p, st, false);
}

template <int MODE>
hipError_t launch_rows(const FewParams &p, int mt, hipStream_t st, bool prepare)
{
    switch (mt) {
    case 1: return launch_one<MODE, 1, -1, false>(p, st, prepare);
    case 2: return launch_one<MODE, 2, -1, false>(p, st, prepare);
    case 4: return launch_one<MODE, 4, -1, false>(p, st, prepare);
    default: return launch_one<MODE, 8, -1, false>(p, st, prepare);
    }
}

// (Up to 16 rows: at 32 rows every workgroup would read 200 to 300 KB of planes to normalise its columns, 14 us for the
// 2048 x 2048 product where the separate normalisation and the product on its bytes take 10.)
hipError_t launch_norm(const FewParams &p, int planes, bool resid, hipStream_t st, bool prepare)
{
    if (planes == 0) return launch_one<TSATTN_MM_I32, 1, 0, true>(p, st, prepare);
    if (resid) {
        if (planes == 1) return launch_one<TSATTN_MM_I32, 1, 1, true>(p, st, prepare);
        if (planes == 2) return launch_one<TSATTN_MM_I32, 1, 2, true>(p, st, prepare);
        return launch_one<TSATTN_MM_I32, 1, 4, true>(p, st, prepare);
    }
    if (planes == 1) return launch_one<TSATTN_MM_I32, 1, 1, false>(p, st, prepare);
    if (planes == 2) return launch_one<TSATTN_MM_I32, 1, 2, false>(p, st, prepare);
    return launch_one<TSATTN_MM_I32, 1, 4, false>(p, st, prepare);
}

// The matrix through LDS (gemm_stream.hpp) from 20 MB on and up to 32 rows: 50257 x 2048 under 32 rows 27.8 -> 22.5 us, under
// one 26.3 -> 20.4; 20000 x 1024: 8.3 -> 8.0 and 8.6 -> 7.7.  Below that its one long run of the matrix per compute unit is no
// gain (8192 x 2048: 6.9 and 7.2 us); with 64 rows the activations leave little room for the waves' rings (20000 x 1024: 9.3
// and 10.2 us), and so does a K of 5000 and more.
bool stream_fits(const FewParams &p)
{
    return p.a && p.m <= 32 && p.n * p.k >= 20000000 && gs_lds_bytes(few_mt(p.m), p.k) <= GF_LDS_MAX;
}

template <int MODE>
hipError_t launch_stream(FewParams p, hipStream_t st, bool prepare)
{
    if (prepare) {
        const hipError_t e = hipFuncSetAttribute((const void *)gemm_stream_kernel<MODE, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, GF_LDS_MAX);
        return e != hipSuccess ? e : hipFuncSetAttribute((const void *)gemm_stream_kernel<MODE, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, GF_LDS_MAX);
    }
    const int mt = few_mt(p.m);
    const unsigned lds = (unsigned)gs_lds_bytes(mt, p.k);
    p.k_chunk = (int)gs_rows_bytes(mt, p.k);
    p.blk_per = (int)((p.n + 15) / 16) / 256; p.blk_more = (int)((p.n + 15) / 16) % 256;
    p.by_row = wg_make_div((uint32_t)p.k / 16);
    if (mt == 1) hipLaunchKernelGGL((gemm_stream_kernel<MODE, 1>), dim3(256), dim3(GS_THREADS), lds, st, p);
    else hipLaunchKernelGGL((gemm_stream_kernel<MODE, 2>), dim3(256), dim3(GS_THREADS), lds, st, p);
    return hipGetLastError();
}

} // namespace

bool few_source_ok(const FewParams &p)
{
    return p.m >= 1 && p.m <= FEW_NORM_ROWS && (p.group == 64 || p.group == 128) && p.k % p.group == 0 && p.k % 64 == 0 &&
           (p.src_planes == 1 || p.src_planes == 2 || p.src_planes == 4 || (p.src_planes == 0 && p.state)) &&
           few_offsets_fit(p.m, p.k, p.state_pitch);
}

int few_parts(const FewParams &p, int max_parts) { return stream_fits(p) ? 1 : few_best(p, 1, max_parts).parts; }

double few_ns(const FewParams &p, int max_parts)
{
    // (through LDS: the matrix, and the result; as measured between 16384 x 2048, 50257 x 512 and 50257 x 2048)
    return stream_fits(p) ? 4000 + (double)p.n * p.k / 6100 + p.m * (15 + (double)p.n * 4 / 4500) : few_best(p, 1, max_parts).ns;
}

double few_split(const FewParams &p, int max_parts, int *parts)
{
    double best = 0.0;
    *parts = 1;
    for (int n = 2; n <= max_parts && p.k / n >= 128; n *= 2) {
        const FewPlan f = few_best(p, n, n);
        const double ns = f.ns + 2700 + (double)(4 * n + 8) * (double)p.m * (double)p.n / 2200;
        if (f.parts && (*parts == 1 || ns < best)) { best = ns; *parts = n; }
    }
    return best;
}

hipError_t launch_gemm_few(const FewParams &params, hipStream_t st)
{
    FewParams p = params;
    if (p.m < 1 || p.m > FEW_ROWS || p.k <= 0 || p.k % 64 || p.parts < 1 || (p.parts > 1 && p.mode != TSATTN_MM_I32) ||
        (!p.a && (p.mode != TSATTN_MM_I32 || !few_source_ok(p))))
        return hipErrorInvalidValue;
    if (p.parts == 1 && stream_fits(p)) {
        if (p.mode == TSATTN_MM_I32) return launch_stream<TSATTN_MM_I32>(p, st, false);
        if (p.mode == TSATTN_MM_F32) return launch_stream<TSATTN_MM_F32>(p, st, false);
        return launch_stream<TSATTN_MM_ADD_SCALED>(p, st, false);
    }
    const FewPlan f = few_best(p, p.parts, p.parts);
    if (f.parts == 0) return hipErrorInvalidValue;
    p.wn_log = f.wn_log; p.wn = 1 << f.wn_log; p.wk = f.waves >> f.wn_log; p.wk_log = log2_of(p.wk); p.group_log = log2_of(p.group);
    p.k_part = f.k_part; p.k_chunk = f.k_chunk;
    p.groups = f.groups; p.walk = (int64_t)f.groups * 16 * p.wn < p.n;
    p.blk_per = (int)((p.n + 15) / 16) / f.groups; p.blk_more = (int)((p.n + 15) / 16) % f.groups;
    p.by_row = wg_make_div((uint32_t)p.k_chunk / (p.a ? 16 : 4));
    const int mt = few_mt(p.m);
    if (!p.a) return launch_norm(p, p.src_planes, p.state != nullptr, st, false);
    if (p.mode == TSATTN_MM_I32) return launch_rows<TSATTN_MM_I32>(p, mt, st, false);
    if (p.mode == TSATTN_MM_F32) return launch_rows<TSATTN_MM_F32>(p, mt, st, false);
    return launch_rows<TSATTN_MM_ADD_SCALED>(p, mt, st, false);
}

// Once per device, before the first product: the kernels may ask for all of a compute unit's LDS.
hipError_t prepare_gemm_few()
{
    const FewParams p = {};
    hipError_t e = hipSuccess;
    for (int mt = 1; mt <= 8 && e == hipSuccess; mt *= 2) {
        e = launch_rows<TSATTN_MM_I32>(p, mt, nullptr, true);
        if (e == hipSuccess) e = launch_rows<TSATTN_MM_F32>(p, mt, nullptr, true);
        if (e == hipSuccess) e = launch_rows<TSATTN_MM_ADD_SCALED>(p, mt, nullptr, true);
    }
    if (e == hipSuccess) e = launch_stream<TSATTN_MM_I32>(p, nullptr, true);
    if (e == hipSuccess) e = launch_stream<TSATTN_MM_F32>(p, nullptr, true);
    if (e == hipSuccess) e = launch_stream<TSATTN_MM_ADD_SCALED>(p, nullptr, true);
    for (int planes = 0; planes <= 4 && e == hipSuccess; planes = planes ? planes * 2 : 1)
        for (int resid = planes ? 0 : 1; resid < 2 && e == hipSuccess; ++resid) e = launch_norm(p, planes, resid != 0, nullptr, true);
    return e;
}

} // namespace tsattn
