// Internal helpers shared by the libwotk translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>

#include "../../include/wotk.h"

namespace wotk {

int fail(int code, const char *fmt, ...);

constexpr double kLog2E = 1.4426950408889634074;  // log2(e)
constexpr double kLn2 = 0.69314718055994530942;   // ln(2)

// Bump allocator over a caller-owned workspace.  With base == nullptr it only
// counts bytes, which is how the *_workspace_size() queries are answered, so
// the size query and the real carve-up can never disagree.
struct Arena {
    char *base;
    size_t cap;
    size_t off = 0;
    bool ok = true;
    Arena(void *b, size_t c) : base(static_cast<char *>(b)), cap(c) {}
    template <typename T>
    T *take(size_t n) {
        off = (off + 255) & ~size_t(255);
        T *p = base ? reinterpret_cast<T *>(base + off) : nullptr;
        off += n * sizeof(T);
        if (base && off > cap) ok = false;
        return p;
    }
};

#ifdef __HIPCC__
// 2^x for x in [-1100, inf): x = n + r, exp(r ln 2) by its Taylor series to degree 13
// (|r ln 2| <= 0.347: remainder under 5e-18), scaled by 2^n.  NaN stays NaN.
__device__ __forceinline__ double exp2_f64(double x) {
    const double n = rint(x), t = (x - n) * kLn2;
    double p = 1.0 / 6227020800.0;
    p = fma(p, t, 1.0 / 479001600.0);
    p = fma(p, t, 1.0 / 39916800.0);
    p = fma(p, t, 1.0 / 3628800.0);
    p = fma(p, t, 1.0 / 362880.0);
    p = fma(p, t, 1.0 / 40320.0);
    p = fma(p, t, 1.0 / 5040.0);
    p = fma(p, t, 1.0 / 720.0);
    p = fma(p, t, 1.0 / 120.0);
    p = fma(p, t, 1.0 / 24.0);
    p = fma(p, t, 1.0 / 6.0);
    p = fma(p, t, 0.5);
    p = fma(p, t, 1.0);
    p = fma(p, t, 1.0);
    return ldexp(p, (int)n);
}

// sums over a wave by DPP, no LDS permutes: row_shr 1, 2, 4, 8 (the last lane of each 16 holds
// their sum), then row_bcast 15 (lanes 31 and 63 hold the sums of their 32 lanes), then row_bcast 31
// (lane 63 holds the sum of all)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_sum_dpp(double v) {
    v = dpp_add<0x111, 0xf>(v);
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    return dpp_add<0x118, 0xf>(v);
}
__device__ __forceinline__ double half_wave_sum_dpp(double v) { return dpp_add<0x142, 0xa>(row_sum_dpp(v)); }
__device__ __forceinline__ double wave_sum_dpp(double v) { return dpp_add<0x143, 0xc>(half_wave_sum_dpp(v)); }

// sum and maximum over a wave in every lane
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
    return v;
}

// two partial sums sum_k 2^(y_k - sg) put together
__device__ __forceinline__ void lse_merge(double &sg, double &sd, double og, double os) {
    const double ng = fmax(sg, og);
    sd = ldexp(sd, (int)(sg - ng)) + ldexp(os, (int)(og - ng));
    sg = ng;
}
#endif

inline int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// Compiled tile variants of the sweep kernels, (rows per workgroup, threads).
// Entry 0 of each list is the built-in default.  The kernels are instantiated
// from these lists, so a variant exists exactly when it is listed here.
struct TileShape {
    int rows, threads;
    int wave_rows = 0;  // > 0: LDS-staged variant, each wave owns wave_rows of the tile's rows
};
constexpr TileShape kRowSweepTiles[] = {{4, 256}, {1, 256}, {2, 256}, {8, 256},
                                        {2, 512}, {4, 512}, {8, 512}, {4, 128}};
constexpr int kNumRowSweepTiles = sizeof(kRowSweepTiles) / sizeof(kRowSweepTiles[0]);
constexpr TileShape kBatchSweepTiles[] = {{2, 256}, {1, 256}, {4, 256}, {1, 512}, {2, 512}};
constexpr int kNumBatchSweepTiles = sizeof(kBatchSweepTiles) / sizeof(kBatchSweepTiles[0]);
constexpr TileShape kBatchSharedTiles[] = {{8, 256, 2},  {4, 256, 1},  {16, 256, 4}, {16, 512, 2},
                                           {8, 512, 1},  {2, 256},     {1, 256},     {2, 512}};
constexpr int kNumBatchSharedTiles = sizeof(kBatchSharedTiles) / sizeof(kBatchSharedTiles[0]);

// variant index (into the lists above) a launch of this shape uses
int tile_for(int kernel, int64_t n_rows, int64_t n_cols, int n_combos);

}  // namespace wotk

#define WOTK_HIP(expr)                                                                       \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            return wotk::fail(WOTK_EHIP, "%s failed: %s", #expr, hipGetErrorString(e_));   \
    } while (0)

#define WOTK_LAUNCH_CHECK()                                                                  \
    do {                                                                                     \
        hipError_t e_ = hipGetLastError();                                                   \
        if (e_ != hipSuccess)                                                                \
            return wotk::fail(WOTK_EHIP, "kernel launch failed at %s:%d: %s", __FILE__,      \
                              __LINE__, hipGetErrorString(e_));                              \
    } while (0)

#define WOTK_REQUIRE(cond, ...)                                                              \
    do {                                                                                     \
        if (!(cond)) return wotk::fail(WOTK_EINVAL, __VA_ARGS__);                            \
    } while (0)
