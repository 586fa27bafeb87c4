// Fixed-iteration solve (transport_stablev2 semantics,
// wot/ot/optimal_transport.py:167-236) on the cost of ot_model.py:242-253
// without ever materialising the cost or the kernel: every sweep recomputes
// C_ij from the coordinates tile by tile on the matrix cores.
//
// Coordinates are centred on the mean of both days and scaled by
// 1/sqrt(median), so C = |x'|^2 + |y'|^2 - 2 x'.y' directly.  The cross term
// x'.y' is a split-BF16 MFMA product (x' = hi + mid + lo):
//   3 terms: hi.hi + hi.lo' + lo'.hi  (lo' = bf16(x' - hi); ~2^-16 relative)
//   6 terms: hi.hi + hi.mid + mid.hi + hi.lo + lo.hi + mid.mid (~2^-24 relative)
// accumulated in FP32 (v_mfma_f32_32x32x16_bf16) in two chains, hi.hi and the
// smaller products.  With 6 terms they are added in FP64 (their FP32 sum would
// round at 2^-24 of the cross term; in FP64 the marginals of a 97 x 131, d = 7
// pair at eps = 0.05 move from 1.6e-6 to 6.7e-7 of the FP64 oracle's, for 6 %
// more sweep time at 60k); with 3 terms, whose missing products already cost
// 2^-16, in FP32.  Per entry the exponent is formed in FP64 against the row's
// previous potential (a fixed shift, as in the batched sweep); rows whose sum
// under- or overflows are recomputed behind the sweep from FP64 direct distances
// with an online maximum.  The median of the exact FP64 distances (the
// reference's normalisation) comes from two passes that regenerate them
// (distance.hip).
#include <type_traits>

#include "common.h"
#include "distance.h"
#include "fused_problem.h"
#include "underway.h"

namespace wotk {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kFThreads = 256;
constexpr int kFusedMaxSplit = 8;        // column splits per sweep, at most
constexpr int kFusedTargetBlocks = 768;
constexpr int kFusedCUs = 256;
// Waves per SIMD (workgroups per CU) that the registers of a wave's rows, two tiles' products
// and the sums leave room for.  One is enough beside the overlap (us per 20000 x 20000 sweep, before
// it at two waves / now at one): d = 66 with 6 terms 413 / 346, d = 96 485 / 394, d = 120 769 / 527
// (with 3 terms 367 / 320).
constexpr int fused_waves(int terms, int nks) { return nks <= (terms == 3 ? 6 : 4) ? 2 : 1; }
constexpr int kFusedBoxWords = 16 * kFThreads * (2 * kFusedCUs + 1);  // 8-byte words, FP32 sums

// ---------------------------------------------------------------------------
// preparation
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fz_mean_kernel(const double *__restrict__ X, int n_i, const double *__restrict__ Y,
                                                      int n_j, int d, double *__restrict__ mean) {
    __shared__ double red[4];
    const int k = blockIdx.x;
    double acc = 0.0;
    for (int i = threadIdx.x; i < n_i; i += blockDim.x) acc += X[(int64_t)i * d + k];
    for (int j = threadIdx.x; j < n_j; j += blockDim.x) acc += Y[(int64_t)j * d + k];
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) mean[k] = (red[0] + red[1] + red[2] + red[3]) / (n_i + n_j);
}

// x' = (x - mean) / sqrt(median): FP64 copy ([d][n]), FP64 norm, bf16 split into
// npiece pieces (hi, mid, lo), a point's pieces next to each other with K padded
// to kp; n_pad - n points of zeros behind the last
__global__ __launch_bounds__(256) void fz_split_kernel(const double *__restrict__ X, int n, int n_pad, int d, int kp,
                                                       const double *__restrict__ mean,
                                                       const double *__restrict__ median, int npiece,
                                                       __bf16 *__restrict__ pieces, double *__restrict__ xs,
                                                       double *__restrict__ norm) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_pad) return;
    const double sc = 1.0 / sqrt(median[0]);
    double acc = 0.0;
    __bf16 *out = pieces + (int64_t)i * npiece * kp;
    for (int k = 0; k < kp; ++k) {
        const double v = i < n && k < d ? (X[(int64_t)i * d + k] - mean[k]) * sc : 0.0;
        if (i < n && k < d) xs[(int64_t)k * n + i] = v;
        acc = fma(v, v, acc);
        const __bf16 h = (__bf16)(float)v;
        const double r1 = v - (double)(float)h;
        const __bf16 m = (__bf16)(float)r1;
        const double r2 = r1 - (double)(float)m;
        out[k] = h;
        out[kp + k] = m;
        if (npiece > 2) out[2 * kp + k] = (__bf16)(float)r2;
    }
    if (i < n) norm[i] = acc;
}

// ---------------------------------------------------------------------------
// fused sweep: row LSE over recomputed cost tiles, potential update epilogue
// ---------------------------------------------------------------------------
struct FusedArgs {
    const __bf16 *A, *B;         // row and column points, pieces [point][piece][kp]
    const double *na, *nb;       // squared norms of the scaled coordinates
    int n_rows, n_cols, kp;
    const double *h;             // column potentials
    double *pot;                 // row potentials (read as the shift, then updated)
    const double *logw;          // per-row log weight or nullptr -> *logw_dev
    const double *logw_dev;
    double log_n_other, alpha, eps, k;
    double *row_sums;            // row-sum mode: write sum_j R_ij / rs_div, leave pot unchanged
    double *part;                // row sums per column split, split-major
    double rs_div;               // row-sum mode divisor (n_cols: rows of R / J; 1: of R)
    int row_blocks, n_split, per_split, n_tiles;  // units: 128 rows x one split's column tiles
    int whole;                   // one unit per workgroup; else an equal run of tiles each
    unsigned long long *box;     // [workgroup][word][thread]: partial sums handed to the next workgroup
    unsigned tag;                // this launch's mark on them
    int polls;                   // looks at them
    TauTrack tau;                // growth of the potentials (prev null: not tracked)
    double *base;                // what they grow from: u or v
    int opens;                   // the iteration's first sweep
    const int *skip;             // device flag: the launches do nothing when it is set (null: never)
};

// tiles of the units, split-major, rows next: unit (x, y) starts at first_tile
struct FusedUnit {
    int x, t0, len;
    int64_t first;
    int y;
};
__device__ __forceinline__ FusedUnit fused_unit(const FusedArgs &fa, int64_t pos) {
    FusedUnit u;
    const int64_t per = (int64_t)fa.row_blocks * fa.per_split;
    u.y = (int)(pos / per);
    u.t0 = u.y * fa.per_split;
    u.len = min(fa.per_split, fa.n_tiles - u.t0);
    u.x = (int)((pos - u.y * per) / u.len);
    u.first = u.y * per + (int64_t)u.x * u.len;
    return u;
}

// Partial sums passed between workgroups: 32 bits of value and the launch's mark
// in one 8-byte word, so a word is either whole or not yet there and no fence is
// needed.  The wait is bounded: after so many looks (FusedProblem::polls, 128: about
// 0.2 ms) the caller computes the missing part itself, so progress never depends on
// which workgroups the chip holds at once.
__device__ __forceinline__ unsigned long long fused_word(unsigned v, unsigned tag) {
    return (unsigned long long)tag << 32 | v;
}
template <typename T>
__device__ __forceinline__ void fused_send(unsigned long long *box, unsigned tag, const T (&s)[16]) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if constexpr (sizeof(T) == 4) {
            __hip_atomic_store(box + r * kFThreads, fused_word(__float_as_uint(s[r]), tag),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            __hip_atomic_store(box + (2 * r) * kFThreads,
                               fused_word((unsigned)__double2loint(s[r]), tag), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(box + (2 * r + 1) * kFThreads,
                               fused_word((unsigned)__double2hiint(s[r]), tag), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}
template <typename T>
__device__ __forceinline__ bool fused_take(unsigned long long *box, unsigned tag, int polls, T (&s)[16]) {
    constexpr int W = sizeof(T) / 4;
    for (int q = 0; q < polls; ++q) {
        bool there = true;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            unsigned v[W];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const unsigned long long m = __hip_atomic_load(box + (W * r + w) * kFThreads,
                                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                there = there && (unsigned)(m >> 32) == tag;
                v[w] = (unsigned)m;
            }
            if constexpr (W == 1) s[r] = __uint_as_float(v[0]);
            else s[r] = __hiloint2double((int)v[1], (int)v[0]);
        }
        if (__syncthreads_and(there)) return true;
    }
    return false;
}

// 128 rows (32 per wave) x a run of 32-column tiles.  Bound: the matrix cores at the clock they
// sustain.  A tile of a wave takes TERMS * NKS MFMAs and 8 vector instructions for each of its 16
// entries per lane; with 6 terms at d = 50 the products alone (no exponentials) take 383 us of a
// 24576 x 24576 sweep's 393 (1.2 PFLOP/s of padded products, what a large bf16 product reaches).
// So both are in the loop body at once, the products of tile t beside the exponentials of tile
// t - 1 (six stages of four entries, each behind an MFMA); one after the other, with the next
// tile's constants waited for at its start, a sweep took 463 us.  Kept out: three waves per SIMD
// without the overlap (434), column tiles by DMA to LDS two at a time (425).
// Work: the tiles of all units (128 rows x one column split) are dealt out in equal runs, one per
// resident workgroup: 20000 x 20000 has 785 units for 512 places, 291 us as equal runs and 329 as
// whole units in turn.  A run that ends inside a unit leaves the lanes' sums to the next workgroup,
// which goes on from them, so the sums are bit for bit those of one workgroup per unit.  Each
// workgroup takes its last unit (whose rest another waits for) first and the unit it continues last.
// EXACT: FP64 exponential (exp2 of the FP64 exponent) and FP64 lane sums, for
// the row and column sums of the duality-gap pass; otherwise v_exp_f32 of the
// exponent rounded to FP32 and FP32 lane sums (the sweeps)
template <int TERMS, int NKS, bool EXACT>
__global__ __launch_bounds__(kFThreads, fused_waves(TERMS, NKS)) void fused_lse_kernel(FusedArgs fa) {
    constexpr int NP = TERMS == 3 ? 2 : 3;  // pieces per point
    constexpr int KP = NKS * 16;
    constexpr int CHUNKS = NP * KP / 8;      // 16-byte chunks per point
    constexpr int PITCH = NP * KP + 8;       // an odd number of chunks: conflict-free 16-byte reads
    constexpr int NCHUNK = (32 * CHUNKS + kFThreads - 1) / kFThreads;
    constexpr bool RAGGED = 32 * CHUNKS % kFThreads != 0;
    using acc_t = typename std::conditional<EXACT, double, float>::type;
    __shared__ __bf16 bsh[2][32 * PITCH];    // double-buffered column tile
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, kg = (lane >> 5) * 8;
    const double k2 = 2.0 * fa.k;
    if (fa.skip && *fa.skip) return;
    if (fa.tau.prev && fa.opens && blockIdx.x == 0 && tid == 0) {
        if (tau_fired(*fa.tau.prev, fa.tau.tau)) fa.tau.counter[0] += 1;
        *fa.tau.cur = tau_key(-INFINITY);
    }

    const int64_t total = (int64_t)fa.row_blocks * fa.n_tiles;
    int64_t lo, hi;
    if (fa.whole) {
        const int y = (int)blockIdx.x / fa.row_blocks, x = (int)blockIdx.x % fa.row_blocks;
        const int len = min(fa.per_split, fa.n_tiles - y * fa.per_split);
        lo = (int64_t)fa.row_blocks * fa.per_split * y + (int64_t)x * len;
        hi = lo + len;
    } else {
        lo = total * blockIdx.x / gridDim.x;
        hi = total * (blockIdx.x + 1) / gridDim.x;
    }

    constexpr int kWords = 16 * kFThreads * (EXACT ? 2 : 1);
    while (hi > lo) {
        const FusedUnit un = fused_unit(fa, hi - 1);
        const int64_t begin = max(un.first, lo);
        int ta = un.t0 + (int)(begin - un.first);
        const int tb = un.t0 + (int)(hi - un.first);
        const bool ends = hi == un.first + un.len;
        hi = begin;

        // row constants for this lane's 16 accumulator rows: (f_old - |x'|^2) * k
        const int r0 = un.x * 128 + wave * 32;
        double wf[16];
        acc_t s[16];
        bool taken = false;
        if (begin > un.first) {
            int64_t at = (int64_t)blockIdx.x * kWords + tid;
            asm volatile("" : "+v"(at));  // the words' 16 addresses are not kept in registers over the tiles
            taken = fused_take(fa.box + at, fa.tag, fa.polls, s);
            if (!taken) ta = un.t0;
        }
        if (!taken) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = min(r0 + 8 * (r / 4) + 4 * (lane >> 5) + (r % 4), fa.n_rows - 1);
            wf[r] = (fa.pot[row] - fa.na[row]) * fa.k;
        }
        // this wave's 32 rows stay in registers
        bf16x8 afr[NKS][NP];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
            for (int p = 0; p < NP; ++p)
                afr[ks][p] = *reinterpret_cast<const bf16x8 *>(fa.A + ((int64_t)(r0 + lr) * NP + p) * KP + ks * 16 + kg);

        // column tiles stream through two LDS buffers: the next tile's global loads are issued
        // before this tile's products and written to LDS after them
        bf16x8 stage[NCHUNK];
        double h_next, nb_next;
        int col_next;
        auto fetch = [&](int t) {
            const __bf16 *src = fa.B + (int64_t)t * 32 * NP * KP;
#pragma unroll
            for (int u = 0; u < NCHUNK; ++u) {
                const int e = RAGGED ? min(tid + u * kFThreads, 32 * CHUNKS - 1) : tid + u * kFThreads;
                stage[u] = *reinterpret_cast<const bf16x8 *>(src + 8 * e);
            }
            col_next = t * 32 + lr;
            const int c = min(col_next, fa.n_cols - 1);
            h_next = fa.h[c];
            nb_next = fa.nb[c];
        };
        // h - |y'|^2 of the fetched tile's column; columns past the last add exp(-inf) = 0
        auto col_const = [&]() { return col_next < fa.n_cols ? h_next - nb_next : -INFINITY; };
        auto commit = [&](int buf) {
#pragma unroll
            for (int u = 0; u < NCHUNK; ++u) {
                const int e = RAGGED ? min(tid + u * kFThreads, 32 * CHUNKS - 1) : tid + u * kFThreads;
                *reinterpret_cast<bf16x8 *>(&bsh[buf][(e / CHUNKS) * PITCH + (e % CHUNKS) * 8]) = stage[u];
            }
        };
        auto read_b = [&](int buf, int ks, bf16x8 (&b)[NP]) {
            const __bf16 *bt = &bsh[buf][lr * PITCH + ks * 16 + kg];
#pragma unroll
            for (int p = 0; p < NP; ++p) b[p] = *reinterpret_cast<const bf16x8 *>(bt + p * KP);
        };
        // product m of a K step: hi.hi in p0, the smaller ones in p1
        auto product = [&](int m, const bf16x8 *a, const bf16x8 (&b)[NP], floatx16 &p0, floatx16 &p1) {
            if (m == 0) p0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], p0, 0, 0, 0);
            if (m == 1) p1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], p1, 0, 0, 0);
            if (m == 2) p1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], p1, 0, 0, 0);
            if (m == 3) p1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[NP - 1], p1, 0, 0, 0);
            if (m == 4) p1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[NP - 1], b[0], p1, 0, 0, 0);
            if (m == 5) p1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], p1, 0, 0, 0);
        };
        // 6 terms: the chains added in FP64; 3 terms (2^-16 of the cross term already
        // lost to the missing products): one FP32 add and one widening
        auto add_entries = [&](const floatx16 &p0, const floatx16 &p1, double d) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const double xy = TERMS == 6 ? (double)p0[r] + (double)p1[r] : (double)(p0[r] + p1[r]);
                const double y = fma(k2, xy, fma(fa.k, d, wf[r]));
                if constexpr (EXACT) {
                    const double z = y < -1100.0 ? -1100.0 : y;
                    s[r] += exp2_f64(z > 2000.0 ? 2000.0 : z);
                } else {
                    s[r] += __builtin_amdgcn_exp2f((float)y);
                }
            }
        };
        // tile t's products into (n0, n1) beside the exponentials of tile t - 1 in (o0, o1): per K
        // step its share of the 16 entries in six stages, one or two behind each MFMA
        auto step = [&](int buf, floatx16 &n0, floatx16 &n1, const floatx16 &o0, const floatx16 &o1, double d) {
            bf16x8 b[2][NP];
            read_b(buf, 0, b[0]);
            n0 = floatx16{};
            n1 = floatx16{};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                constexpr int kMost = (16 + NKS - 1) / NKS;
                const int rb = 16 * ks / NKS, re = 16 * (ks + 1) / NKS;
                if (ks + 1 < NKS) read_b(buf, ks + 1, b[(ks + 1) & 1]);
                double u[kMost], v[kMost];
                float e[kMost];
#pragma unroll
                for (int m = 0; m < TERMS; ++m) {
                    product(m, afr[ks], b[ks & 1], n0, n1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int st = 6 * m / TERMS; st < 6 * (m + 1) / TERMS; ++st) {
#pragma unroll
                        for (int r = rb; r < re; ++r) {
                            const int i = r - rb;
                            if (st == 0) u[i] = TERMS == 6 ? (double)o0[r] : (double)(o0[r] + o1[r]);
                            if (st == 1 && TERMS == 6) v[i] = (double)o1[r];
                            if (st == 2 && TERMS == 6) u[i] = u[i] + v[i];
                            if (st == 2) v[i] = fma(fa.k, d, wf[r]);
                            if (st == 3) v[i] = fma(k2, u[i], v[i]);
                            if (st == 4) e[i] = (float)v[i];
                            if (st == 4) e[i] = __builtin_amdgcn_exp2f(e[i]);
                            if (st == 5) s[r] += (acc_t)e[i];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        };
        floatx16 pa0, pa1, pb0, pb1;
        __syncthreads();  // the buffers are free
        fetch(ta);
        commit(0);
        double d_old = col_const(), d_cur;
        __syncthreads();
        if constexpr (EXACT) {  // 28 FP64 instructions per entry: the products are the smaller part
            for (int t = ta; t < tb; ++t) {
                const int buf = (t - ta) & 1;
                fetch(min(t + 1, tb - 1));
                pa0 = floatx16{};
                pa1 = floatx16{};
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks) {
                    bf16x8 b[NP];
                    read_b(buf, ks, b);
#pragma unroll
                    for (int m = 0; m < TERMS; ++m) product(m, afr[ks], b, pa0, pa1);
                }
                add_entries(pa0, pa1, d_old);
                commit(buf ^ 1);
                d_old = col_const();
                __syncthreads();
            }
        } else {
            fetch(min(ta + 1, tb - 1));
            pa0 = floatx16{};
            pa1 = floatx16{};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                bf16x8 b[NP];
                read_b(0, ks, b);
#pragma unroll
                for (int m = 0; m < TERMS; ++m) product(m, afr[ks], b, pa0, pa1);
            }
            commit(1);
            d_cur = col_const();
            __syncthreads();
            auto turn = [&](int t, floatx16 &n0, floatx16 &n1, const floatx16 &o0, const floatx16 &o1) {
                const int buf = (t - ta) & 1;
                fetch(min(t + 1, tb - 1));
                __builtin_amdgcn_sched_barrier(0);
                step(buf, n0, n1, o0, o1, d_old);
                commit(buf ^ 1);
                d_old = d_cur;
                d_cur = col_const();
                __syncthreads();
            };
            int t = ta + 1;
            for (; t + 1 < tb; t += 2) {
                turn(t, pb0, pb1, pa0, pa1);
                turn(t + 1, pa0, pa1, pb0, pb1);
            }
            if (t < tb) {
                turn(t, pb0, pb1, pa0, pa1);
                pa0 = pb0;
                pa1 = pb1;
            }
            add_entries(pa0, pa1, d_old);
        }

        if (!ends) {
            int64_t at = ((int64_t)blockIdx.x + 1) * kWords + tid;
            asm volatile("" : "+v"(at));
            fused_send(fa.box + at, fa.tag, s);
            continue;
        }
        // sum over the 32 lanes that share a row set
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const double v = half_wave_sum_dpp((double)s[r]);
            const int row = r0 + 8 * (r / 4) + 4 * (lane >> 5) + (r % 4);
            if (lr == 31 && row < fa.n_rows) fa.part[(int64_t)un.y * fa.n_rows + row] = v;
        }
    }
}

// From the rows' fixed-shift sums S (the splits' added in order): the new potential, or the
// plan's row sum in row-sum mode.  A NaN sum propagates as in the reference's arithmetic.  Rows
// whose sum under- or overflowed are computed again by their workgroup from FP64 direct
// distances of the scaled coordinates ([d][n], read coalesced) with a per-lane online maximum.
// Such a row costs one read of all column points through one CU (8 MB at 20000 x 50), so up to
// four share it.  One launch behind a sweep; clearing a list, adding the splits and repairing by
// three took 20 us of a sweep at 20000 x 20000, this takes 6.  The growth that the tau check looks at
// is kept here too: a launch of its own per iteration made a 3000 x 3000 duality-gap solve 22.9 ms,
// now 21.2.
constexpr int kFinishRows = 32, kFinishThreads = 1024, kFinishWaves = kFinishThreads / 64, kRepairRows = 4;

template <int NB>
__device__ void repair_rows(const FusedArgs &fa, const int *rows, const double *__restrict__ xr,
                            const double *__restrict__ xc, int d, double (*x_sh)[kRepairRows],
                            double (*sg_sh)[kFinishWaves], double (*sd_sh)[kFinishWaves]) {
    const int tid = threadIdx.x;
    for (int e = tid; e < d * NB; e += kFinishThreads) x_sh[e / NB][e % NB] = xr[(int64_t)(e / NB) * fa.n_rows + rows[e % NB]];
    __syncthreads();
    double sg[NB], sd[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        sg[q] = -1.0e6;
        sd[q] = 0.0;
    }
    for (int j = tid; j < fa.n_cols; j += kFinishThreads) {
        double c[NB];
#pragma unroll
        for (int q = 0; q < NB; ++q) c[q] = 0.0;
        for (int t0 = 0; t0 < d; t0 += 8) {
            double v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = xc[(int64_t)min(t0 + u, d - 1) * fa.n_cols + j];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (t0 + u >= d) continue;  // uniform
#pragma unroll
                for (int q = 0; q < NB; ++q) {
                    const double z = x_sh[t0 + u][q] - v[u];
                    c[q] = fma(z, z, c[q]);
                }
            }
        }
        const double hj = fa.h[j];
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const double y = (hj - c[q]) * fa.k;
            if (y > sg[q]) {
                const double ns = ceil(y);
                sd[q] = ldexp(sd[q], (int)(sg[q] - ns));
                sg[q] = ns;
            }
            sd[q] += exp2(y - sg[q]);
        }
    }
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        for (int off = 32; off > 0; off >>= 1) {
            const double og = __shfl_xor(sg[q], off), os = __shfl_xor(sd[q], off);
            const double ng = fmax(sg[q], og);
            sd[q] = ldexp(sd[q], (int)(sg[q] - ng)) + ldexp(os, (int)(og - ng));
            sg[q] = ng;
        }
        if ((tid & 63) == 0) {
            sg_sh[q][tid >> 6] = sg[q];
            sd_sh[q][tid >> 6] = sd[q];
        }
    }
    __syncthreads();
    if (tid < NB) {
        double g = sg_sh[tid][0], v = sd_sh[tid][0];
        for (int w = 1; w < kFinishWaves; ++w) {
            const double ng = fmax(g, sg_sh[tid][w]);
            v = ldexp(v, (int)(g - ng)) + ldexp(sd_sh[tid][w], (int)(sg_sh[tid][w] - ng));
            g = ng;
        }
        const double lse = (g + log2(v)) * kLn2;
        const int row = rows[tid];
        if (fa.row_sums) {
            fa.row_sums[row] = exp(fa.pot[row] / fa.eps + lse) / fa.rs_div;
        } else {
            const double lw = fa.logw ? fa.logw[row] : *fa.logw_dev;
            fa.pot[row] = fa.alpha * fa.eps * (lw + fa.log_n_other - lse);
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(kFinishThreads) void fused_finish_kernel(FusedArgs fa, const double *__restrict__ xr,
                                                                      const double *__restrict__ xc, int d) {
    __shared__ double x_sh[128][kRepairRows];
    __shared__ double sg_sh[kRepairRows][kFinishWaves], sd_sh[kRepairRows][kFinishWaves];
    __shared__ int bad[kFinishRows];
    __shared__ int n_bad;
    const int tid = threadIdx.x;
    if (fa.skip && *fa.skip) return;
    const bool absorb = fa.tau.prev && tau_fired(*fa.tau.prev, fa.tau.tau);
    if (tid == 0) n_bad = 0;
    __syncthreads();
    const int row = blockIdx.x * kFinishRows + tid;
    if (tid < kFinishRows && row < fa.n_rows) {
        if (absorb) fa.base[row] = fa.pot[row];
        double S = 0.0;
        for (int q = 0; q < fa.n_split; ++q) S += fa.part[(int64_t)q * fa.n_rows + row];
        if (isnan(S)) {
            if (fa.row_sums) fa.row_sums[row] = S;
            else fa.pot[row] = S;
        } else if (!(S > 0.0) || isinf(S)) {
            bad[atomicAdd(&n_bad, 1)] = row;
        } else if (fa.row_sums) {  // the shift is the final potential: S = sum_j R_ij
            fa.row_sums[row] = S / fa.rs_div;
        } else {
            const double lse = log(S) - fa.pot[row] / fa.eps;  // ln sum_j exp((h_j - C_ij)/eps)
            const double lw = fa.logw ? fa.logw[row] : *fa.logw_dev;
            fa.pot[row] = fa.alpha * fa.eps * (lw + fa.log_n_other - lse);
        }
    }
    __syncthreads();
    int q = 0;
    for (; q + 1 < n_bad; q += kRepairRows) {
        // a short batch repeats its last row
        __shared__ int batch[kRepairRows];
        if (tid < kRepairRows) batch[tid] = bad[min(q + tid, n_bad - 1)];
        __syncthreads();
        repair_rows<kRepairRows>(fa, batch, xr, xc, d, x_sh, sg_sh, sd_sh);
    }
    if (q < n_bad) repair_rows<1>(fa, bad + q, xr, xc, d, x_sh, sg_sh, sd_sh);
    if (fa.tau.prev && tid < 64) {  // largest growth over the workgroup's rows
        double m = -INFINITY;
        if (tid < kFinishRows && row < fa.n_rows) m = (fa.pot[row] - fa.base[row]) * fa.tau.inv_eps;
        for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
        if (tid == 0) atomicMax(fa.tau.cur, tau_key(m));
    }
}

__global__ __launch_bounds__(1024) void fz_growth_kernel(const double *__restrict__ G, int n, double *__restrict__ logp,
                                                         double *__restrict__ misc) {
    __shared__ double red[16];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        logp[i] = log(G[i]);
        acc += G[i];
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += red[w];
        misc[0] = log(t / n);
    }
}

__global__ void fz_zero_kernel(double *x, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) x[i] = 0.0;
}

// Column splits per sweep: 768 units of 128 rows x one split if the columns give as many, at least
// 8 column tiles and at most kFusedMaxSplit splits
static int fused_splits(int n_rows, int n_cols) {
    const int blocks = (n_rows + 127) / 128;
    const int ntiles = (n_cols + 31) / 32;
    const int want = (kFusedTargetBlocks + blocks - 1) / blocks;
    return std::max(1, std::min(std::min(want, kFusedMaxSplit), ntiles / 8));
}

template <int TERMS, int NKS, bool EXACT>
static void launch_fused(FusedArgs fa, hipStream_t s) {
    // equal runs once every place has a unit (568 units: 79 us, as whole units 82); below that cutting
    // only adds hand-overs (376 units on 256 places: 49 us, whole units 42)
    const int units = fa.row_blocks * fa.n_split;
    const int resident = kFusedCUs * fused_waves(TERMS, NKS);
    const int grid = std::min(units, resident);
    fa.whole = units == grid;
    fused_lse_kernel<TERMS, NKS, EXACT><<<(unsigned)grid, kFThreads, 0, s>>>(fa);
}

template <int TERMS, bool EXACT>
static int fused_sweep(FusedArgs fa, const double *xr, const double *xc, int d, hipStream_t s) {
    fa.row_blocks = (fa.n_rows + 127) / 128;
    fa.n_tiles = (fa.n_cols + 31) / 32;
    fa.per_split = (fa.n_tiles + fused_splits(fa.n_rows, fa.n_cols) - 1) / fused_splits(fa.n_rows, fa.n_cols);
    fa.n_split = (fa.n_tiles + fa.per_split - 1) / fa.per_split;
    switch (fa.kp / 16) {
        case 1: launch_fused<TERMS, 1, EXACT>(fa, s); break;
        case 2: launch_fused<TERMS, 2, EXACT>(fa, s); break;
        case 3: launch_fused<TERMS, 3, EXACT>(fa, s); break;
        case 4: launch_fused<TERMS, 4, EXACT>(fa, s); break;
        case 5: launch_fused<TERMS, 5, EXACT>(fa, s); break;
        case 6: launch_fused<TERMS, 6, EXACT>(fa, s); break;
        case 7: launch_fused<TERMS, 7, EXACT>(fa, s); break;
        default: launch_fused<TERMS, 8, EXACT>(fa, s); break;
    }
    fused_finish_kernel<<<(fa.n_rows + kFinishRows - 1) / kFinishRows, kFinishThreads, 0, s>>>(fa, xr, xc, d);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

// whether a sweep's units outnumber the places of any instance, so that sums are handed over
static bool fused_hands_over(int64_t n_rows, int64_t n_cols) {
    return (n_rows + 127) / 128 * fused_splits((int)n_rows, (int)n_cols) > kFusedCUs;
}

// ---------------------------------------------------------------------------
// the problem helpers shared with the duality-gap schedule
// ---------------------------------------------------------------------------
static void problem_carve(Arena &ar, int64_t I, int64_t J, int64_t d, FusedProblem *fp) {
    const int64_t kp = round_up(d, 16);
    fp->mean = ar.take<double>(d);
    fp->xs = ar.take<double>((size_t)I * d);
    fp->ys = ar.take<double>((size_t)J * d);
    fp->nx = ar.take<double>(I);
    fp->ny = ar.take<double>(J);
    fp->zeros = ar.take<double>(std::max(I, J));
    // padded to whole row blocks (and so to whole column tiles)
    fp->xp = ar.take<__bf16>((size_t)3 * kp * round_up(I, 128));
    fp->yp = ar.take<__bf16>((size_t)3 * kp * round_up(J, 128));
    fp->part = ar.take<double>((size_t)kFusedMaxSplit * std::max(I, J));
    fp->part2 = ar.take<double>((size_t)kFusedMaxSplit * std::max(I, J));
    fp->box_words = fused_hands_over(I, J) || fused_hands_over(J, I) ? kFusedBoxWords : 0;
    fp->box = ar.take<unsigned long long>((size_t)fp->box_words);
    fp->box2 = ar.take<unsigned long long>((size_t)2 * fp->box_words);
    fp->median_ws = ar.take<char>(distance_median_bytes(I, J, true));
}

size_t fused_problem_bytes(int64_t I, int64_t J, int64_t d) {
    Arena ar(nullptr, 0);
    FusedProblem fp;
    problem_carve(ar, I, J, d, &fp);
    return ar.off;
}

int fused_problem_setup(const double *X, const double *Y, int64_t I, int64_t J, int64_t d, int terms,
                        void *workspace, size_t workspace_bytes, FusedProblem *fp, size_t *used, hipStream_t s) {
    WOTK_REQUIRE(I > 0 && J > 0 && d > 0 && I < (1ll << 30) && J < (1ll << 30), "bad shape");
    WOTK_REQUIRE(d <= 128, "the fused solver keeps a 128-dimensional row tile in registers: d <= 128");
    WOTK_REQUIRE(terms == 3 || terms == 6, "terms must be 3 or 6");
    WOTK_REQUIRE(X && Y, "coordinates are required");
    Arena ar(workspace, workspace_bytes);
    problem_carve(ar, I, J, d, fp);
    if (!workspace || !ar.ok) return fail(WOTK_EWORKSPACE, "fused workspace too small");
    *used = ar.off;
    fp->X = X;
    fp->Y = Y;
    fp->I = (int)I;
    fp->J = (int)J;
    fp->d = (int)d;
    fp->kp = (int)round_up(d, 16);
    fp->terms = terms;

    // exact median of the FP64 distances, regenerated per pass
    const DistanceProblem dp{X, Y, (int)I, (int)J, (int)d, 0, 0, {}, {}};
    int rc = distance_median(dp, true, fp->median_ws, nullptr, &fp->median, s);
    if (rc) return rc;

    // scaled, centred coordinates and their bf16 pieces
    fz_mean_kernel<<<(unsigned)d, 256, 0, s>>>(X, (int)I, Y, (int)J, (int)d, fp->mean);
    const int np = terms == 3 ? 2 : 3;
    const int pi = (int)round_up(I, 128), pj = (int)round_up(J, 128);
    fz_split_kernel<<<(unsigned)((pi + 255) / 256), 256, 0, s>>>(X, (int)I, pi, (int)d, fp->kp, fp->mean, fp->median,
                                                                 np, fp->xp, fp->xs, fp->nx);
    fz_split_kernel<<<(unsigned)((pj + 255) / 256), 256, 0, s>>>(Y, (int)J, pj, (int)d, fp->kp, fp->mean, fp->median,
                                                                 np, fp->yp, fp->ys, fp->ny);
    // no word of the boxes carries a launch's mark yet
    if (fp->box_words) {
        fz_zero_kernel<<<1024, 256, 0, s>>>(reinterpret_cast<double *>(fp->box), fp->box_words);
        fz_zero_kernel<<<1024, 256, 0, s>>>(reinterpret_cast<double *>(fp->box2), 2 * fp->box_words);
    }
    fp->tag = 0;
    fz_zero_kernel<<<64, 256, 0, s>>>(fp->zeros, (int)std::max(I, J));
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

// FusedArgs of a sweep over source rows (over_targets = false) or target rows
static FusedArgs problem_args(const FusedProblem &fp, bool target_rows, const double *h, double *pot,
                              const double *logw, const double *logw_dev, double alpha, double eps, double *row_sums,
                              double rs_div, bool second_set) {
    const int nr = target_rows ? fp.J : fp.I, nc = target_rows ? fp.I : fp.J;
    return FusedArgs{target_rows ? fp.yp : fp.xp, target_rows ? fp.xp : fp.yp, target_rows ? fp.ny : fp.nx,
                     target_rows ? fp.nx : fp.ny, nr, nc, fp.kp, h, pot, logw, logw_dev, std::log((double)nc), alpha,
                     eps, kLog2E / eps, row_sums, second_set ? fp.part2 : fp.part, rs_div, 0, 0, 0, 0, 0,
                     second_set ? fp.box2 : fp.box, ++fp.tag, fp.polls, TauTrack{}, nullptr, 0, nullptr};
}

template <bool EXACT>
static int problem_sweep(const FusedProblem &fp, const FusedArgs &fa, bool target_rows, hipStream_t s) {
    const double *xr = target_rows ? fp.ys : fp.xs, *xc = target_rows ? fp.xs : fp.ys;
    return fp.terms == 3 ? fused_sweep<3, EXACT>(fa, xr, xc, fp.d, s) : fused_sweep<6, EXACT>(fa, xr, xc, fp.d, s);
}

int fused_problem_iterate(const FusedProblem &fp, double *f, double *g, const double *logp,
                          const double *logq_dev, double lambda1, double lambda2, double eps, const TauTrack &tau,
                          const int *skip, hipStream_t s) {
    FusedArgs fr = problem_args(fp, false, g, f, logp, nullptr, lambda1 / (lambda1 + eps), eps, nullptr, 1.0,
                                      false);
    fr.tau = tau;
    fr.base = tau.u;
    fr.opens = 1;
    fr.skip = skip;
    int rc = problem_sweep<false>(fp, fr, false, s);
    if (rc) return rc;
    FusedArgs fc = problem_args(fp, true, f, g, nullptr, logq_dev, lambda2 / (lambda2 + eps), eps, nullptr, 1.0,
                                      false);
    fc.tau = tau;
    fc.base = tau.v;
    fc.skip = skip;
    return problem_sweep<false>(fp, fc, true, s);
}

int fused_problem_sums(const FusedProblem &fp, bool over_targets, const double *f, const double *g, double eps,
                       double div, bool exact, double *out, hipStream_t s) {
    // row-sum mode: the shift is the row's own potential, which is not updated
    const double *h = over_targets ? f : g;
    double *pot = const_cast<double *>(over_targets ? g : f);
    const FusedArgs fa = problem_args(fp, over_targets, h, pot, nullptr, nullptr, 0.0, eps, out, div, true);
    return exact ? problem_sweep<true>(fp, fa, over_targets, s) : problem_sweep<false>(fp, fa, over_targets, s);
}

}  // namespace wotk

using namespace wotk;

// solver state of the fixed-iteration schedule beside the problem buffers
struct FzState {
    double *f, *g, *logp, *misc;
};

static size_t fz_state_carve(Arena &ar, int64_t I, int64_t J, FzState *st) {
    st->f = ar.take<double>(I);
    st->g = ar.take<double>(J);
    st->logp = ar.take<double>(I);
    st->misc = ar.take<double>(8);
    return ar.off;
}

extern "C" size_t wotk_fused_workspace_size(int64_t I, int64_t J, int64_t d) {
    Arena ar(nullptr, 0);
    FzState st;
    return fused_problem_bytes(I, J, d) + 256 + fz_state_carve(ar, I, J, &st);
}

static int stablev2_coords_call(const double *X, const double *Y, int64_t I, int64_t J, int64_t d, const double *G,
                                double lambda1, double lambda2, double epsilon, int64_t scaling_iter,
                                double epsilon0, int64_t extra_iter, int64_t inner_iter_max, int32_t terms,
                                double *f_out, double *g_out, double *row_sums, double *median_out,
                                void *workspace, size_t workspace_bytes, int32_t polls, wotk_stats *stats,
                                hipStream_t s) {
    const UnderWay here;
    WOTK_REQUIRE(scaling_iter >= 0 && extra_iter >= 0 && scaling_iter + extra_iter > 0 && inner_iter_max > 0,
                 "bad iteration counts");
    WOTK_REQUIRE(G != nullptr, "G is required");
    FusedProblem fp;
    if (polls >= 0) fp.polls = polls;
    size_t used = 0;
    int rc = fused_problem_setup(X, Y, I, J, d, terms, workspace, workspace_bytes, &fp, &used, s);
    if (rc) return rc;
    used = (used + 255) & ~size_t(255);
    Arena ar(static_cast<char *>(workspace) + used, workspace_bytes > used ? workspace_bytes - used : 0);
    FzState w;
    fz_state_carve(ar, I, J, &w);
    if (!ar.ok) return fail(WOTK_EWORKSPACE, "fused workspace too small");
    if (median_out) WOTK_HIP(hipMemcpyAsync(median_out, fp.median, sizeof(double), hipMemcpyDeviceToDevice, s));
    fz_zero_kernel<<<64, 256, 0, s>>>(w.f, (int)I);
    fz_zero_kernel<<<64, 256, 0, s>>>(w.g, (int)J);
    fz_growth_kernel<<<1, 1024, 0, s>>>(G, (int)I, w.logp, w.misc);
    WOTK_LAUNCH_CHECK();

    auto reg = [&](int64_t m) { return (epsilon0 - epsilon) * std::exp(-(double)m) + epsilon; };
    hipEvent_t ev[2] = {nullptr, nullptr};
    struct Events {
        hipEvent_t *e;
        ~Events() {
            for (int i = 0; i < 2; ++i)
                if (e[i]) (void)hipEventDestroy(e[i]);
        }
    } guard{ev};
    WOTK_HIP(hipEventCreate(&ev[0]));
    WOTK_HIP(hipEventCreate(&ev[1]));
    WOTK_HIP(hipEventRecord(ev[0], s));
    const int64_t n_iter = scaling_iter + extra_iter;
    for (int64_t it = 0; it < n_iter; ++it) {
        const double eps = it < scaling_iter ? reg(it / inner_iter_max) : reg(scaling_iter / inner_iter_max);
        rc = fused_problem_iterate(fp, w.f, w.g, w.logp, w.misc, lambda1, lambda2, eps, TauTrack{}, nullptr, s);
        if (rc) return rc;
    }
    WOTK_HIP(hipEventRecord(ev[1], s));
    const double e_end = reg(scaling_iter / inner_iter_max);
    if (row_sums) {
        // the returned plan is built with the eps after the last iteration
        rc = fused_problem_sums(fp, false, w.f, w.g, e_end, (double)J, false, row_sums, s);
        if (rc) return rc;
    }
    if (f_out) WOTK_HIP(hipMemcpyAsync(f_out, w.f, sizeof(double) * I, hipMemcpyDeviceToDevice, s));
    if (g_out) WOTK_HIP(hipMemcpyAsync(g_out, w.g, sizeof(double) * J, hipMemcpyDeviceToDevice, s));
    WOTK_HIP(hipStreamSynchronize(s));
    float ms = 0.f;
    WOTK_HIP(hipEventElapsedTime(&ms, ev[0], ev[1]));
    if (stats) {
        *stats = wotk_stats{};
        stats->iterations = n_iter;
        stats->sweeps = 2 * n_iter;
        stats->sweep_ms = ms;
        stats->epsilon_final = e_end;
    }
    return WOTK_OK;
}

extern "C" int wotk_transport_stablev2_coords(const double *X, const double *Y, int64_t I, int64_t J, int64_t d,
                                              const double *G, double lambda1, double lambda2, double epsilon,
                                              int64_t scaling_iter, double tau, double epsilon0, int64_t extra_iter,
                                              int64_t inner_iter_max, int32_t terms, double *f_out, double *g_out,
                                              double *row_sums, double *median_out, void *workspace,
                                              size_t workspace_bytes, wotk_stats *stats, void *stream) {
    (void)tau;
    return stablev2_coords_call(X, Y, I, J, d, G, lambda1, lambda2, epsilon, scaling_iter, epsilon0, extra_iter,
                                inner_iter_max, terms, f_out, g_out, row_sums, median_out, workspace,
                                workspace_bytes, -1, stats, (hipStream_t)stream);
}

extern "C" int wotk_probe_stablev2_coords_limits(const double *X, const double *Y, int64_t I, int64_t J, int64_t d,
                                                 const double *G, double lambda1, double lambda2, double epsilon,
                                                 int64_t scaling_iter, double tau, double epsilon0, int64_t extra_iter,
                                                 int64_t inner_iter_max, int32_t terms, double *f_out, double *g_out,
                                                 double *row_sums, double *median_out, void *workspace,
                                                 size_t workspace_bytes, wotk_stats *stats, void *stream,
                                                 int32_t polls) {
    (void)tau;
    return stablev2_coords_call(X, Y, I, J, d, G, lambda1, lambda2, epsilon, scaling_iter, epsilon0, extra_iter,
                                inner_iter_max, terms, f_out, g_out, row_sums, median_out, workspace,
                                workspace_bytes, polls, stats, (hipStream_t)stream);
}
