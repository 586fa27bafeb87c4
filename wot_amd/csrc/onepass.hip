// A whole Sinkhorn iteration over ONE read of the stored cost.
//
// Two sweeps (f over C, then g over C^T) read 8 bytes per entry and evaluate every
// exponential twice.  The two are the same numbers: with f_i just updated,
//   sum_i exp((f_i - C_ij)/eps) = exp(-g_j/eps) sum_i E_ij w_i,
//   E_ij = 2^(k (g_j - C_ij) - N_i),  w_i = 2^(k f_i + N_i),  k = log2(e)/eps,
// where E_ij are the row pass's own terms and N_i = rint(-k f_i(old)) is the row's
// integer shift.  So a workgroup that holds whole rows in registers can finish f_i
// and then add the row's terms, times one factor, to its column sums: half the
// HBM bytes and half the exponentials.
//
// Up to 15 waves own all columns, thread t of their T the groups of four at 4 (t + T c)
// (as many waves as fill the last group: at most a wave's worth of lanes idles), so a
// column's running sum stays in one register of one thread for all the rows of
// the workgroup (one workgroup per CU, rows dealt round robin).  A step takes R rows:
//   exponentials of the current rows | wave sums to LDS | barrier |
//   column sums of the PREVIOUS rows
// while one more wave turns the sums of the previous step into f_i and w_i (their
// logarithm and exponential, and the registers these need, stay out of the other
// waves).  One barrier per step; the loads of the next one or two steps are in flight
// throughout.  The column shifts k g_j lie in LDS (FP64).  Exponents are formed in
// FP64 and split exactly, 2^y = ldexp(exp2(y - rint y), rint y - N_i).
//
// Sums.  A column's terms span many binades; in FP32 every term under 2^-25 of the
// running sum is dropped, always downwards: the sums came out 4e-8 low and the plan
// 5e-8 high at 10000 x 8001.  So the columns are summed in FP64 (and the rows, four
// terms at a time): a convert and an FP64 multiply-add per entry beside the 11
// instructions of the term.
//
// Range.  A row whose sum leaves [2^-40, 2^40] or whose weight exceeds 2^40 (its
// potential moved far: a large change of eps, an outlier cell) is left out of the
// column sums (weight 0, terms kept finite) and redone at the end of the workgroup
// with its true maximum.  Terms below 2^-126 are lost: at most I 2^-126 w_i, so a
// column sum of at least 2^-30 has lost less than 2^-28 of itself; smaller (or
// overflowed) columns are redone from C^T with an online maximum.  A sum that is no
// number comes from a NaN in the inputs and stays one.
#include <algorithm>
#include <cmath>

#include "onepass.h"

namespace wotk {
namespace {

constexpr int kT = 1024;           // most threads
constexpr int kW = kT / 64;        // most waves; the last one finishes rows
constexpr int kCT = kT - 64;       // most threads that own columns; LDS stride of their shifts
constexpr int kMaxRows = 8192;     // rows per workgroup (bad-row bits in LDS)
constexpr int kMaxChunks = 5;      // groups of four columns per thread (registers; LDS 30 KB each)
constexpr double kRowLo = 9.094947017729282e-13, kRowHi = 1.099511627776e12;  // 2^-40, 2^40
constexpr double kWeightHi = 1.099511627776e12;  // 2^40
constexpr double kColLo = 9.313225746154785e-10, kColHi = 1.2379400392853803e27;  // 2^-30, 2^90

struct RowArgs {
    const float *C;
    int64_t ldc;
    int n_i, n_j;
    double *f;
    const double *g;
    const double *logp;
    double log_nj, alpha, eps, k;
    float *part;
    int ld_part;
    TauTrack tau;
    const int *skip;
};

typedef const __attribute__((address_space(4))) double *ScalarPtr;

// workgroup barrier that orders LDS only: loads from global memory stay in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));

template <int NC, int R>
struct RowBuf {
    f4 v[R][NC];
};

__device__ __forceinline__ int first_row(int it, int R) { return ((int)blockIdx.x + it * (int)gridDim.x) * R; }

__device__ __forceinline__ int shift_of(double kf) {  // N_i; any integer serves, a non-finite potential takes 0
    return fabs(kf) < 1e9 ? (int)rint(-kf) : 0;
}

// LDS of one workgroup
template <int R>
struct RowShared {
    double wsum[2][4][kW];        // wave sums of a step's rows (a wave without columns: 0)
    double wrow[2][R];            // w_i of a step's rows
    unsigned bad[kMaxRows / 32];  // rows of this workgroup to redo
    double red[kW];
};

// ---- the waves that own columns ----
template <int NC, int R, int DEPTH>
struct RowPass {
    const RowArgs &ra;
    RowShared<R> &sh;
    const double2 *h;
    const int tid, lane, wave, n_steps;
    const int chunk;           // columns per chunk: 4 T
    const unsigned t4, last4;  // first column of the thread in a chunk / in the last chunk (clamped to the row)
    d4 acc[NC];                // column sums
    double f_next[R];          // wave-uniform: old potentials of the next step's rows
    RowBuf<NC, R> b0, b1, b2, b3;

    // column shift pairs of chunk c: two 16-byte reads, 16 bytes apart between lanes
    __device__ void shifts(int c, double2 &a, double2 &b) const {
        a = h[c * 2 * kCT + tid];
        b = h[c * 2 * kCT + kCT + tid];
    }

    // Every lane loads on every step, so that the waits count the same loads on every
    // path: threads without columns repeat the last group, steps past the end the last rows.
    __device__ void load(RowBuf<NC, R> &o, int it) const {
        const int r0 = first_row(min(it, n_steps - 1), R);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float *p = ra.C + (int64_t)min(r0 + r, ra.n_i - 1) * ra.ldc;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                o.v[r][c] = __builtin_nontemporal_load(
                    reinterpret_cast<const f4 *>(p + c * chunk + (c < NC - 1 ? t4 : last4)));
        }
    }

    // scalar loads: a vector load here would wait for the rows in flight.  (A row's old potential is
    // read before its own workgroup stores the new one, so a cached line serves.)
    __device__ void load_f(int it) {
        const int r0 = first_row(min(it, n_steps - 1), R);
#pragma unroll
        for (int r = 0; r < R; ++r) f_next[r] = ((ScalarPtr)ra.f)[min(r0 + r, ra.n_i - 1)];
    }

    // the rows' terms in place of their costs, their sums to LDS
    __device__ void terms(RowBuf<NC, R> &cur, int it) {
        int N[R];
        double s[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            N[r] = __builtin_amdgcn_readfirstlane(shift_of(ra.k * f_next[r]));
            s[r] = 0.0;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            double2 ha, hb;
            shifts(c, ha, hb);
            const double hk[4] = {ha.x, ha.y, hb.x, hb.y};
#pragma unroll
            for (int r = 0; r < R; ++r) {
                f4 e;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const double y = fma(-ra.k, (double)cur.v[r][c][q], hk[q]);
                    const double n = rint(y);
                    // saturating: a cost far above 2^31 / k is a term of 0, not a wrapped exponent
                    e[q] = ldexpf(__builtin_amdgcn_exp2f((float)(y - n)), __builtin_elementwise_sub_sat((int)n, N[r]));
                }
                float t = (e[0] + e[1]) + (e[2] + e[3]);
                // An infinite cost (y - n is no number) is a term of 0; a term that overflows stays finite:
                // its row's sum tells that it has to be redone, and its weight in the columns is 0.
                if (__builtin_expect(!(t < INFINITY), 0)) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (fma(-ra.k, (double)cur.v[r][c][q], hk[q]) == -INFINITY) e[q] = 0.f;
                        if (e[q] == INFINITY) e[q] = 3.0e38f;
                    }
                    t = (e[0] + e[1]) + (e[2] + e[3]);
                }
                s[r] += (double)t;
                cur.v[r][c] = e;
            }
            // keep the next chunk's shifts and exponents out of this one's registers
            __builtin_amdgcn_sched_barrier(0);
        }
        load_f(it + 1);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double t = wave_sum_dpp(s[r]);
            if (lane == 63) sh.wsum[it & 1][r][wave] = t;
        }
    }

    __device__ void add_columns(const RowBuf<NC, R> &prev, int it) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double w = sh.wrow[it & 1][r];
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[c][q] = fma((double)prev.v[r][c][q], w, acc[c][q]);
        }
        // summed here: sunk below the next steps, the sums would keep every step's terms in registers
#pragma unroll
        for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(acc[c]));
    }

    // one step (step 0 adds a zeroed buffer with weight 0)
    __device__ void step(const RowBuf<NC, R> &prev, RowBuf<NC, R> &cur, RowBuf<NC, R> &ahead, int it) {
        load(ahead, it + DEPTH);
        terms(cur, it);
        lds_barrier();
        add_columns(prev, it + 1);  // parity of it - 1
    }

    // the first rows' loads, before anything else
    __device__ void begin() {
        load(b0, 0);
        if (DEPTH > 1) load(b1, 1);
        load_f(0);
    }

    // n steps, n + 1 barriers; buffers in turn: previous terms, current rows, one or two steps ahead
    __device__ void run(int n) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            acc[c] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int r = 0; r < R; ++r) (DEPTH > 1 ? b3 : b2).v[r][c] = f4{0.f, 0.f, 0.f, 0.f};
        }
        int it = 0;
        if constexpr (DEPTH > 1) {
            for (; it + 4 <= n; it += 4) {
                step(b3, b0, b2, it);
                step(b0, b1, b3, it + 1);
                step(b1, b2, b0, it + 2);
                step(b2, b3, b1, it + 3);
            }
            const int left = n - it;  // 0 .. 3
            if (left > 0) step(b3, b0, b2, it);
            if (left > 1) step(b0, b1, b3, it + 1);
            if (left > 2) step(b1, b2, b0, it + 2);
            lds_barrier();
            if (left == 0) add_columns(b3, n - 1);
            else if (left == 1) add_columns(b0, n - 1);
            else if (left == 2) add_columns(b1, n - 1);
            else add_columns(b2, n - 1);
        } else {
            for (; it + 3 <= n; it += 3) {
                step(b2, b0, b1, it);
                step(b0, b1, b2, it + 1);
                step(b1, b2, b0, it + 2);
            }
            const int left = n - it;  // 0 .. 2
            if (left > 0) step(b2, b0, b1, it);
            if (left > 1) step(b0, b1, b2, it + 1);
            lds_barrier();
            if (left == 0) add_columns(b2, n - 1);
            else if (left == 1) add_columns(b0, n - 1);
            else add_columns(b1, n - 1);
        }
    }
};

// ---- the wave that finishes rows: 16 lanes per row, up to four rows at once ----
template <int R>
__device__ void finish_rows(const RowArgs &ra, RowShared<R> &sh, int n) {
    const int lane = threadIdx.x & 63, r = lane >> 4;
    const bool absorb = ra.tau.prev && tau_fired(*ra.tau.prev, ra.tau.tau);
    if (ra.tau.prev && blockIdx.x == 0 && lane == 0) {
        if (absorb) ra.tau.counter[0] += 1;
        *ra.tau.cur = tau_key(-INFINITY);
    }
    for (int it = 0; it < n; ++it) {
        const int row = first_row(it, R) + r;
        const bool mine = r < R && row < ra.n_i;
        const int rw = mine ? row : 0;
        const double fo = ra.f[rw], lp = ra.logp[rw];
        lds_barrier();
        const double S = row_sum_dpp(sh.wsum[it & 1][r][lane & 15]);  // in the last lane of each 16
        const int N = shift_of(ra.k * fo);
        const double lse2 = log2(S) + (double)N;
        const double fn = ra.alpha * ra.eps * (lp + ra.log_nj - lse2 * kLn2);
        const double w = exp2(ra.k * fn + (double)N);
        if ((lane & 15) == 15 && r < R) {
            const bool out = S < kRowLo || S > kRowHi || w > kWeightHi;
            if (mine && absorb) ra.tau.u[row] = fo;
            if (mine && out) atomicOr(&sh.bad[(it * R + r) >> 5], 1u << ((it * R + r) & 31));
            if (mine && !out) ra.f[row] = fn;
            sh.wrow[it & 1][r] = mine && !out ? w : 0.0;
        }
    }
    lds_barrier();
}

// rows outside the safe range, from their true maximum, added to the column sums already
// written; every thread of the workgroup takes part
template <int NC, int R>
__device__ void redo_bad(const RowArgs &ra, RowShared<R> &sh, const double2 *h, int n, int waves, float *out) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n4 = (ra.n_j + 3) >> 2, ct = (waves - 1) * 64;
    for (int b = 0; b < n * R; ++b) {
        if (!((sh.bad[b >> 5] >> (b & 31)) & 1u)) continue;  // uniform
        const int row = first_row(b / R, R) + b % R;
        const float *p = ra.C + (int64_t)row * ra.ldc;
        // exponent of column 4 (t + c T) + q; threads without columns: none
        auto exponent = [&](int c, int q) {
            const double2 hk = h[c * 2 * kCT + (q >> 1) * kCT + tid];
            return fma(-ra.k, (double)p[4 * (tid + c * ct) + q], q & 1 ? hk.y : hk.x);
        };
        const int chunks = tid >= ct ? 0 : tid + (NC - 1) * ct < n4 ? NC : NC - 1;
        double m = -1.0e300;
        for (int c = 0; c < chunks; ++c)
            for (int q = 0; q < 4; ++q) m = fmax(m, exponent(c, q));
        m = wave_max(m);
        __syncthreads();
        if (lane == 0) sh.red[wave] = m;
        __syncthreads();
        for (int w = 0; w < waves; ++w) m = fmax(m, sh.red[w]);
        const double top = ceil(m);
        double s = 0.0;
        for (int c = 0; c < chunks; ++c)
            for (int q = 0; q < 4; ++q) s += (double)__builtin_amdgcn_exp2f((float)(exponent(c, q) - top));
        s = wave_sum(s);
        __syncthreads();
        if (lane == 0) sh.red[wave] = s;
        __syncthreads();
        s = 0.0;
        for (int w = 0; w < waves; ++w) s += sh.red[w];
        const double fn = ra.alpha * ra.eps * (ra.logp[row] + ra.log_nj - (log2(s) + top) * kLn2);
        if (tid == 0) ra.f[row] = fn;
        for (int c = 0; c < chunks; ++c)
            for (int q = 0; q < 4; ++q) out[4 * (tid + c * ct) + q] += (float)exp2(exponent(c, q) + ra.k * fn);
    }
}

template <int NC, int R, int DEPTH, int T>
__global__ __launch_bounds__(T) void one_pass_rows_kernel(RowArgs ra) {
    extern __shared__ __align__(16) double2 h_lds[];
    __shared__ RowShared<R> sh;
    if (ra.skip && *ra.skip) return;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int waves = (int)blockDim.x >> 6, ct = (waves - 1) * 64;
    const int n4 = (ra.n_j + 3) >> 2;
    const int n_groups = (ra.n_i + R - 1) / R;
    const int n = (n_groups - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;  // steps, at least 1
    RowPass<NC, R, DEPTH> rp{ra, sh, h_lds, tid, tid & 63, wave, n, 4 * ct, 4u * tid,
                             4u * min(tid, n4 - 1 - (NC - 1) * ct)};
    const bool owner = wave < waves - 1;
    if (owner) rp.begin();
    for (int q = tid; q < kMaxRows / 32; q += blockDim.x) sh.bad[q] = 0u;
    if (tid < 2 * R) sh.wrow[tid / R][tid % R] = 0.0;
    for (int q = tid; q < 8 * kW; q += blockDim.x) sh.wsum[q / (4 * kW)][(q / kW) % 4][q % kW] = 0.0;
    // column shifts k g_j (padding columns and lanes without columns: far below every other)
    if (owner) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            double v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = 4 * (tid + c * ct) + q;
                const double x = ra.k * ra.g[min(j, ra.n_j - 1)];
                v[q] = j >= ra.n_j || x < -1.0e9 ? -1.0e9 : x;
            }
            h_lds[c * 2 * kCT + tid] = make_double2(v[0], v[1]);
            h_lds[c * 2 * kCT + kCT + tid] = make_double2(v[2], v[3]);
        }
    }
    lds_barrier();
    float *out = ra.part + (int64_t)blockIdx.x * ra.ld_part;
    if (owner) {
        rp.run(n);
#pragma unroll
        for (int c = 0; c < NC; ++c)
            if (tid + c * ct < n4)
                *reinterpret_cast<f4 *>(out + c * 4 * ct + 4 * tid) = __builtin_convertvector(rp.acc[c], f4);
    } else {
        finish_rows<R>(ra, sh, n);
    }
    __syncthreads();
    redo_bad<NC, R>(ra, sh, h_lds, n, waves, out);
}

struct ColArgs {
    const float *CT;
    int64_t ldct;
    int n_i, n_j;
    const double *f;
    double *g;
    const double *logq_dev;
    double log_ni, alpha, eps, k;
    const float *part;
    int ld_part, n_part;
    TauTrack tau;
    const int *skip;
};

// g from the workgroups' column sums: 64 columns per workgroup, 16 threads per
// column over the partials, combined in a fixed order.
__global__ __launch_bounds__(kT) void one_pass_cols_kernel(ColArgs ca) {
    __shared__ double red[kW][64];
    __shared__ int bad[64];
    __shared__ int n_bad;
    __shared__ double wred[kW];
    if (ca.skip && *ca.skip) return;
    const bool absorb = ca.tau.prev && tau_fired(*ca.tau.prev, ca.tau.tau);
    const int c = threadIdx.x & 63, p = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + c;
    if (threadIdx.x == 0) n_bad = 0;
    double s = 0.0;
    if (j < ca.n_j) {
        const float *src = ca.part + j;
#pragma unroll 8
        for (int b = p; b < ca.n_part; b += kW) s += (double)src[(int64_t)b * ca.ld_part];
    }
    red[p][c] = s;
    __syncthreads();
    if (p == 0 && j < ca.n_j) {
        for (int q = 1; q < kW; ++q) s += red[q][c];
        if (absorb) ca.tau.v[j] = ca.g[j];
        if (s < kColLo || s > kColHi) {
            bad[atomicAdd(&n_bad, 1)] = j;
        } else {
            const double lse = log(s) - ca.g[j] / ca.eps;
            ca.g[j] = ca.alpha * ca.eps * (*ca.logq_dev + ca.log_ni - lse);
        }
    }
    __syncthreads();
    const int nb = n_bad;
    for (int q = 0; q < nb; ++q) {  // from C^T, with the true maximum
        const int col = bad[q];
        const float *row = ca.CT + (int64_t)col * ca.ldct;
        double m = -1.0e300;
        for (int i = threadIdx.x; i < ca.n_i; i += kT) m = fmax(m, (ca.f[i] - (double)row[i]) * ca.k);
        m = wave_max(m);
        if (c == 0) wred[p] = m;
        __syncthreads();
        for (int w = 0; w < kW; ++w) m = fmax(m, wred[w]);
        __syncthreads();
        const double sh = ceil(m);
        double t = 0.0;
        for (int i = threadIdx.x; i < ca.n_i; i += kT)
            t += (double)__builtin_amdgcn_exp2f((float)((ca.f[i] - (double)row[i]) * ca.k - sh));
        t = wave_sum(t);
        if (c == 0) wred[p] = t;
        __syncthreads();
        if (threadIdx.x == 0) {
            t = 0.0;
            for (int w = 0; w < kW; ++w) t += wred[w];
            ca.g[col] = ca.alpha * ca.eps * (*ca.logq_dev + ca.log_ni - (log2(t) + sh) * kLn2);
        }
        __syncthreads();
    }
    if (ca.tau.prev) {  // largest growth over this workgroup's columns and its share of the rows
        double m = -INFINITY;
        if (p == 0 && j < ca.n_j) m = (ca.g[j] - ca.tau.v[j]) * ca.tau.inv_eps;
        for (int i = blockIdx.x * kT + threadIdx.x; i < ca.n_i; i += (int)gridDim.x * kT)
            m = fmax(m, (ca.f[i] - ca.tau.u[i]) * ca.tau.inv_eps);
        m = wave_max(m);
        __syncthreads();
        if (c == 0) wred[p] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < kW; ++w) m = fmax(m, wred[w]);
            atomicMax(ca.tau.cur, tau_key(m));
        }
    }
}

constexpr int kCus = 256;

// columns per thread and waves of a width: the fewest groups of four that 15 waves cover
int chunks_of(int64_t J) { return (int)((J + 4 * kCT - 1) / (4 * kCT)); }

int waves_of(int64_t J) {
    const int nc = chunks_of(J);
    return (int)((J + 3) / 4 + 64 * nc - 1) / (64 * nc) + 1;
}

int rows_per_step(int64_t J) {
    const int nc = chunks_of(J);
    return nc == 1 ? 4 : nc == 2 || (nc == 3 && waves_of(J) <= 12) ? 2 : 1;
}

// one workgroup per CU; narrow ones share it up to 16 waves (and 4 x 33 KB of LDS)
int grid_of(int64_t I, int64_t J) {
    const int r = rows_per_step(J), per_cu = std::min(4, kW / waves_of(J));
    return (int)std::min<int64_t>((int64_t)kCus * std::max(1, per_cu), (I + r - 1) / r);
}

template <int NC, int R, int DEPTH, int T>
int launch_rows(const RowArgs &ra, int grid, hipStream_t s) {
    constexpr int lds = NC * 2 * kCT * (int)sizeof(double2);
    // above 64 KB of LDS the runtime has to be told
    WOTK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(one_pass_rows_kernel<NC, R, DEPTH, T>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    one_pass_rows_kernel<NC, R, DEPTH, T><<<grid, waves_of(ra.n_j) * 64, lds, s>>>(ra);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

}  // namespace

// Where one read of C beats two sweeps over C and C^T (us per iteration, two sweeps against one
// read): 2900 x 2900 19.2 / 17.7, 9000 x 1001 24.8 / 22.6, 600 x 19000 42.4 / 30.5, 6000 x 5000
// 43.7 / 33.1, 10000 x 8001 105 / 65.5, 15000 x 15000 275 / 155, 19000 x 19000 (the widest rows whose
// sums fit in registers) 439 / 236.  The line at 2^23 entries is not a crossing of times: it is
// where results change.  Up to it a pair's potentials have the two sweeps' bits, by the resident
// solver or, with a side it does not take, by the sweeps themselves (9000 x 800: 24.9); above it
// columns are summed in FP64.
bool one_pass_fits(int64_t I, int64_t J) {
    if (chunks_of(J) > kMaxChunks || I > (int64_t)kCus * kMaxRows) return false;
    return I * J >= (1ll << 23);
}

size_t one_pass_partials(int64_t I, int64_t J) { return (size_t)grid_of(I, J) * round_up(J, 4); }

int one_pass_iterate(const OnePass &op, double lambda1, double lambda2, double eps, hipStream_t s) {
    const double k = kLog2E / eps;
    const int grid = grid_of(op.n_i, op.n_j), ld = (int)round_up(op.n_j, 4);
    const RowArgs ra{op.C, op.ldc, op.n_i, op.n_j, op.f, op.g, op.logp, std::log((double)op.n_j),
                     lambda1 / (lambda1 + eps), eps, k, op.part, ld, op.tau, op.skip};
    const bool narrow = waves_of(op.n_j) <= 12;
    int rc;
    switch (chunks_of(op.n_j)) {
        case 1: rc = launch_rows<1, 4, 2, 1024>(ra, grid, s); break;
        case 2: rc = launch_rows<2, 2, 2, 1024>(ra, grid, s); break;
        case 3: rc = narrow ? launch_rows<3, 2, 1, 768>(ra, grid, s) : launch_rows<3, 1, 2, 1024>(ra, grid, s); break;
        case 4: rc = launch_rows<4, 1, 2, 1024>(ra, grid, s); break;
        default: rc = launch_rows<5, 1, 1, 1024>(ra, grid, s); break;
    }
    if (rc) return rc;
    const ColArgs ca{op.CT, op.ldct, op.n_i, op.n_j, op.f, op.g, op.logq_dev, std::log((double)op.n_i),
                     lambda2 / (lambda2 + eps), eps, k, op.part, ld, grid, op.tau, op.skip};
    one_pass_cols_kernel<<<(op.n_j + 63) / 64, kT, 0, s>>>(ca);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

}  // namespace wotk
