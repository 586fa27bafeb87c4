// Whole solves of small pairs in one persistent launch.
//
// Below about 8 million entries a sweep's data (C or C^T, FP32) takes under 10 us to
// read and half of that to compute, but every sweep of the launched solver pays a kernel
// boundary, reloads the cost from cache, and the duality-gap solver adds a third
// launch per iteration for its tau check and a host round trip per five.  Here the
// cost stays in registers for the whole solve (C and C^T of 8.4 million entries are 67 of
// the chip's 128 MB) and the workgroups pass the potentials to each other.
// Per iteration, launched -> resident: 300 x 400 8.4 -> 5.1 us (the exchange alone is
// 4.5), 2000 x 2500 15.8 -> 11.0, 2749 x 3001 20.0 -> 14.5; the duality-gap map of
// 2749 x 3001, checks included, 15.2 -> 9.7 ms.
//
// Arithmetic.  The sweep's own (lse_rows_kernel<4, 256>): a team of 256 threads per
// row, thread t the columns 4 t + 1024 m, running per-lane maximum, lanes merged by
// the same xor tree and waves in order, so the potentials are the same bits.
//
// Exchange.  A potential travels as its 8 bytes in one of two buffers (parity of the
// iteration); a buffer not yet written holds kEmpty, a NaN pattern no result has, and
// readers poll the values themselves: one store and one load stand between a producer
// and a consumer, no counter, no barrier.  Reuse is safe by data flow: only workgroups with rows of
// C read g_n, and each publishes its part of f_n+1 after that, so whoever has all of f_n+1 knows
// that g_n has been read and may empty its part of it; it waits for those stores before it
// publishes its part of g_n+1, which every poller of g_n+2 has read.  The same holds for f_n, its
// readers (the workgroups with rows of C^T) and g_n.  (A workgroup without rows on a side, such as
// 25 of 100 at 300 x 400, publishes nothing there that could tell that it has read the other
// side, so it does not read it.)  The tau check's maxima and the gap sums are read by every workgroup
// and published by every workgroup, in three buffers: whoever has all of one step's has proof that
// everybody has read the step before, and empties that one's buffer, the next step's, before it
// publishes its own.  Every workgroup adds them up in the same order and takes the same decisions.
// tests/test_resident_exchange.py holds a model of this that delays workgroups at will.
//
// Progress.  The workgroups fit on an idle device all at once (the occupancy is asked), one such
// launch of a process is under way at a time (underway.h), and whatever else runs ends by itself, so
// all of them get their CUs.  Every wait is bounded (ResidentLimits): where CUs stay taken, by another
// process or a long kernel, a workgroup gives up and raises a flag that ends all others' waits, and
// the caller solves again by launched sweeps.  (A cooperative launch would see to residence by itself,
// but its queue comes on top of the process's four: with 8 threads at 300 x 400, solves beside it
// took 14.5 us per iteration each, beside the plain launch 2.5, 2.4 by sweeps alone.)
#include <algorithm>
#include <cmath>

#include "resident.h"

namespace wotk {
namespace {

typedef unsigned long long u64;
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kT = 1024;                 // threads: four teams of 256
constexpr int kTeams = kT / 256;
constexpr int kMaxWg = 256;              // one workgroup per CU
constexpr int kMaxSlots = 9;             // float4 per thread and side held in registers
constexpr int kMaxOwn = 36;              // rows a workgroup may own per side (kTeams x kMaxSlots)
constexpr int kMaxSide = 8704;           // potentials of one side in LDS (two sides: 139 KB)
constexpr int kMaxLds = 2 * 8 * 1024 * ((kMaxSide + 1023) / 1024);  // bytes of both sides' potentials
constexpr int kSums = 8;                 // values a workgroup contributes to a check
constexpr int kSegments = 96;            // eps segments per launch
constexpr u64 kEmpty = 0x7ffddeadc0ffee01ull;
constexpr u64 kPlainNan = 0x7ff8000000000000ull;
constexpr double kSigInit = -1.0e6;      // "no term yet", as in the sweep

struct Segments {
    int count;
    double eps[kSegments];
    long long iters[kSegments];
};

struct GapParams {
    double factor, tolerance, tau;
    long long batch, max_iter;
    ResidentResult from;  // the state at the launch: all zero but eps, or where the last launch stopped
};

struct Args {
    ResidentProblem rp;
    u64 *fx, *gx;     // [2][n] exchange
    u64 *flags;       // [3][kMaxWg]
    u64 *sums;        // [3][kMaxWg * kSums]
    ResidentResult *res;
    int n_wg;
    int rf, cf, rg, cg;  // rows per team and chunks per row: C rows, C^T rows
    double lambda1, lambda2, log_ni, log_nj;
    long long launches;  // this one included
    ResidentLimits lim;
    GapParams gap;
};

__device__ __forceinline__ u64 load_x(const u64 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_x(u64 *p, u64 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 pack(double v) {
    const u64 b = (u64)__double_as_longlong(v);
    return b == kEmpty ? kPlainNan : b;
}
__device__ __forceinline__ double unpack(u64 b) { return __longlong_as_double((long long)b); }

template <int CTRL>
__device__ __forceinline__ int dpp_mov(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}

// the wave's sum in every lane by the xor tree 32, 16, 8, 4, 2, 1.  Once the lanes agree modulo
// 16 (8, 4, 2), a rotation by 8 (4, 2, 1) within the row brings the xor partner's value.
__device__ __forceinline__ double xor_sum(double v) {
    {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    }
    v += __hiloint2double(dpp_mov<0x128>(__double2hiint(v)), dpp_mov<0x128>(__double2loint(v)));
    v += __hiloint2double(dpp_mov<0x124>(__double2hiint(v)), dpp_mov<0x124>(__double2loint(v)));
    v += __hiloint2double(dpp_mov<0x122>(__double2hiint(v)), dpp_mov<0x122>(__double2loint(v)));
    v += __hiloint2double(dpp_mov<0x121>(__double2hiint(v)), dpp_mov<0x121>(__double2loint(v)));
    return v;
}

__device__ __forceinline__ int xor_max(int v) {
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = max((int)a[0], (int)a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = max((int)b[0], (int)b[1]);
    v = max(v, dpp_mov<0x128>(v));
    v = max(v, dpp_mov<0x124>(v));
    v = max(v, dpp_mov<0x122>(v));
    return max(v, dpp_mov<0x121>(v));
}

struct Shared {
    double2 red[kMaxOwn][4];      // per owned row and wave: (shift, sum); or row sums
    double wsum[16][kSums];       // per wave, for the checks
    double total[kSums];
    // owned rows: potentials, absorbed potentials, both before the last iteration, log weight
    double f[kMaxOwn], u[kMaxOwn], fp[kMaxOwn], up[kMaxOwn], lw[kMaxOwn];
    double g[kMaxOwn], v[kMaxOwn], gp[kMaxOwn], vp[kMaxOwn];
    int aborted[2];               // by the parity of sync_ok's calls
};

template <int S>
struct Solver {
    const Args &a;
    Shared &sh;
    double *hf, *hg;              // LDS: potentials of the source / target side, in thread order
    const int tid, tt, team, wv, lane, wg, n_teams;
    f4 c[S], ct[S];               // this thread's pieces of its team's C and C^T rows
    // owner threads (tid < kMaxOwn): the workgroup's rows tid
    int row_f, row_g;             // or -1
    // potentials that the workgroup reads: all, or none where it owns no row of C (need_g) or of C^T
    int need_f, need_g;
    int pf;                       // parity of the last published f and g
    int pt;                       // buffer of the last published maxima
    int pc;                       // buffer of the last published sums
    int phase;                    // of sync_ok
    bool flag_open;               // the last iteration's maxima have not been read yet

    // LDS place of potential j: float4 group t of chunk m, halves apart (16-byte lane stride)
    __device__ static int place(int j) { return ((j >> 10) << 10) + (((j >> 1) & 1) << 9) + (((j >> 2) & 255) << 1) + (j & 1); }

    __device__ void load_cost() {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            c[s] = ct[s] = f4{0.f, 0.f, 0.f, 0.f};
            const int rf = s / a.cf, mf = s - rf * a.cf;
            const int64_t row = (int64_t)wg * kTeams + team + (int64_t)rf * n_teams;
            const int col = 4 * tt + 1024 * mf;
            if (rf < a.rf && row < a.rp.n_i && col < a.rp.n_j)
                c[s] = *reinterpret_cast<const f4 *>(a.rp.C + row * a.rp.ldc + col);
            const int rg = s / a.cg, mg = s - rg * a.cg;
            const int64_t rowt = (int64_t)wg * kTeams + team + (int64_t)rg * n_teams;
            const int colt = 4 * tt + 1024 * mg;
            if (rg < a.rg && rowt < a.rp.n_j && colt < a.rp.n_i)
                ct[s] = *reinterpret_cast<const f4 *>(a.rp.CT + rowt * a.rp.ldct + colt);
        }
    }

    // Polls one value until it is there; false when the wait was given up.
    __device__ bool wait_value(const u64 *p, u64 &x) {
        const long long start = wall_clock64();
        for (int n = 1; x == kEmpty; ++n) {
            __builtin_amdgcn_s_sleep(1);
            x = load_x(p);
            if ((n & a.lim.look_mask) == 0 && x == kEmpty) {
                if (__hip_atomic_load(&a.res->aborted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
                    wall_clock64() - start > a.lim.wait_ticks) {
                    __hip_atomic_store(&a.res->aborted, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    sh.aborted[phase] = 1;
                    return false;
                }
            }
        }
        return true;
    }

    // a side's potentials into LDS, times scale; loads of four in flight
    __device__ void take(const u64 *src, int n, double *h, double scale) {
        for (int b = tid; b < n; b += 4 * kT) {
            u64 x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = b + q * kT < n ? load_x(src + b + q * kT) : 0ull;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = b + q * kT;
                if (j >= n || !wait_value(src + j, x[q])) continue;
                h[place(j)] = unpack(x[q]) * scale;
            }
        }
    }

    // ends the workgroup when any wait was given up; every thread calls it.  Two flags in turn: a
    // wave that is past the barrier and gives up its next wait must not change what a slower wave
    // is about to read here, or the workgroup's waves part.
    __device__ bool sync_ok() {
        __syncthreads();
        const bool ok = sh.aborted[phase] == 0;
        phase ^= 1;
        return ok;
    }

    // log-sum-exp of the team's rows over the potentials in h (times k), wave results to sh.red
    __device__ void sweep(const f4 (&cost)[S], int rows, int chunks, const double *h, double k) {
        double sig = kSigInit;
        float s = 0.f;
        int m = 0, r = 0;
        const int n = rows * chunks;
#pragma unroll
        for (int i = 0; i < S; ++i) {
            if (i >= n) continue;  // uniform
            // opaque here: widened outside the iteration loop, the pieces would take three times the registers
            f4 x = cost[i];
            asm volatile("" : "+v"(x));
            const double2 h01 = *reinterpret_cast<const double2 *>(h + m * 1024 + 2 * tt);
            const double2 h23 = *reinterpret_cast<const double2 *>(h + m * 1024 + 512 + 2 * tt);
            const double y0 = fma(-k, (double)x[0], h01.x);
            const double y1 = fma(-k, (double)x[1], h01.y);
            const double y2 = fma(-k, (double)x[2], h23.x);
            const double y3 = fma(-k, (double)x[3], h23.y);
            const double top = fmax(fmax(y0, y1), fmax(y2, y3));
            if (top > sig) {
                const double ns = ceil(top);
                s = ldexpf(s, (int)(sig - ns));
                sig = ns;
            }
            const float e0 = __builtin_amdgcn_exp2f((float)(y0 - sig));
            const float e1 = __builtin_amdgcn_exp2f((float)(y1 - sig));
            const float e2 = __builtin_amdgcn_exp2f((float)(y2 - sig));
            const float e3 = __builtin_amdgcn_exp2f((float)(y3 - sig));
            s += (e0 + e1) + (e2 + e3);
            if (++m == chunks) {  // uniform: the row is complete
                const int si = (int)sig, mx = xor_max(si);
                const double t = xor_sum(ldexp((double)s, si - mx));
                if (lane == 0) sh.red[r * kTeams + team][wv] = make_double2((double)mx, t);
                m = 0;
                ++r;
                sig = kSigInit;
                s = 0.f;
            }
            __builtin_amdgcn_sched_barrier(0);  // the pieces hold the registers: one exponent group at a time
        }
    }

    // the potential of an owned row from its four waves (the sweep's epilogue)
    __device__ double potential(double lw, double log_n, double alpha, double eps) const {
        double sg = sh.red[tid][0].x, sd = sh.red[tid][0].y;
#pragma unroll
        for (int w = 1; w < 4; ++w) lse_merge(sg, sd, sh.red[tid][w].x, sh.red[tid][w].y);
        const double lse = (sg + log2(sd)) * kLn2;
        return alpha * eps * (lw + log_n - lse);
    }

    // one (a, b) iteration; checks: also publishes the workgroup's largest growth since the absorption
    __device__ bool iterate(double eps, bool first, bool checks) {
        const double k = kLog2E / eps, inv_eps = 1.0 / eps;
        const double al1 = a.lambda1 / (a.lambda1 + eps), al2 = a.lambda2 / (a.lambda2 + eps);
        const int n_i = a.rp.n_i, n_j = a.rp.n_j;
        if (first) {
            for (int j = tid; j < n_j; j += kT) hg[place(j)] = a.rp.g[j] * k;
        } else {
            take(a.gx + (int64_t)pf * n_j, need_g, hg, k);
        }
        if (!sync_ok()) return false;
        if (checks && flag_open && !absorb()) return false;
        const int p = pf ^ 1;  // this iteration's buffers; the other ones hold what their readers have read
        if (row_f >= 0 && !first) store_x(a.fx + (int64_t)pf * n_i + row_f, kEmpty);
        sweep(c, a.rf, a.cf, hg, k);
        __syncthreads();
        if (row_f >= 0) {
            sh.fp[tid] = sh.f[tid];
            sh.up[tid] = sh.u[tid];
            const double f = potential(sh.lw[tid], a.log_nj, al1, eps);
            sh.f[tid] = f;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the emptied buffer first
            store_x(a.fx + (int64_t)p * n_i + row_f, pack(f));
        }
        take(a.fx + (int64_t)p * n_i, need_f, hf, k);
        if (!sync_ok()) return false;
        if (row_g >= 0 && !first) store_x(a.gx + (int64_t)pf * n_j + row_g, kEmpty);
        sweep(ct, a.rg, a.cg, hf, k);
        __syncthreads();
        double grown = -INFINITY;
        if (row_g >= 0) {
            sh.gp[tid] = sh.g[tid];
            sh.vp[tid] = sh.v[tid];
            const double g = potential(a.rp.misc[0], a.log_ni, al2, eps);
            sh.g[tid] = g;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            store_x(a.gx + (int64_t)p * n_j + row_g, pack(g));
            grown = (g - sh.v[tid]) * inv_eps;
        }
        if (checks) {
            if (row_f >= 0) grown = fmax(grown, (sh.f[tid] - sh.u[tid]) * inv_eps);
            const int q = pt == 2 ? 0 : pt + 1, after = q == 2 ? 0 : q + 1;
            if (tid < 64) {
                grown = wave_max(grown);
                if (tid == 0) {
                    // the next iteration's buffer held the maxima before the last ones
                    store_x(a.flags + (int64_t)after * kMaxWg + wg, kEmpty);
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    store_x(a.flags + (int64_t)q * kMaxWg + wg, pack(grown));
                }
            }
            pt = q;
            flag_open = true;
        }
        pf = p;
        return true;
    }

    // tau-triggered absorption (optimal_transport.py:137-141) after the last iteration
    long long n_stab;
    __device__ bool absorb() {
        double m = -INFINITY;
        if (tid < a.n_wg) {
            u64 x = load_x(a.flags + (int64_t)pt * kMaxWg + tid);
            if (wait_value(a.flags + (int64_t)pt * kMaxWg + tid, x)) m = unpack(x);
        }
        m = wave_max(m);
        if (lane == 0) sh.wsum[tid >> 6][0] = m;
        if (!sync_ok()) return false;
        m = sh.wsum[0][0];
#pragma unroll
        for (int w = 1; w < kMaxWg / 64; ++w) m = fmax(m, sh.wsum[w][0]);
        if (exp(m) > a.gap.tau) {
            if (tid < kMaxOwn) {
                sh.u[tid] = sh.f[tid];
                sh.v[tid] = sh.g[tid];
            }
            ++n_stab;
        }
        flag_open = false;
        __syncthreads();  // sh.wsum is written again
        return true;
    }

    // sums over the workgroups of val[0 .. n): every workgroup gets the same totals in sh.total.
    // val: this thread's contribution.
    __device__ bool all_sum(const double (&val)[kSums], int n) {
        const int p = pc == 2 ? 0 : pc + 1, after = p == 2 ? 0 : p + 1;
#pragma unroll
        for (int q = 0; q < kSums; ++q) {
            if (q >= n) continue;
            const double t = xor_sum(val[q]);
            if (lane == 0) sh.wsum[tid >> 6][q] = t;
        }
        __syncthreads();
        // the next check's buffer held the check before the last one, which everybody had added up
        // before publishing the last one's sums; all its words, whatever the checks' widths
        if (tid < kSums) store_x(a.sums + ((int64_t)after * kMaxWg + wg) * kSums + tid, kEmpty);
        if (tid < n) {
            double t = sh.wsum[0][tid];
            for (int w = 1; w < 16; ++w) t += sh.wsum[w][tid];
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the emptied words of this wave first
            store_x(a.sums + ((int64_t)p * kMaxWg + wg) * kSums + tid, pack(t));
        }
        const int w = tid >> 6;
        if (w < n) {  // one wave per value, workgroups in order over the lanes
            double t = 0.0;
            for (int b = lane; b < a.n_wg; b += 64) {
                const u64 *src = a.sums + ((int64_t)p * kMaxWg + b) * kSums + w;
                u64 x = load_x(src);
                if (wait_value(src, x)) t += unpack(x);
            }
            t = xor_sum(t);
            if (lane == 0) sh.total[w] = t;
        }
        pc = p;
        return sync_ok();
    }

    // FP64 row sums of exp((row + col - cost)/eps) over the potentials in h; adds
    // [sum R y, sum R cost] or (KT) sum exp(-cost/eps) of the team's rows to val
    template <bool PARTS, bool KT>
    __device__ void plan_rows(const f4 (&cost)[S], int rows, int chunks, int n_rows, int n_cols, const double *h,
                              const double *hr, double inv_eps, double &s_ry, double &s_rc) {
        const int n = rows * chunks;
        double acc = 0.0;
        int m = 0, r = 0;
#pragma unroll
        for (int i = 0; i < S; ++i) {
            if (i >= n) continue;  // uniform
            const int row = wg * kTeams + team + r * n_teams;
            const double fr = row < n_rows ? hr[place(row)] : -INFINITY;
            f4 x = cost[i];
            asm volatile("" : "+v"(x));
#pragma unroll 1
            for (int q = 0; q < 4; ++q) {
                const int j = 4 * tt + 1024 * m + q;
                const double cv = (double)(q == 0 ? x[0] : q == 1 ? x[1] : q == 2 ? x[2] : x[3]);
                if (KT) {
                    if (row < n_rows && j < n_cols) s_ry += exp(-cv * inv_eps);
                } else {
                    const double gv = j < n_cols ? h[place(j)] : -INFINITY;
                    const double y = (fr + gv - cv) * inv_eps;
                    const double R = exp(y);
                    acc += R;
                    if (PARTS) {
                        if (R > 0.0) s_ry = fma(R, y, s_ry);
                        s_rc = fma(R, cv, s_rc);
                    }
                }
            }
            if (++m == chunks) {
                if (!KT) {
                    const double t = xor_sum(acc);
                    if (lane == 0) sh.red[r * kTeams + team][wv] = make_double2(t, 0.0);
                }
                acc = 0.0;
                m = 0;
                ++r;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // dual-variable evolution (optimal_transport.py:157-160) after a batch
    __device__ bool evolution(double eps, double &gap) {
        const double ie = 1.0 / eps;
        double val[kSums] = {};
        if (row_f >= 0) {
            const double A = exp(sh.f[tid] * ie), Ao = exp((sh.fp[tid] - sh.up[tid]) * ie) * exp(sh.u[tid] * ie);
            val[0] = (A - Ao) * (A - Ao);
            val[1] = A * A;
        }
        if (row_g >= 0) {
            const double B = exp(sh.g[tid] * ie), Bo = exp((sh.gp[tid] - sh.vp[tid]) * ie) * exp(sh.v[tid] * ie);
            val[2] = (B - Bo) * (B - Bo);
            val[3] = B * B;
        }
        if (!all_sum(val, 4)) return false;
        const double ga = sqrt(sh.total[0]) / (1.0 + sqrt(sh.total[1]));
        const double gb = sqrt(sh.total[2]) / (1.0 + sqrt(sh.total[3]));
        gap = gb > ga ? gb : ga;
        return true;
    }

    // sum of exp(-C/eps)
    __device__ bool ktilde(double eps, double &sum) {
        double val[kSums] = {}, unused = 0.0;
        plan_rows<false, true>(c, a.rf, a.cf, a.rp.n_i, a.rp.n_j, hg, hf, 1.0 / eps, val[0], unused);
        if (!all_sum(val, 1)) return false;
        sum = sh.total[0];
        return true;
    }

    // primal, dual, gap (optimal_transport.py:45-62, 152-156) at the last iteration's potentials
    __device__ bool duality(double eps, double skt, double &pri, double &dua, double &gap) {
        const int n_i = a.rp.n_i, n_j = a.rp.n_j;
        // everybody waits for everybody's sums below, so these buffers stay until all have read them
        take(a.gx + (int64_t)pf * n_j, n_j, hg, 1.0);
        take(a.fx + (int64_t)pf * n_i, n_i, hf, 1.0);
        if (!sync_ok()) return false;
        const double ie = 1.0 / eps, inv_i = 1.0 / n_i, inv_j = 1.0 / n_j, q = a.rp.misc[1];
        double val[kSums] = {}, none = 0.0;
        plan_rows<true, false>(c, a.rf, a.cf, n_i, n_j, hg, hf, ie, val[5], val[6]);
        __syncthreads();
        if (row_f >= 0) {
            const double r = ((sh.red[tid][0].x + sh.red[tid][1].x) + sh.red[tid][2].x) + sh.red[tid][3].x;
            const double p = a.rp.G[row_f], x = r * inv_j;
            val[0] = inv_i * (x * log(x / p) - x + p);
            val[2] = (p * inv_i) * (exp(-sh.f[tid] / a.lambda1) - 1.0);
            val[4] = r;
        }
        __syncthreads();
        plan_rows<false, false>(ct, a.rg, a.cg, n_j, n_i, hf, hg, ie, none, none);
        __syncthreads();
        if (row_g >= 0) {
            const double r = ((sh.red[tid][0].x + sh.red[tid][1].x) + sh.red[tid][2].x) + sh.red[tid][3].x;
            const double x = r * inv_i;
            val[1] = inv_j * (x * log(x / q) - x + q);
            val[3] = (q * inv_j) * (exp(-sh.g[tid] / a.lambda2) - 1.0);
        }
        if (!all_sum(val, 7)) return false;
        const double *t = sh.total;
        const double ij = (double)n_i * (double)n_j;
        pri = a.lambda1 * t[0] + a.lambda2 * t[1] + (eps * (t[5] - t[4] + skt) + t[6]) / ij;
        dua = -a.lambda1 * t[2] - a.lambda2 * t[3] - eps * (t[4] - skt) / ij;
        gap = (pri - dua) / fabs(pri);
        __syncthreads();  // sh.total is written again
        return true;
    }

    // the duality-gap schedule, at most launch_iters iterations of it; false when a wait was given up
    __device__ bool run_gap(ResidentResult &out) {
        const GapParams &gp_ = a.gap;
        const int n_scal = 5;
        out = gp_.from;
        out.stopped = 0;
        bool resumed = gp_.from.stopped, first = true;
        const long long stop_at = out.iterations + a.lim.launch_iters;
        long long t = out.in_batch;
        for (int e = out.scaling; e <= n_scal; ++e) {
            if (!resumed) {
                out.gap = INFINITY;
                if (tid < kMaxOwn) {
                    sh.u[tid] = sh.f[tid];
                    sh.v[tid] = sh.g[tid];
                }
                out.eps = out.eps / gp_.factor;
                if (e == n_scal && !ktilde(out.eps, out.sum_ktilde)) return false;
            }
            resumed = false;
            const double thr = e == n_scal ? gp_.tolerance : 1e-6;
            const long long nb = e == n_scal ? gp_.batch : 5;
            while (out.gap > thr) {
                for (; t < nb; ++t) {
                    if (out.iterations == stop_at) {  // every workgroup counts the same
                        if (flag_open && !absorb()) return false;
                        out.stopped = 1;
                        out.scaling = e;
                        out.in_batch = t;
                        out.stabilisations = n_stab;
                        return true;
                    }
                    ++out.iterations;
                    if (!iterate(out.eps, first, true)) return false;
                    first = false;
                    if (out.iterations >= gp_.max_iter) {
                        if (!absorb()) return false;
                        out.max_iter_reached = 1;
                        out.stabilisations = n_stab;
                        return true;
                    }
                }
                t = 0;
                if (!absorb()) return false;
                ++out.checks;
                if (e < n_scal) {
                    if (!evolution(out.eps, out.gap)) return false;
                    __syncthreads();
                } else if (!duality(out.eps, out.sum_ktilde, out.primal, out.dual, out.gap)) {
                    return false;
                }
            }
        }
        out.stabilisations = n_stab;
        return true;
    }
};

template <int S, bool GAP>
__global__ __launch_bounds__(kT) void resident_kernel(Args a, Segments seg) {
    extern __shared__ __align__(16) double h_lds[];
    __shared__ Shared sh;
    const int tid = threadIdx.x, wg = blockIdx.x, n_teams = a.n_wg * kTeams;
    const int n_i = a.rp.n_i, n_j = a.rp.n_j;
    double *hf = h_lds, *hg = h_lds + 1024 * a.cg;  // cg chunks of the source side, cf of the target side
    if (tid < 2) sh.aborted[tid] = 0;
    for (int j = tid; j < 1024 * (a.cg + a.cf); j += kT) h_lds[j] = -INFINITY;  // padding stays so
    Solver<S> so{a, sh, hf, hg, tid, tid & 255, __builtin_amdgcn_readfirstlane(tid >> 8), (tid >> 6) & 3, tid & 63, wg,
                 n_teams};
    so.load_cost();
    const int own = wg * kTeams + (tid & (kTeams - 1)) + (tid / kTeams) * n_teams;
    so.row_f = tid < kTeams * a.rf && own < n_i ? own : -1;
    so.row_g = tid < kTeams * a.rg && own < n_j ? own : -1;
    if (tid < kMaxOwn) {
        sh.f[tid] = sh.u[tid] = sh.fp[tid] = sh.up[tid] = so.row_f >= 0 ? a.rp.f[so.row_f] : 0.0;
        sh.g[tid] = sh.v[tid] = sh.gp[tid] = sh.vp[tid] = so.row_g >= 0 ? a.rp.g[so.row_g] : 0.0;
        sh.lw[tid] = so.row_f >= 0 ? a.rp.logp[so.row_f] : 0.0;
        if (GAP && a.gap.from.stopped) {
            if (so.row_f >= 0) sh.u[tid] = a.rp.u[so.row_f];
            if (so.row_g >= 0) sh.v[tid] = a.rp.v[so.row_g];
        }
    }
    so.need_g = wg * kTeams < n_i ? n_j : 0;
    so.need_f = wg * kTeams < n_j ? n_i : 0;
    so.pf = 1;
    so.pt = 2;
    so.pc = 2;
    so.phase = 0;
    so.flag_open = false;
    so.n_stab = a.gap.from.stabilisations;
    __syncthreads();
    ResidentResult out{};
    if constexpr (GAP) {
        if (!so.run_gap(out)) return;
    } else {
        bool first = true;
        for (int q = 0; q < seg.count; ++q)
            for (long long n = 0; n < seg.iters[q]; ++n) {
                if (!so.iterate(seg.eps[q], first, false)) return;
                first = false;
            }
    }
    if (so.row_f >= 0) a.rp.f[so.row_f] = sh.f[tid];
    if (so.row_g >= 0) a.rp.g[so.row_g] = sh.g[tid];
    if (wg == 0 && tid == 0) a.res->launches = a.launches;
    if constexpr (GAP) {
        if (out.stopped) {
            if (so.row_f >= 0) a.rp.u[so.row_f] = sh.u[tid];
            if (so.row_g >= 0) a.rp.v[so.row_g] = sh.v[tid];
        }
        if (wg == 0 && tid == 0) {
            ResidentResult &r = *a.res;  // all but the flag that any workgroup may raise
            r.max_iter_reached = out.max_iter_reached;
            r.iterations = out.iterations;
            r.stabilisations = out.stabilisations;
            r.checks = out.checks;
            r.gap = out.gap;
            r.primal = out.primal;
            r.dual = out.dual;
            r.eps = out.eps;
            r.stopped = out.stopped;
            r.scaling = out.scaling;
            r.in_batch = out.in_batch;
            r.sum_ktilde = out.sum_ktilde;
        }
    }
}

// every exchange value empty, the result cleared
__global__ __launch_bounds__(256) void resident_clear_kernel(u64 *x, int64_t n, ResidentResult *res) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) x[i] = kEmpty;
    if (blockIdx.x == 0 && threadIdx.x == 0) *res = ResidentResult{};
}

struct Shape {
    int n_wg, rf, cf, rg, cg, slots;
};

Shape shape_of(int64_t I, int64_t J) {
    Shape s;
    s.n_wg = (int)std::min<int64_t>(kMaxWg, (std::max(I, J) + kTeams - 1) / kTeams);
    const int64_t teams = (int64_t)s.n_wg * kTeams;
    s.rf = (int)((I + teams - 1) / teams);
    s.rg = (int)((J + teams - 1) / teams);
    s.cf = (int)((J + 1023) / 1024);
    s.cg = (int)((I + 1023) / 1024);
    s.slots = std::max(s.rf * s.cf, s.rg * s.cg);
    return s;
}

struct Exchange {
    ResidentResult *res;
    u64 *x;
    int64_t n;
};

Exchange carve(void *base, int64_t I, int64_t J) {
    Exchange e;
    e.res = static_cast<ResidentResult *>(base);
    e.x = reinterpret_cast<u64 *>(static_cast<char *>(base) + 256);
    e.n = 2 * (I + J) + 3 * kMaxWg + 3 * kMaxWg * kSums;
    return e;
}

template <int S, bool GAP>
int launch(Args &a, Segments &seg, int *launched, hipStream_t s) {
    const int lds = (int)sizeof(double) * 1024 * (a.cf + a.cg);
    const void *fn = reinterpret_cast<const void *>(resident_kernel<S, GAP>);
    // the limit belongs to the function, not to the launch: the largest any pair needs, so that
    // threads with pairs of different shapes set the same
    WOTK_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds));
    int per_cu = 0, dev = 0, cus = 0;
    WOTK_HIP(hipGetDevice(&dev));
    WOTK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    WOTK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kT, lds));
    *launched = 0;
    if ((int64_t)per_cu * cus < a.n_wg) return WOTK_OK;
    resident_kernel<S, GAP><<<(unsigned)a.n_wg, kT, lds, s>>>(a, seg);
    WOTK_LAUNCH_CHECK();
    *launched = 1;
    return WOTK_OK;
}

template <bool GAP>
int dispatch(Args &a, Segments &seg, int slots, int *launched, hipStream_t s) {
    if (slots <= 2) return launch<2, GAP>(a, seg, launched, s);
    if (slots <= 4) return launch<4, GAP>(a, seg, launched, s);
    if (slots <= 6) return launch<6, GAP>(a, seg, launched, s);
    return launch<kMaxSlots, GAP>(a, seg, launched, s);
}

Args make_args(const ResidentProblem &rp, const Shape &sh, double lambda1, double lambda2,
               const ResidentLimits &lim) {
    const Exchange e = carve(rp.exchange, rp.n_i, rp.n_j);
    Args a{};
    a.rp = rp;
    a.fx = e.x;
    a.gx = a.fx + 2 * (int64_t)rp.n_i;
    a.flags = a.gx + 2 * (int64_t)rp.n_j;
    a.sums = a.flags + 3 * kMaxWg;
    a.res = e.res;
    a.n_wg = sh.n_wg;
    a.rf = sh.rf;
    a.cf = sh.cf;
    a.rg = sh.rg;
    a.cg = sh.cg;
    a.lambda1 = lambda1;
    a.lambda2 = lambda2;
    a.log_ni = std::log((double)rp.n_i);
    a.log_nj = std::log((double)rp.n_j);
    a.lim = lim;
    return a;
}

int clear(const ResidentProblem &rp, hipStream_t s) {
    const Exchange e = carve(rp.exchange, rp.n_i, rp.n_j);
    resident_clear_kernel<<<(unsigned)std::min<int64_t>(256, (e.n + 255) / 256), 256, 0, s>>>(e.x, e.n, e.res);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

}  // namespace

// Where the resident solver beats launched sweeps: everywhere its registers hold the pair (us per
// iteration, launched / resident): 50 x 60 8.0 / 4.4, 300 x 400 8.3 / 4.9, 1000 x 1000 8.9 / 6.0,
// 2000 x 2500 15.8 / 11.0, 2890 x 2890 19.8 / 14.5, 900 x 8000 23.1 / 15.8; solves of a few iterations
// aside (sinkhorn.hip).  Nine pieces a thread would reach 3072 x 3072, where the one-read iteration
// takes 18; the line stands at 2^23 entries, from which on results come from that one's FP64 column
// sums.
bool resident_fits(int64_t I, int64_t J) {
    if (I > kMaxSide || J > kMaxSide || I * J > (1ll << 23)) return false;
    const Shape s = shape_of(I, J);
    return s.slots <= kMaxSlots && kTeams * std::max(s.rf, s.rg) <= kMaxOwn;
}

size_t resident_bytes(int64_t I, int64_t J) { return 256 + sizeof(u64) * (size_t)carve(nullptr, I, J).n; }

int resident_fixed(const ResidentProblem &rp, double lambda1, double lambda2, double epsilon, double epsilon0,
                   int64_t scaling_iter, int64_t inner_iter_max, int64_t extra_iter, const ResidentLimits &lim,
                   int *launched, hipStream_t s) {
    const Shape sh = shape_of(rp.n_i, rp.n_j);
    const int64_t total = scaling_iter + extra_iter;
    auto reg = [&](int64_t n) { return (epsilon0 - epsilon) * std::exp(-(double)n) + epsilon; };
    *launched = 0;
    long long launches = 0;
    for (int64_t at = 0; at < total;) {
        Segments seg{};
        int64_t queued = 0;
        while (at < total && seg.count < kSegments && queued < lim.launch_iters) {
            // up to the next change of eps
            const int64_t block = at < scaling_iter ? at / inner_iter_max : scaling_iter / inner_iter_max;
            const int64_t end = at < scaling_iter ? std::min(scaling_iter, (block + 1) * inner_iter_max) : total;
            const int64_t n = std::min<int64_t>(end - at, lim.launch_iters - queued);
            seg.eps[seg.count] = reg(block);
            seg.iters[seg.count++] = n;
            queued += n;
            at += n;
        }
        int rc = clear(rp, s);
        if (rc) return rc;
        Args a = make_args(rp, sh, lambda1, lambda2, lim);
        a.launches = ++launches;
        rc = dispatch<false>(a, seg, sh.slots, launched, s);
        if (rc || !*launched) return rc;
        if (at < total) {  // the next launch clears the flag: look before
            ResidentResult r;
            rc = resident_result(rp, &r, s);
            if (rc || r.aborted) return rc;
        }
    }
    return WOTK_OK;
}

int resident_gap(const ResidentProblem &rp, double lambda1, double lambda2, double epsilon, long long batch_size,
                 double tolerance, double tau, double epsilon0, long long max_iter, const ResidentLimits &lim,
                 int *launched, ResidentResult *out, hipStream_t s) {
    const Shape sh = shape_of(rp.n_i, rp.n_j);
    const double factor = std::exp(-std::log(epsilon) / 5);
    *out = ResidentResult{};
    out->eps = epsilon0 * factor;
    do {
        int rc = clear(rp, s);
        if (rc) return rc;
        Args a = make_args(rp, sh, lambda1, lambda2, lim);
        a.launches = out->launches + 1;
        a.gap = GapParams{factor, tolerance, tau, batch_size, max_iter, *out};
        Segments seg{};
        rc = dispatch<true>(a, seg, sh.slots, launched, s);
        if (rc || !*launched) return rc;
        rc = resident_result(rp, out, s);
        if (rc) return rc;
    } while (out->stopped && !out->aborted);
    return WOTK_OK;
}

int resident_pass_by(const ResidentProblem &rp, hipStream_t s) { return clear(rp, s); }

int resident_result(const ResidentProblem &rp, ResidentResult *out, hipStream_t s) {
    WOTK_HIP(hipMemcpyAsync(out, rp.exchange, sizeof(ResidentResult), hipMemcpyDeviceToHost, s));
    WOTK_HIP(hipStreamSynchronize(s));
    return WOTK_OK;
}

}  // namespace wotk
