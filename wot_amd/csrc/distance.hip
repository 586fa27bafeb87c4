// Squared distances of a day pair and their exact median, without an I x J
// FP64 matrix in memory: every pass regenerates the distances tile by tile.
//
// A stored FP64 matrix costs 16 bytes per entry to write and read back for each
// use; regenerating an entry costs 2 d FP64 operations (60 at d = 30: 0.34 ms for
// 15000 x 15000 at the FP64 rate, against 0.65 ms for the write and one read at
// the copy rate), so the median's one counting pass and the cost's write pass
// both regenerate.  The median is an order statistic over the bit patterns (for
// non-negative doubles the uint64 order is the value order; NaNs sort on top):
//   sample  -> a bracket [lo, hi] of keys that holds the median's rank with a
//              6-sigma margin (65536 sampled pairs: 2.3 % of the entries)
//   collect -> entries below lo counted, entries inside kept as (key, index)
//   select  -> the exact rank among the kept ones (histogram, then the bins
//              holding the one or two middle ranks in one workgroup)
// When the bracket misses the rank or heavy ties overflow the kept list, a device
// flag starts a six-digit radix select that regenerates the distances per digit;
// otherwise its launches exit at once.  (Coordinates of 4 integers, d = 30: 6.8 ms for
// 15000 x 15000, 0.70 ms for 4000 x 3500; read from a stored matrix 68.8 and 4.7 ms.)
// Bound: FP64 issue (2 d operations per entry and pass at 3.4e13 / s).  15000 x 15000,
// d = 30, cost and median: 1.57 ms (0.75 ms collect, 0.7 ms write, 0.08 ms selection)
// against 4.73 ms with a stored FP64 matrix read by six digit passes, a next-above, an
// index and a normalise pass (88 bytes per entry); 1215 x 1163: 0.11 ms against 0.38 ms.
#include <algorithm>

#include "distance.h"

namespace wotk {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned long long u64;

// ---------------------------------------------------------------------------
// Tile engines: a 256-thread workgroup computes a ROWS x COLS tile, thread by
// thread NE entries in registers; row(e) / col(e) place entry e.
// ---------------------------------------------------------------------------
// FP64 direct differences.  8 x 4 entries per thread, rows and columns 16 apart:
// 64 FP64 operations for 12 8-byte LDS reads per k (two thirds of the LDS rate), the
// next k's operands read while this one's are used.  (8 x 8 entries need fewer reads
// but leave no registers for that: it spilled at 2 waves per SIMD.)  Coordinates lie in LDS as they lie
// in memory, row after row, so staging is a linear copy in 16-byte pieces with every
// load in flight at once; the row pitch is twice an odd number, which puts the 16
// rows a quarter wave reads on distinct banks.  (A transposing, 8-byte staging of the
// same tile cost 0.2 ms per pass of 15000 x 15000.)
// TR x TC entries per thread.  Where 8 x 4 leaves CUs without a tile, 4 x 2 (a fourth of the entries in a
// third of the time; sums and bits the same).
template <int TR, int TC>
struct F64TileOf {
    static constexpr int ROWS = 16 * TR, COLS = 16 * TC, NE = TR * TC, WAVES = 3;
    static constexpr int P = 34;  // row pitch and largest k chunk: 2 * 17
    static constexpr size_t LDS = sizeof(double) * (ROWS + COLS) * P;
    double v[NE];
    int i0, j0, tx, ty;

    __device__ int row(int e) const { return i0 + ty + 16 * (e / TC); }
    __device__ int col(int e) const { return j0 + tx + 16 * (e % TC); }

    // coordinates [k0, k0 + km) of N points from p0, zeros past the last point and past an odd km;
    // B 16-byte pieces per thread in flight
    template <int N, int B>
    __device__ static void stage(const double *pts, int n, int p0, int d, int k0, int km, double *out) {
        const int tid = threadIdx.x, np = (km + 1) >> 1;
        const float inv = 1.0f / (float)np;
        const double *src = pts + (int64_t)p0 * d + k0;
        const int left = min(n - p0, N);
        const bool wide = ((uintptr_t)src & 15) == 0 && (d & 1) == 0 && (km & 1) == 0;  // uniform
        for (int e0 = tid; e0 < N * np; e0 += 256 * B) {
            double2 t[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int e = e0 + 256 * u;
                const int r = (int)(((float)e + 0.5f) * inv), q = e - r * np;  // e / np: exact, e < 2^13
                t[u] = make_double2(0.0, 0.0);
                if (r < left) {
                    const double *s = src + r * d + 2 * q;
                    if (wide) {
                        t[u] = *reinterpret_cast<const double2 *>(s);
                    } else {
                        t[u].x = s[0];
                        if (2 * q + 1 < km) t[u].y = s[1];
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int e = e0 + 256 * u;
                const int r = (int)(((float)e + 0.5f) * inv), q = e - r * np;
                if (r < N) *reinterpret_cast<double2 *>(out + r * P + 2 * q) = t[u];
            }
        }
    }

    struct Operands {
        double x[TR], y[TC];
        __device__ void load(const double *xk, const double *yk) {
#pragma unroll
            for (int q = 0; q < TR; ++q) x[q] = xk[q * 16 * P];
#pragma unroll
            for (int q = 0; q < TC; ++q) y[q] = yk[q * 16 * P];
        }
    };

    __device__ void step(const Operands &o) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const double t = o.x[e / TC] - o.y[e % TC];
            v[e] = fma(t, t, v[e]);
        }
    }

    __device__ void compute(const DistanceProblem &pb, int ti, int tj, unsigned char *lds) {
        const int tid = threadIdx.x;
        tx = tid & 15;
        ty = tid >> 4;
        i0 = ti * ROWS;
        j0 = tj * COLS;
        // equal k chunks of at most P; the first one staged before the sums take their registers
        const int chunks = (pb.d + P - 1) / P;
        const int kc = ((pb.d + chunks - 1) / chunks + 1) & ~1;
        double *xs = reinterpret_cast<double *>(lds);
        double *ys = xs + ROWS * P;
        stage<ROWS, (ROWS * P / 2 + 255) / 256>(pb.X, pb.n_i, i0, pb.d, 0, min(kc, pb.d), xs);
        stage<COLS, (COLS * P / 2 + 255) / 256>(pb.Y, pb.n_j, j0, pb.d, 0, min(kc, pb.d), ys);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NE; ++e) v[e] = 0.0;
        const double *xk = xs + ty * P, *yk = ys + tx * P;
        for (int k0 = 0;;) {
            const int km = min(kc, pb.d - k0);
            Operands a, b;
            a.load(xk, yk);
            for (int k = 0; k < km; k += 2) {  // an odd km ends on a staged zero: it adds 0
                b.load(xk + k + 1, yk + k + 1);
                step(a);
                const int kn = min(k + 2, km - 1);
                a.load(xk + kn, yk + kn);
                step(b);
            }
            k0 += kc;
            __syncthreads();
            if (k0 >= pb.d) break;
            stage<ROWS, 3>(pb.X, pb.n_i, i0, pb.d, k0, min(kc, pb.d - k0), xs);
            stage<COLS, 3>(pb.Y, pb.n_j, j0, pb.d, k0, min(kc, pb.d - k0), ys);
            __syncthreads();
        }
    }
};
using F64Tile = F64TileOf<8, 4>;
using F64SmallTile = F64TileOf<4, 2>;

// Distances that lie in memory, a wave's lanes along the columns.
struct StoredTile {
    static constexpr int ROWS = 128, COLS = 64, NE = 32, WAVES = 4;
    static constexpr size_t LDS = 0;
    double v[NE];
    int i0, j0;

    __device__ int row(int e) const { return i0 + ((int)threadIdx.x >> 6) * NE + e; }
    __device__ int col(int) const { return j0 + ((int)threadIdx.x & 63); }

    __device__ void compute(const DistanceProblem &pb, int ti, int tj, unsigned char *) {
        i0 = ti * ROWS;
        j0 = tj * COLS;
        const double *p = pb.D + min(col(0), pb.n_j - 1);
#pragma unroll
        for (int e = 0; e < NE; ++e) v[e] = p[(int64_t)min(row(e), pb.n_i - 1) * pb.n_j];
    }
};

// Split-BF16 cross term on the matrix cores: v_mfma_f32_32x32x16_bf16, lane l
// supplies row l%32 and k = 8*(l/32)..+7 of A, column l%32 and the same k of B;
// accumulator register r holds row 8*(r/4) + 4*(l/32) + r%4, column l%32.  Four
// waves own 64 x 64 quadrants of a 128 x 128 tile; K (the PCA dimension, padded
// to a multiple of 16) is read straight from global memory.
template <int TERMS>
struct Bf16Tile {
    static constexpr int ROWS = 128, COLS = 128, NE = 64, WAVES = 2;
    static constexpr size_t LDS = 0;
    double v[NE];
    int m0, n0;

    __device__ int row(int e) const {
        const int lane = threadIdx.x & 63, r = e & 15;
        return m0 + (e >> 5) * 32 + 8 * (r / 4) + 4 * (lane >> 5) + (r % 4);
    }
    __device__ int col(int e) const { return n0 + ((e >> 4) & 1) * 32 + (threadIdx.x & 31); }

    __device__ void compute(const DistanceProblem &pb, int ti, int tj, unsigned char *) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        m0 = ti * ROWS + (wave >> 1) * 64;
        n0 = tj * COLS + (wave & 1) * 64;
        const int lr = lane & 31, kg = (lane >> 5) * 8;
        floatx16 acc[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
        for (int k0 = 0; k0 < pb.kp; k0 += 16) {
            bf16x8 ah[2], am[2], al[2], bh[2], bm[2], bl[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int64_t o = (int64_t)min(m0 + a * 32 + lr, pb.n_i - 1) * pb.kp + k0 + kg;
                ah[a] = *reinterpret_cast<const bf16x8 *>(pb.xs.h + o);
                am[a] = *reinterpret_cast<const bf16x8 *>(pb.xs.m + o);
                if (TERMS == 6) al[a] = *reinterpret_cast<const bf16x8 *>(pb.xs.l + o);
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int64_t o = (int64_t)min(n0 + b * 32 + lr, pb.n_j - 1) * pb.kp + k0 + kg;
                bh[b] = *reinterpret_cast<const bf16x8 *>(pb.ys.h + o);
                bm[b] = *reinterpret_cast<const bf16x8 *>(pb.ys.m + o);
                if (TERMS == 6) bl[b] = *reinterpret_cast<const bf16x8 *>(pb.ys.l + o);
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    // smallest products first: they are accumulated before the large hi.hi term
                    if (TERMS == 6) {
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[a], bm[b], acc[a][b], 0, 0, 0);
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[a], bh[b], acc[a][b], 0, 0, 0);
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a], bl[b], acc[a][b], 0, 0, 0);
                    }
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am[a], bh[b], acc[a][b], 0, 0, 0);
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a], bm[b], acc[a][b], 0, 0, 0);
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[a], bh[b], acc[a][b], 0, 0, 0);
                }
        }
        double nx[2][16], ny[2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 16; ++r) nx[a][r] = pb.xs.norm[min(row(a * 32 + r), pb.n_i - 1)];
#pragma unroll
        for (int b = 0; b < 2; ++b) ny[b] = pb.ys.norm[min(col(b * 16), pb.n_j - 1)];
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int a = e >> 5, b = (e >> 4) & 1, r = e & 15;
            v[e] = fmax(nx[a][r] + ny[b] - 2.0 * (double)acc[a][b][r], 0.0);
        }
    }
};

// ---------------------------------------------------------------------------
// median state and buffers
// ---------------------------------------------------------------------------
// candidate lists (one append counter each, spread over the tiles), at most; 16 below 2^22 entries, where
// a tile's worth of slack in each would be most of the workspace
constexpr int kSegments = 256;
constexpr int kCandBins = 4096;
constexpr int kListCap = 1 << 18, kListMost = 1 << 20;  // entries of the middle bins, at least and at most
constexpr int kRadixBins = 2048;
// Pairs up to this many entries: every entry is a candidate, and one workgroup selects among all of
// them (us for cost and median, so / with the bracket; normal, then integer coordinates: 120 x 127
// 95 / 120, 99 / 118; 150 x 157 107 / 121, 115 / 116; 180 x 187 120 / 122, 135 / 118; 300 x 307 197 / 123).
constexpr int64_t kCollectAll = 3 << 13;
// Above this many entries the candidate lists (2 bytes per entry) are not worth their
// memory: one more regeneration (0.4 ms per 2^28 entries) takes their place.
constexpr int64_t kLeanEntries = 1ll << 28;
constexpr int kSamplesSmall = 1 << 14, kSamplesLarge = 1 << 16;

struct MedianState {
    u64 lo, hi;               // bracket, inclusive
    int shift;                // candidate bin = (key - lo) >> shift
    int fallback;             // bracket missed or lists overflowed: radix select with regenerated distances
    unsigned ticket[8];       // last-block election of the multi-block steps
    long long rank;           // of the lower middle value among the kept entries / the list
    u64 list_lo, list_hi;     // keys of the middle bins, inclusive
    unsigned n_list;
    // radix fallback
    u64 prefix, mask, eq, next;
    long long frank;
    // result
    u64 lo_key, hi_key;
    double median;
};

struct MedianBuffers {
    MedianState *st;
    unsigned *key32;          // samples
    unsigned *seg_count;      // per segment, 64 unsigneds apart
    u64 *seg_below;           // per segment, 32 u64 apart
    u64 *hist;                // candidate bins
    u64 *fhist;               // fallback digit bins
    u64 *cand_key, *cand_idx;
    u64 *list_key, *list_idx;
    unsigned seg_cap, list_cap;
    int n_seg, seg_shift;     // 2^(32 - seg_shift) lists
    int n_samples;
    int lean;                 // no candidate lists: a counting pass and a gathering pass
};

static size_t median_carve(Arena &ar, int64_t I, int64_t J, bool lean, MedianBuffers *b) {
    const int64_t n = I * J;
    const bool all = n <= kCollectAll;
    b->lean = !all && (lean || n > kLeanEntries);
    b->n_samples = all ? 0 : (n < (1ll << 22) ? kSamplesSmall : kSamplesLarge);
    b->n_seg = all ? 1 : n < (1ll << 22) ? 16 : kSegments;
    b->seg_shift = b->n_seg == kSegments ? 24 : 28;
    // 12.5 % of the entries (the bracket holds 2.3-4.7 %), spread over the segments, and a tile each
    const int64_t cap = all ? n : b->lean ? 0 : n / 8 + b->n_seg * 16384;
    b->seg_cap = (unsigned)((cap + b->n_seg - 1) / b->n_seg);
    b->st = ar.take<MedianState>(1);
    b->key32 = ar.take<unsigned>(kSamplesLarge);
    b->seg_count = ar.take<unsigned>(kSegments * 64);
    b->seg_below = ar.take<u64>(kSegments * 32);
    b->hist = ar.take<u64>(kCandBins);
    b->fhist = ar.take<u64>(kRadixBins);
    b->cand_key = ar.take<u64>((size_t)b->seg_cap * b->n_seg);
    b->cand_idx = ar.take<u64>((size_t)b->seg_cap * b->n_seg);
    // One distance in 64 may lie in the middle bins: tied ones (integer coordinates: about 1 % each)
    // are then still selected from the list, one workgroup's work, instead of by eight more passes
    // (split bf16, 8000 x 8003, d = 200: 1.7 ms against 4.3).  2.2 million took it 3.5 ms, the passes 1.9.
    b->list_cap = (unsigned)std::max<int64_t>(kListCap, b->lean ? 0 : std::min<int64_t>(n / 64, kListMost));
    b->list_key = ar.take<u64>(b->list_cap);
    b->list_idx = ar.take<u64>(b->list_cap);
    return ar.off;
}

size_t distance_median_bytes(int64_t I, int64_t J, bool lean) {
    Arena ar(nullptr, 0);
    MedianBuffers b;
    return median_carve(ar, I, J, lean, &b) + 256;
}

// inclusive scan over a workgroup; red: one entry per wave
template <typename T>
__device__ inline T block_scan(T x, T *red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const T y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) red[wave] = x;
    __syncthreads();
    T before = 0;
    for (int w = 0; w < wave; ++w) before += red[w];
    __syncthreads();
    return x + before;
}

// true in the workgroup that finishes last, which reads with load_dev what the others added up with
// atomics: each wave has waited for its own by then.  (A fence per thread instead, whose release
// writes back the L2, made a pass over 3000 x 3000 take 130 us, now 50.)
__device__ inline bool last_block(unsigned *ticket, int *flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) *flag = atomicAdd(ticket, 1u) == gridDim.x - 1;
    __syncthreads();
    return *flag != 0;
}

__device__ inline u64 load_dev(const u64 *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline unsigned load_dev(const unsigned *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sampled pairs: high words of their FP64 distances (the BF16 modes' distances
// differ by about 1e-5 of the value, far inside the margin)
__global__ __launch_bounds__(256) void dist_sample_kernel(const double *__restrict__ X, const double *__restrict__ Y,
                                                          const double *__restrict__ D, int n_i, int n_j, int d,
                                                          unsigned *__restrict__ key32) {
    const unsigned t = blockIdx.x * 256 + threadIdx.x;
    // two rounds of a 64-bit mixer (splitmix64's constants): independent row and column draws
    u64 z = (u64)(t + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    const int64_t i = (int64_t)(((z & 0xffffffffull) * (u64)n_i) >> 32);
    const int64_t j = (int64_t)(((z >> 32) * (u64)n_j) >> 32);
    double acc = 0.0;
    if (D) {
        acc = D[i * n_j + j];
    } else {
        for (int k = 0; k < d; ++k) {
            const double q = X[i * d + k] - Y[j * d + k];
            acc = fma(q, q, acc);
        }
    }
    key32[t] = (unsigned)((u64)__double_as_longlong(acc) >> 32);
}

// One workgroup: clears the state and turns the samples into the bracket.  Two
// histogram levels (4096 bins over the samples' key range, then 2048 bins inside
// the bin of either bracket end) place both ends to 2^-23 of the range.
// M: samples per thread, held in registers over the three passes (0: no samples).
template <int M>
__global__ __launch_bounds__(1024) void dist_bracket_kernel(const unsigned *__restrict__ key32, long long rank,
                                                            double n, MedianBuffers b) {
    constexpr int m = M * 1024;
    __shared__ unsigned h[kCandBins];
    __shared__ unsigned red[16], mm[2];
    __shared__ unsigned edge[2], base_rank[2], res[2];
    const int t = threadIdx.x;
    MedianState *st = b.st;
    for (int k = t; k < kSegments * 64; k += 1024) b.seg_count[k] = 0u;
    for (int k = t; k < kSegments * 32; k += 1024) b.seg_below[k] = 0ull;
    for (int k = t; k < kCandBins; k += 1024) b.hist[k] = 0ull;
    for (int k = t; k < kRadixBins; k += 1024) b.fhist[k] = 0ull;
    if (t == 0) {
        st->fallback = 0;
        for (int k = 0; k < 8; ++k) st->ticket[k] = 0u;
        st->rank = rank;
        st->n_list = 0u;
        st->prefix = st->mask = st->eq = 0ull;
        st->next = ~0ull;
        st->frank = rank;
        st->lo = 0ull;
        st->hi = ~0ull;
        st->shift = 52;
        mm[0] = ~0u;
        mm[1] = 0u;
    }
    if constexpr (M == 0) return;
    unsigned x[M ? M : 1];
#pragma unroll
    for (int q = 0; q < M; q += 4) {
        const uint4 y = *reinterpret_cast<const uint4 *>(key32 + q * 1024 + t * 4);
        x[q] = y.x;
        x[q + 1] = y.y;
        x[q + 2] = y.z;
        x[q + 3] = y.w;
    }
    __syncthreads();
    unsigned kmin = ~0u, kmax = 0u;
#pragma unroll
    for (int q = 0; q < M; ++q) {
        kmin = min(kmin, x[q]);
        kmax = max(kmax, x[q]);
    }
    atomicMin(&mm[0], kmin);
    atomicMax(&mm[1], kmax);
    // 6 standard deviations of a quantile of m draws at one half
    const double margin = 3.0 * sqrt((double)m) + 2.0;
    const double centre = (double)rank / n * m;
    const long long want[2] = {(long long)floor(centre - margin), (long long)ceil(centre + margin)};
    for (int k = t; k < kCandBins; k += 1024) h[k] = 0u;
    __syncthreads();
    const unsigned k0 = mm[0], range = mm[1] - mm[0];
    const int s1 = max(0, 32 - __clz(range) - 12);  // (range >> s1) < 4096
#pragma unroll
    for (int q = 0; q < M; ++q) atomicAdd(&h[(x[q] - k0) >> s1], 1u);
    __syncthreads();
    {
        unsigned c[4], mine = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            c[q] = h[4 * t + q];
            mine += c[q];
        }
        unsigned before = block_scan(mine, red) - mine;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
            for (int w = 0; w < 2; ++w)
                if (want[w] >= (long long)before && want[w] < (long long)before + c[q]) {
                    edge[w] = k0 + ((unsigned)(4 * t + q) << s1);
                    base_rank[w] = before;
                }
            before += c[q];
        }
    }
    __syncthreads();
    for (int k = t; k < kCandBins; k += 1024) h[k] = 0u;
    __syncthreads();
    const int s2 = max(0, s1 - 11);
    for (int w = 0; w < 2; ++w) {
        if (want[w] < 0 || want[w] >= m) continue;  // uniform
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const unsigned o = x[q] - edge[w];
            if ((o >> s1) == 0u && x[q] >= edge[w]) atomicAdd(&h[w * 2048 + (o >> s2)], 1u);
        }
    }
    __syncthreads();
    for (int w = 0; w < 2; ++w) {
        if (want[w] < 0 || want[w] >= m) continue;  // uniform
        const unsigned c0 = h[w * 2048 + 2 * t], c1 = h[w * 2048 + 2 * t + 1];
        const unsigned before = block_scan(c0 + c1, red) - (c0 + c1);
        const long long r = want[w] - (long long)base_rank[w];
        if (r >= (long long)before && r < (long long)before + c0) res[w] = 2 * t;
        else if (r >= (long long)before + c0 && r < (long long)before + c0 + c1) res[w] = 2 * t + 1;
    }
    __syncthreads();
    if (t == 0) {
        const u64 lo = want[0] < 0 ? 0ull : (u64)(edge[0] + (res[0] << s2)) << 32;
        const u64 hi = want[1] >= m ? ~0ull
                                    : (((u64)(edge[1] + (res[1] << s2)) + (1ull << s2)) << 32) - 1ull;
        st->lo = lo;
        st->hi = hi;
        st->shift = max(0, 64 - __clzll(hi - lo) - 12);  // ((hi - lo) >> shift) < 4096
    }
}

// ---------------------------------------------------------------------------
// passes over the regenerated tiles
// ---------------------------------------------------------------------------
enum PassMode { kCollect, kBins, kGather, kDigit, kNextAbove, kIndex };

struct PassArgs {
    DistanceProblem pb;
    MedianBuffers b;
    int tiles_i, tiles_j;
    int shift, width, last;   // kDigit
    long long rank;
    int odd;
    u64 *index_out;
};

// Every pass: entries of tile after tile.
//   kCollect   candidates to the segment lists (a workgroup per tile)
//   kBins      candidates counted per bin only; kGather: those of the middle
//              bins to the list (two regenerations, no candidate storage)
//   kDigit, kNextAbove, kIndex   the fallback; they leave at once unless the flag is set
template <class Tile, int MODE>
__global__ __launch_bounds__(256, MODE == kBins || MODE == kDigit ? 2 : Tile::WAVES) void dist_pass_kernel(PassArgs pa) {
    constexpr int NH = MODE == kDigit ? kRadixBins : MODE == kBins ? kCandBins : 1;
    __shared__ __align__(16) unsigned char lds[Tile::LDS ? Tile::LDS : 16];
    __shared__ unsigned h[NH];
    __shared__ unsigned wsum[4], wbase;
    __shared__ u64 wbelow[4];
    __shared__ int is_last;
    MedianState *st = pa.b.st;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (MODE >= kDigit && !st->fallback) return;
    if (MODE == kGather && st->fallback) return;
    if (NH > 1) {
        for (int q = tid; q < NH; q += 256) h[q] = 0u;
        __syncthreads();
    }
    const u64 lo = MODE == kGather ? st->list_lo : st->lo, hi = MODE == kGather ? st->list_hi : st->hi;
    const int bin_shift = st->shift;
    u64 below_all = 0;
    const u64 prefix = st->prefix, mask = st->mask;
    const u64 lo_key = st->lo_key, hi_key = st->hi_key;
    u64 best = ~0ull, best_hi = ~0ull;
    // Equal bins one after the other go to LDS as one add: where distances are tied, all lanes of a
    // wave meet in one bin, entry after entry.
    int run_bin = -1;
    unsigned run = 0;
    auto count_bin = [&](int bin) {
        if (bin != run_bin) {
            if (run) atomicAdd(&h[run_bin], run);
            run_bin = bin;
            run = 0;
        }
        ++run;
    };
    const int64_t n_tiles = (int64_t)pa.tiles_i * pa.tiles_j;
    for (int64_t t = blockIdx.x; t < n_tiles; t += gridDim.x) {
        Tile tile;
        tile.compute(pa.pb, (int)(t / pa.tiles_j), (int)(t % pa.tiles_j), lds);
        if constexpr (MODE == kCollect || MODE == kGather) {
            unsigned below = 0;
            u64 keep = 0;  // bit e: entry e is a candidate
#pragma unroll
            for (int e = 0; e < Tile::NE; ++e) {
                const u64 k = (u64)__double_as_longlong(tile.v[e]);
                const bool in = tile.row(e) < pa.pb.n_i && tile.col(e) < pa.pb.n_j;
                below += in && k < lo;
                keep |= (u64)(in && k >= lo && k <= hi) << e;
            }
            if (MODE == kGather && !__syncthreads_or(keep != 0)) continue;  // most tiles hold none
            const unsigned mine = (unsigned)__popcll(keep);
            unsigned incl = mine;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned y = __shfl_up(incl, off);
                if (lane >= off) incl += y;
            }
            unsigned bel = below;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) bel += __shfl_xor(bel, off);
            if (lane == 63) {
                wsum[wave] = incl;
                wbelow[wave] = bel;
            }
            __syncthreads();
            // lists spread over the tiles by a multiplicative hash, so that runs of similar tiles
            // (cells sorted by cluster) do not fill one segment
            const int seg = pa.b.n_seg == 1 ? 0 : (int)(((unsigned)t * 2654435761u) >> pa.b.seg_shift);
            if (tid == 0) {
                const unsigned all = wsum[0] + wsum[1] + wsum[2] + wsum[3];
                if (MODE == kCollect) {
                    wbase = atomicAdd(&pa.b.seg_count[seg * 64], all);
                    atomicAdd(&pa.b.seg_below[seg * 32], wbelow[0] + wbelow[1] + wbelow[2] + wbelow[3]);
                } else if (all) {  // one add per tile: an add per entry took 11 ns, one after the other
                    wbase = atomicAdd(&st->n_list, all);
                }
            }
            __syncthreads();
            unsigned at = wbase + incl - mine;
            for (int w = 0; w < wave; ++w) at += wsum[w];
            if (mine) {
                const int64_t seg0 = (int64_t)seg * pa.b.seg_cap;
                const unsigned cap = MODE == kCollect ? pa.b.seg_cap : pa.b.list_cap;
                u64 *ck = MODE == kCollect ? pa.b.cand_key + seg0 : pa.b.list_key;
                u64 *ci = MODE == kCollect ? pa.b.cand_idx + seg0 : pa.b.list_idx;
#pragma unroll
                for (int g = 0; g < Tile::NE; g += 8) {
                    if (((keep >> g) & 255ull) == 0) continue;
#pragma unroll
                    for (int e = g; e < g + 8; ++e) {
                        if ((keep >> e) & 1ull) {
                            if (at < cap) {
                                ck[at] = (u64)__double_as_longlong(tile.v[e]);
                                ci[at] = (u64)tile.row(e) * (u64)pa.pb.n_j + (u64)tile.col(e);
                            }
                            ++at;
                        }
                    }
                }
            }
            __syncthreads();  // wsum, wbase are rewritten by the next tile
        } else {
#pragma unroll
            for (int e = 0; e < Tile::NE; ++e) {
                if (tile.row(e) >= pa.pb.n_i || tile.col(e) >= pa.pb.n_j) continue;
                const u64 k = (u64)__double_as_longlong(tile.v[e]);
                if (MODE == kBins) {
                    below_all += k < lo;
                    if (k >= lo && k <= hi) count_bin((int)((k - lo) >> bin_shift));
                } else if (MODE == kDigit) {
                    if ((k & mask) == prefix) count_bin((int)((k >> pa.shift) & ((1ull << pa.width) - 1ull)));
                } else if (MODE == kNextAbove) {
                    if (k > prefix && k < best) best = k;
                } else {
                    const u64 idx = (u64)tile.row(e) * (u64)pa.pb.n_j + (u64)tile.col(e);
                    if (k == lo_key && idx < best) best = idx;
                    if (k == hi_key && idx < best_hi) best_hi = idx;
                }
            }
        }
    }
    if constexpr (NH > 1) {
        if (run) atomicAdd(&h[run_bin], run);
        __syncthreads();
    }
    if constexpr (MODE == kBins) {
        for (int q = tid; q < kCandBins; q += 256)
            if (h[q]) atomicAdd(&pa.b.hist[q], (u64)h[q]);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) below_all += __shfl_xor(below_all, off);
        if (lane == 0) atomicAdd(&pa.b.seg_below[(blockIdx.x % kSegments) * 32], below_all);
    }
    if constexpr (MODE == kDigit) {
        for (int q = tid; q < kRadixBins; q += 256)
            if (h[q]) atomicAdd(&pa.b.fhist[q], (u64)h[q]);
        if (!last_block(&st->ticket[0], &is_last)) return;
        // the digit's bin that holds the rank: eight bins per thread
        constexpr int PER = kRadixBins / 256;
        const u64 want = (u64)st->frank;
        u64 c[PER], mine = 0;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            c[q] = load_dev(&pa.b.fhist[PER * tid + q]);
            mine += c[q];
        }
        u64 before = block_scan(mine, wbelow) - mine;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            if (want >= before && want < before + c[q]) {  // one thread, one bin
                st->prefix |= (u64)(PER * tid + q) << pa.shift;
                st->mask |= ((1ull << pa.width) - 1ull) << pa.shift;
                st->frank -= (long long)before;
                if (pa.last) st->eq = c[q];
            }
            before += c[q];
        }
        if (tid == 0) st->ticket[0] = 0u;
        for (int q = tid; q < kRadixBins; q += 256) pa.b.fhist[q] = 0ull;
    }
    if constexpr (MODE == kIndex) {  // one atomic per wave: tied keys are many
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const u64 o = __shfl_xor(best, off), p = __shfl_xor(best_hi, off);
            best = o < best ? o : best;
            best_hi = p < best_hi ? p : best_hi;
        }
        if (lane == 0 && best != ~0ull) atomicMin(&pa.index_out[0], best);
        if (lane == 0 && best_hi != ~0ull) atomicMin(&pa.index_out[1], best_hi);
    }
    if constexpr (MODE == kNextAbove) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const u64 o = __shfl_xor(best, off);
            best = o < best ? o : best;
        }
        if (lane == 0 && best != ~0ull) atomicMin(&st->next, best);
        if (!last_block(&st->ticket[1], &is_last)) return;
        if (tid == 0) {
            // the upper middle value equals the lower one when enough ties remain
            const bool tie = (u64)(st->frank + 1) < st->eq;
            st->lo_key = st->prefix;
            st->hi_key = (pa.odd || tie) ? st->prefix : load_dev(&st->next);
            const double a = __longlong_as_double((long long)st->lo_key);
            st->median = pa.odd ? a : (a + __longlong_as_double((long long)st->hi_key)) / 2.0;
            if (pa.index_out) pa.index_out[0] = pa.index_out[1] = ~0ull;
        }
    }
}

// One 1024-thread workgroup, from the candidates' bins and the counts below the
// bracket: the bins [list_lo, list_hi] that hold the middle rank(s), and the rank
// inside them.
__global__ __launch_bounds__(1024) void place_rank_kernel(MedianBuffers b, int odd) {
    __shared__ u64 red[16];
    __shared__ int over, bin[2];
    __shared__ u64 start[2], end[2];
    const int t = threadIdx.x;
    MedianState *st = b.st;
    if (t == 0) over = 0;
    if (t < 2) bin[t] = -1;
    __syncthreads();
    u64 below = 0;
    if (t < kSegments) {
        below = load_dev(&b.seg_below[t * 32]);
        if (load_dev(&b.seg_count[t * 64]) > b.seg_cap) over = 1;
    }
    const u64 below_all = block_scan(below, red);
    if (t == 1023) start[0] = below_all;
    __syncthreads();
    const long long r = st->rank - (long long)start[0];  // rank of the lower middle among the candidates
    __syncthreads();
    u64 c[4], mine = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        c[q] = load_dev(&b.hist[4 * t + q]);
        mine += c[q];
    }
    u64 before = block_scan(mine, red) - mine;
    const long long want[2] = {r, odd ? r : r + 1};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int w = 0; w < 2; ++w)
            if (want[w] >= (long long)before && want[w] < (long long)(before + c[q])) {
                bin[w] = 4 * t + q;
                start[w] = before;
                end[w] = before + c[q];
            }
        before += c[q];
    }
    __syncthreads();
    if (t == 0) {
        // heavy ties in the middle bins: no list holds them
        if (over || bin[0] < 0 || bin[1] < 0 || end[1] - start[0] > (u64)b.list_cap) {
            st->fallback = 1;
        } else {
            const u64 lo = st->lo;
            st->rank = r - (long long)start[0];
            st->list_lo = lo + ((u64)bin[0] << st->shift);
            st->list_hi = lo + ((u64)bin[1] << st->shift) + ((1ull << st->shift) - 1ull);
        }
    }
}

// candidates' bins over (key - lo) >> shift
__global__ __launch_bounds__(1024) void cand_hist_kernel(MedianBuffers b) {
    __shared__ unsigned h[kCandBins];
    const int t = threadIdx.x;
    MedianState *st = b.st;
    for (int q = t; q < kCandBins; q += 1024) h[q] = 0u;
    __syncthreads();
    const u64 lo = st->lo;
    const int shift = st->shift;
    for (int seg = blockIdx.x; seg < b.n_seg; seg += gridDim.x) {
        const unsigned n = min(b.seg_count[seg * 64], b.seg_cap);
        const u64 *keys = b.cand_key + (int64_t)seg * b.seg_cap;
        for (unsigned e = t; e < n; e += 1024) atomicAdd(&h[(keys[e] - lo) >> shift], 1u);
    }
    __syncthreads();
    for (int q = t; q < kCandBins; q += 1024)
        if (h[q]) atomicAdd(&b.hist[q], (u64)h[q]);
}

// f(e, keys[e]) for the thread's entries, eight loads in flight (one at a time, a list of 600000 tied
// distances took 2 ms)
template <class F>
__device__ inline void each_key(const u64 *keys, unsigned n, F f) {
    for (unsigned e0 = threadIdx.x; e0 < n; e0 += 8 * 1024) {
        u64 x[8];
#pragma unroll
        for (unsigned u = 0; u < 8; ++u) x[u] = e0 + u * 1024 < n ? keys[e0 + u * 1024] : 0ull;
#pragma unroll
        for (unsigned u = 0; u < 8; ++u)
            if (e0 + u * 1024 < n) f(e0 + u * 1024, x[u]);
    }
}

// Exact order statistics of n (key, index) pairs, n >= 1, by one 1024-thread
// workgroup: radix select on key - min, 11 bits a time, then the smallest key
// above and the smallest indices.
__device__ void list_select(const u64 *keys, const u64 *idx, unsigned n, long long rank, int odd, MedianState *st,
                            u64 *index_out) {
    __shared__ unsigned h[kRadixBins];
    __shared__ unsigned red[16];
    __shared__ u64 lo_s, hi_s, above_s, ix[2];
    __shared__ unsigned sel_bin, sel_cum, sel_cnt;
    const int t = threadIdx.x;
    if (t == 0) {
        lo_s = ~0ull;
        hi_s = 0ull;
        above_s = ix[0] = ix[1] = ~0ull;
    }
    __syncthreads();
    u64 a = ~0ull, z = 0ull;
    each_key(keys, n, [&](unsigned, u64 k) {
        a = k < a ? k : a;
        z = k > z ? k : z;
    });
    for (int off = 32; off > 0; off >>= 1) {
        const u64 p = __shfl_xor(a, off), q = __shfl_xor(z, off);
        a = p < a ? p : a;
        z = q > z ? q : z;
    }
    if ((t & 63) == 0) {
        atomicMin(&lo_s, a);
        atomicMax(&hi_s, z);
    }
    __syncthreads();
    u64 base = lo_s, span = hi_s - lo_s;  // keys in [base, base + span]
    unsigned eq = n, r = (unsigned)rank;
    int shift = span ? max(0, 64 - __clzll(span) - 11) : 0;
    while (span) {  // uniform
        for (int q = t; q < kRadixBins; q += 1024) h[q] = 0u;
        __syncthreads();
        each_key(keys, n, [&](unsigned, u64 k) {
            if (k >= base && k - base <= span) atomicAdd(&h[(k - base) >> shift], 1u);
        });
        __syncthreads();
        const unsigned c0 = h[2 * t], c1 = h[2 * t + 1];
        const unsigned before = block_scan(c0 + c1, red) - (c0 + c1);
        if (r >= before && r < before + c0) {
            sel_bin = 2 * t;
            sel_cum = before;
            sel_cnt = c0;
        } else if (r >= before + c0 && r < before + c0 + c1) {
            sel_bin = 2 * t + 1;
            sel_cum = before + c0;
            sel_cnt = c1;
        }
        __syncthreads();
        base += (u64)sel_bin << shift;
        r -= sel_cum;
        eq = sel_cnt;
        span = (1ull << shift) - 1ull;
        shift = max(0, shift - 11);
        __syncthreads();
    }
    // base is the lower middle key, held by eq entries, r of them before the rank
    u64 above = ~0ull;
    if (!odd && r + 1 >= eq) {
        each_key(keys, n, [&](unsigned, u64 k) {
            if (k > base && k < above) above = k;
        });
        for (int off = 32; off > 0; off >>= 1) {
            const u64 p = __shfl_xor(above, off);
            above = p < above ? p : above;
        }
        if ((t & 63) == 0) atomicMin(&above_s, above);
        __syncthreads();
        above = above_s;
    } else {
        above = base;
    }
    if (index_out) {
        u64 i0 = ~0ull, i1 = ~0ull;
        each_key(keys, n, [&](unsigned e, u64 k) {
            if (k == base && idx[e] < i0) i0 = idx[e];
            if (k == above && idx[e] < i1) i1 = idx[e];
        });
        for (int off = 32; off > 0; off >>= 1) {
            const u64 p = __shfl_xor(i0, off), q = __shfl_xor(i1, off);
            i0 = p < i0 ? p : i0;
            i1 = q < i1 ? q : i1;
        }
        if ((t & 63) == 0) {
            atomicMin(&ix[0], i0);
            atomicMin(&ix[1], i1);
        }
        __syncthreads();
        if (t < 2) index_out[t] = ix[t];
    }
    if (t == 0) {
        st->lo_key = base;
        st->hi_key = above;
        const double x = __longlong_as_double((long long)base);
        st->median = odd ? x : (x + __longlong_as_double((long long)above)) / 2.0;
    }
}

// entries of the middle bins to the list
__global__ __launch_bounds__(1024) void cand_gather_kernel(MedianBuffers b) {
    MedianState *st = b.st;
    if (st->fallback) return;
    const u64 lo = st->list_lo, hi = st->list_hi;
    for (int seg = blockIdx.x; seg < b.n_seg; seg += gridDim.x) {
        const unsigned n = min(b.seg_count[seg * 64], b.seg_cap);
        const int64_t s0 = (int64_t)seg * b.seg_cap;
        for (unsigned e = threadIdx.x; e < n; e += 1024) {
            const u64 k = b.cand_key[s0 + e];
            if (k >= lo && k <= hi) {
                const unsigned at = atomicAdd(&st->n_list, 1u);
                if (at < b.list_cap) {
                    b.list_key[at] = k;
                    b.list_idx[at] = b.cand_idx[s0 + e];
                }
            }
        }
    }
}

// the one or two middle values among the gathered entries
__global__ __launch_bounds__(1024) void list_select_kernel(MedianBuffers b, int odd, u64 *index_out) {
    MedianState *st = b.st;
    if (st->fallback) return;
    list_select(b.list_key, b.list_idx, st->n_list, st->rank, odd, st, index_out);
}

// pairs of at most kCollectAll entries: select straight from the one list
__global__ __launch_bounds__(1024) void all_select_kernel(MedianBuffers b, int odd, u64 *index_out) {
    list_select(b.cand_key, b.cand_idx, b.seg_count[0], b.st->rank, odd, b.st, index_out);
}

template <class Tile>
static int median_passes(const DistanceProblem &pb, const MedianBuffers &b, int64_t *index_out, hipStream_t s) {
    const long long n = (long long)pb.n_i * pb.n_j;
    const long long rank = (n % 2) ? n / 2 : n / 2 - 1;
    const int odd = (int)(n % 2);
    u64 *idx = reinterpret_cast<u64 *>(index_out);
    if (b.n_samples)
        dist_sample_kernel<<<b.n_samples / 256, 256, 0, s>>>(pb.X, pb.Y, pb.D, pb.n_i, pb.n_j, pb.d, b.key32);
    if (b.n_samples == kSamplesLarge)
        dist_bracket_kernel<kSamplesLarge / 1024><<<1, 1024, 0, s>>>(b.key32, rank, (double)n, b);
    else if (b.n_samples == kSamplesSmall)
        dist_bracket_kernel<kSamplesSmall / 1024><<<1, 1024, 0, s>>>(b.key32, rank, (double)n, b);
    else
        dist_bracket_kernel<0><<<1, 1024, 0, s>>>(b.key32, rank, (double)n, b);
    PassArgs pa{pb, b, (pb.n_i + Tile::ROWS - 1) / Tile::ROWS, (pb.n_j + Tile::COLS - 1) / Tile::COLS, 0, 0, 0, rank,
                odd, idx};
    const int64_t tiles = (int64_t)pa.tiles_i * pa.tiles_j;
    const unsigned grid = (unsigned)std::min<int64_t>(tiles, 1024);
    if (b.lean) {
        dist_pass_kernel<Tile, kBins><<<grid, 256, 0, s>>>(pa);
        place_rank_kernel<<<1, 1024, 0, s>>>(b, odd);
        dist_pass_kernel<Tile, kGather><<<grid, 256, 0, s>>>(pa);
        list_select_kernel<<<1, 1024, 0, s>>>(b, odd, idx);
    } else {
        dist_pass_kernel<Tile, kCollect><<<(unsigned)std::min<int64_t>(tiles, 1 << 20), 256, 0, s>>>(pa);
        if (b.n_samples) {
            cand_hist_kernel<<<b.n_seg, 1024, 0, s>>>(b);
            place_rank_kernel<<<1, 1024, 0, s>>>(b, odd);
            cand_gather_kernel<<<b.n_seg, 1024, 0, s>>>(b);
            list_select_kernel<<<1, 1024, 0, s>>>(b, odd, idx);
        }
    }
    if (!b.n_samples) {
        all_select_kernel<<<1, 1024, 0, s>>>(b, odd, idx);
        WOTK_LAUNCH_CHECK();
        return WOTK_OK;
    }
    static const int shifts[6] = {53, 42, 31, 20, 10, 0}, widths[6] = {11, 11, 11, 11, 10, 10};
    for (int p = 0; p < 6; ++p) {
        pa.shift = shifts[p];
        pa.width = widths[p];
        pa.last = p == 5;
        dist_pass_kernel<Tile, kDigit><<<grid, 256, 0, s>>>(pa);
    }
    dist_pass_kernel<Tile, kNextAbove><<<grid, 256, 0, s>>>(pa);
    if (idx) dist_pass_kernel<Tile, kIndex><<<grid, 256, 0, s>>>(pa);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

int distance_median(const DistanceProblem &pb, bool lean, void *workspace, int64_t *index_out, const double **median,
                    hipStream_t s) {
    Arena ar(workspace, distance_median_bytes(pb.n_i, pb.n_j, lean));
    MedianBuffers b;
    median_carve(ar, pb.n_i, pb.n_j, lean, &b);
    *median = &b.st->median;
    if (pb.D) return median_passes<StoredTile>(pb, b, index_out, s);
    if (pb.terms == 0) return median_passes<F64Tile>(pb, b, index_out, s);
    if (pb.terms == 3) return median_passes<Bf16Tile<3>>(pb, b, index_out, s);
    return median_passes<Bf16Tile<6>>(pb, b, index_out, s);
}

// ---------------------------------------------------------------------------
// cost write: C and C^T in FP32 from the regenerated tile
// ---------------------------------------------------------------------------
// c / m as the FP64 division rounds it: q = c * (1/m) and one residual step.  For a
// median outside the normal range (0, subnormal, infinite, NaN) the division itself.
struct Divisor {
    double m, inv;
    bool plain;
    __device__ explicit Divisor(double v) : m(v), inv(1.0 / v), plain(!(v > 1e-290 && v < 1e290)) {}
    __device__ float operator()(double c) const {
        if (plain) return (float)(c / m);
        const double q = c * inv;
        return (float)(isfinite(q) ? fma(fma(-q, m, c), inv, q) : q);
    }
};

struct CostWriteArgs {
    DistanceProblem pb;
    int tiles_j;
    const double *median;
    float *C;
    int64_t ldc;
    float *CT;
    int64_t ldct;
};

// FP64 tiles: C goes out from the registers, C^T through LDS as float4 along the rows.
__global__ __launch_bounds__(256, F64Tile::WAVES) void cost_write_f64_kernel(CostWriteArgs ca) {
    constexpr int P = F64Tile::ROWS + 4;  // float pitch of the transposed tile
    static_assert(sizeof(float) * F64Tile::COLS * P <= F64Tile::LDS, "the transposed tile reuses the staging LDS");
    __shared__ __align__(16) unsigned char lds[F64Tile::LDS];
    F64Tile t;
    t.compute(ca.pb, (int)(blockIdx.x / ca.tiles_j), (int)(blockIdx.x % ca.tiles_j), lds);
    const Divisor div(*ca.median);
    const int n_i = ca.pb.n_i, n_j = ca.pb.n_j;
    const int pad_j = (n_j + 3) & ~3, pad_i = (n_i + 3) & ~3;
    float *tt = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int a = 0; a < 8; ++a) {
        const int i = t.row(4 * a);
        float *crow = ca.C + (int64_t)i * ca.ldc + t.col(0);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int j = t.col(b);
            const float o = (i < n_i && j < n_j) ? div(t.v[4 * a + b]) : 0.f;
            if (i < n_i && j < pad_j) crow[16 * b] = o;
            tt[(t.tx + 16 * b) * P + t.ty + 16 * a] = o;
        }
    }
    __syncthreads();
    const int ri = (threadIdx.x & 31) * 4;
#pragma unroll 4
    for (int c = threadIdx.x >> 5; c < F64Tile::COLS; c += 8) {
        const int j = t.j0 + c;
        if (j < n_j && t.i0 + ri < pad_i)
            *reinterpret_cast<float4 *>(ca.CT + (int64_t)j * ca.ldct + t.i0 + ri) =
                *reinterpret_cast<const float4 *>(tt + c * P + ri);
    }
}

// MFMA tiles: a register group holds 4 consecutive rows of one column, so C^T
// goes out as float4 directly and C through LDS, one 64 x 32 piece per wave.
template <int TERMS>
__global__ __launch_bounds__(256) void cost_write_bf16_kernel(CostWriteArgs ca) {
    constexpr int P = 36;  // float pitch of a wave's 64 x 32 piece
    __shared__ __align__(16) float tt[4][64 * P];
    Bf16Tile<TERMS> t;
    t.compute(ca.pb, (int)(blockIdx.x / ca.tiles_j), (int)(blockIdx.x % ca.tiles_j), nullptr);
    const Divisor div(*ca.median);
    const int n_i = ca.pb.n_i, n_j = ca.pb.n_j;
    const int pad_j = (n_j + 3) & ~3, pad_i = (n_i + 3) & ~3;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *mine = tt[wave];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int j = t.n0 + b * 32 + (lane & 31);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int lr = a * 32 + 8 * g + 4 * (lane >> 5);  // first of 4 rows, inside the quadrant
                float o[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    o[q] = (t.m0 + lr + q < n_i && j < n_j) ? div(t.v[a * 32 + b * 16 + g * 4 + q]) : 0.f;
                    mine[(lr + q) * P + (lane & 31)] = o[q];
                }
                if (j < n_j && t.m0 + lr < pad_i)
                    *reinterpret_cast<float4 *>(ca.CT + (int64_t)j * ca.ldct + t.m0 + lr) =
                        make_float4(o[0], o[1], o[2], o[3]);
            }
        __syncthreads();
        const int cc = (lane & 7) * 4;
#pragma unroll
        for (int r = lane >> 3; r < 64; r += 8) {
            const int i = t.m0 + r, jj = t.n0 + b * 32 + cc;
            if (i < n_i && jj < pad_j)
                *reinterpret_cast<float4 *>(ca.C + (int64_t)i * ca.ldc + jj) =
                    *reinterpret_cast<const float4 *>(mine + r * P + cc);
        }
        __syncthreads();
    }
}

int launch_cost_write(const DistanceProblem &pb, const double *median, float *C, int64_t ldc, float *CT,
                      int64_t ldct, hipStream_t s) {
    const int rows = pb.terms == 0 ? F64Tile::ROWS : Bf16Tile<6>::ROWS;
    const int cols = pb.terms == 0 ? F64Tile::COLS : Bf16Tile<6>::COLS;
    const int tj = (int)((round_up(pb.n_j, 4) + cols - 1) / cols), ti = (int)((round_up(pb.n_i, 4) + rows - 1) / rows);
    const int64_t tiles = (int64_t)ti * tj;
    WOTK_REQUIRE(tiles < (1ll << 31), "cost matrix too large");
    const CostWriteArgs ca{pb, tj, median, C, ldc, CT, ldct};
    if (pb.terms == 0) cost_write_f64_kernel<<<(unsigned)tiles, 256, 0, s>>>(ca);
    else if (pb.terms == 3) cost_write_bf16_kernel<3><<<(unsigned)tiles, 256, 0, s>>>(ca);
    else cost_write_bf16_kernel<6><<<(unsigned)tiles, 256, 0, s>>>(ca);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

// the FP64 distances as they are
template <class Tile>
__global__ __launch_bounds__(256, Tile::WAVES) void dist_store_kernel(DistanceProblem pb, int tiles_j,
                                                                      double *__restrict__ D, int64_t ld) {
    __shared__ __align__(16) unsigned char lds[Tile::LDS ? Tile::LDS : 16];
    Tile t;
    t.compute(pb, (int)(blockIdx.x / tiles_j), (int)(blockIdx.x % tiles_j), lds);
#pragma unroll
    for (int e = 0; e < Tile::NE; ++e)
        if (t.row(e) < pb.n_i && t.col(e) < pb.n_j) D[(int64_t)t.row(e) * ld + t.col(e)] = t.v[e];
}

template <class Tile>
static int64_t tiles_of(const DistanceProblem &pb) {
    return (((int64_t)pb.n_i + Tile::ROWS - 1) / Tile::ROWS) * (((int64_t)pb.n_j + Tile::COLS - 1) / Tile::COLS);
}

template <class Tile>
static int launch_store(const DistanceProblem &pb, double *D, int64_t ld, hipStream_t s) {
    const int64_t tiles = tiles_of<Tile>(pb);
    WOTK_REQUIRE(tiles < (1ll << 31), "cost matrix too large");
    dist_store_kernel<Tile><<<(unsigned)tiles, 256, 0, s>>>(pb, (pb.n_j + Tile::COLS - 1) / Tile::COLS, D, ld);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

// one tile per CU at most: a fourth of the tile (us, 128 x 64 / 64 x 32: 300 x 303, d = 200 71 / 46; 1000 x
// 1003, d = 30 31 / 28, d = 1000 288 / 179; at 512 tiles, 2000 x 2003, 38 / 39, 430 / 455)
constexpr int64_t kSmallTiles = 256;

int launch_distances(const DistanceProblem &pb, double *D, int64_t ld, hipStream_t s) {
    if (pb.terms == 3) return launch_store<Bf16Tile<3>>(pb, D, ld, s);
    if (pb.terms == 6) return launch_store<Bf16Tile<6>>(pb, D, ld, s);
    if (tiles_of<F64Tile>(pb) <= kSmallTiles) return launch_store<F64SmallTile>(pb, D, ld, s);
    return launch_store<F64Tile>(pb, D, ld, s);
}

int launch_sqeuclid_f64(const double *X, const double *Y, int64_t I, int64_t J, int64_t d, double *C64, int64_t ld,
                        hipStream_t s) {
    return launch_distances(DistanceProblem{X, Y, (int)I, (int)J, (int)d, 0, 0, {}, {}}, C64, ld, s);
}

// Regenerated or stored once and read twice: 2 d operations per entry against 24 bytes (us for cost and
// median, regenerated / stored).  FP64: d = 50 at 5000 x 5003 424 / 393, at 15000 x 15003 2475 / 2503; d = 64 482 /
// 418 and 3060 / 2793; d = 200 1203 / 726 and 8018 / 5405.  Split bf16, whose products cost less: 1000 x 1003 d = 64
// 234 / 223, 3000 x 3003 d = 100 415 / 375; 15000 x 15003 d = 160 2634 / 2974, d = 200 3294 / 3303, d = 300 4516 / 3920.
bool distances_stored(const DistanceProblem &pb) {
    const bool small = (int64_t)pb.n_i * pb.n_j <= 1 << 24;
    return pb.d > (pb.terms == 0 || small ? 64 : 256);
}

}  // namespace wotk
