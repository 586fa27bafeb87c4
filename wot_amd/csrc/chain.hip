// Long-range couplings (wot/tmap/util.py:74-94, wot/tmap/chaining.py:4-40):
// T_0k = T_01 T_12 ... T_(k-1)k, successive transport-map products with no
// normalisation.  FP32 GEMM on the CDNA matrix cores (v_mfma_f32_32x32x2f32).
//
// Bound: the matrix pipe (157 TFLOP/s FP32; one 32x32x2 product per SIMD every 64
// cycles).  A workgroup of four waves owns a 128 x 128 tile, a wave a 64 x 64
// quadrant: per 8 k a wave reads 4 KB from LDS (32 cycles of its rate) for 16
// products (1024 cycles).  K goes through LDS in chunks of 32, double-buffered: the
// next chunk's global loads are issued before this chunk's products and written to
// the other buffer after them, one barrier per chunk, two workgroups per CU.
// A lies in LDS as in memory (row pitch 36: 16-byte reads of 16 consecutive rows hit
// all banks once); a lane's 16 bytes are four products' operands, so the half-wave
// that a 32x32x2 product gives k and k + 1 here holds k and k + 4 -- B's rows are
// read accordingly (pitch +8: k and k + 4 fall on the other 32 banks).
// Where 128 x 128 tiles leave much of the last round of CUs idle, 64 x 64 tiles; below
// one round of those, four groups of waves per tile each take every fourth chunk and
// add up in LDS (fixed order).  12000^3: 130 TFLOP/s (26.5 ms; 54.8 ms with single
// buffers and scalar loads), 5003 x 4000 x 6001: 108 (was 58), 1500^3: 73.
#include <algorithm>

#include "common.h"

namespace wotk {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // any row start

constexpr int kGK = 32;  // K chunk

struct GemmArgs {
    const float *A;
    int64_t lda;
    const float *B;
    int64_t ldb;
    float *C;
    int64_t ldc;
    int M, N, K;
    int tiles_m, tiles_n;
};

// Tile of a workgroup.  Workgroups go to the 8 XCDs round robin; each XCD takes a
// contiguous run of the tiles in bands of 8 tile rows, so that the panels its
// workgroups stream together are shared in its L2.
__device__ inline bool gemm_tile(const GemmArgs &ga, int &tm, int &tn) {
    const int total = ga.tiles_m * ga.tiles_n, per = (total + 7) / 8;
    const int t = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (((int)blockIdx.x >> 3) >= per || t >= total) return false;
    const int band = t / (8 * ga.tiles_n), in = t % (8 * ga.tiles_n);
    const int rows = min(8, ga.tiles_m - 8 * band);
    tm = 8 * band + in % rows;
    tn = in / rows;
    return true;
}

// C (M x N, ldc) = A (M x K, lda) * B (K x N, ldb); all FP32 row-major.
// MFMA 32x32x2 operand layout (lane l of a wave64): A element (row l%32, k l/32),
// B element (k l/32, column l%32); accumulator register r holds row
// 8*(r/4) + 4*(l/32) + r%4, column l%32.
// TM: tile rows and columns; KS: groups of four waves that share the tile's K; BUFS: 1 where K is one
// chunk (half the LDS: twice the workgroups per CU).
template <int TM, int KS, int BUFS>
__global__ __launch_bounds__(256 * KS) void gemm_f32_mfma_kernel(GemmArgs ga) {
    constexpr int NB = TM / 64;          // 32-wide blocks per wave and side
    constexpr int AP = kGK + 4, BP = TM + 8;
    constexpr int BUF = TM * AP + kGK * BP;
    constexpr int U = TM * kGK / 1024;   // 16-byte pieces per thread and operand
    __shared__ __align__(16) float lds[KS][BUFS][BUF];
    int tm, tn;
    if (!gemm_tile(ga, tm, tn)) return;
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, ks = threadIdx.x >> 8;
    const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TM / 2);
    const int m0 = tm * TM, n0 = tn * TM;
    const int lr = lane & 31, lk = lane >> 5;
    const int chunks = (ga.K + kGK - 1) / kGK;
    const int mine = (chunks - ks + KS - 1) / KS;  // chunks ks, ks + KS, ...
    const int rounds = (chunks + KS - 1) / KS;     // barriers are common to all groups

    // this thread's pieces: A rows ar + 32 u at k ak; B rows bk + (1024 / TM) u at column bn
    const int ar = tid >> 3, ak = (tid & 7) * 4;
    const int bk = tid / (TM / 4), bn = (tid % (TM / 4)) * 4;
    constexpr int BS = 1024 / TM;
    f4 ra[U], rb[U];
    const float *arow[U];
#pragma unroll
    for (int u = 0; u < U; ++u) arow[u] = ga.A + (int64_t)min(m0 + ar + 32 * u, ga.M - 1) * ga.lda + ak;
    // Chunks before the last take whole pieces without tests: rows past M repeat the last
    // one, pieces past N the first (their products are not stored), and a piece that
    // straddles N reads on into the next row, which these chunks always have.
    const float *bcol = ga.B + (n0 + bn < ga.N ? n0 + bn : 0);
    const int whole = ga.ldb >= 4 ? chunks - 1 : 0;
    auto fetch = [&](int ch) {
        const int k0 = ch * kGK;
        if (ch < whole) {  // uniform
#pragma unroll
            for (int u = 0; u < U; ++u) ra[u] = *reinterpret_cast<const f4u *>(arow[u] + k0);
#pragma unroll
            for (int u = 0; u < U; ++u)
                rb[u] = *reinterpret_cast<const f4u *>(bcol + (int64_t)(k0 + bk + BS * u) * ga.ldb);
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + bk + BS * u;
                const float *p = ga.B + (int64_t)min(k, ga.K - 1) * ga.ldb;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ra[u][e] = k0 + ak + e < ga.K ? arow[u][k0 + e] : 0.f;
                    rb[u][e] = k < ga.K && n0 + bn + e < ga.N ? p[n0 + bn + e] : 0.f;
                }
            }
        }
    };
    auto commit = [&](int buf) {
        float *as = lds[ks][buf], *bs = as + TM * AP;
#pragma unroll
        for (int u = 0; u < U; ++u) *reinterpret_cast<f4 *>(as + (ar + 32 * u) * AP + ak) = ra[u];
#pragma unroll
        for (int u = 0; u < U; ++u) *reinterpret_cast<f4 *>(bs + (bk + BS * u) * BP + bn) = rb[u];
    };

    floatx16 acc[NB][NB];
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
    if (mine > 0) {
        fetch(ks);
        commit(0);
    }
    __syncthreads();
    for (int i = 0; i < rounds; ++i) {
        const bool more = BUFS > 1 && i + 1 < (KS == 1 ? rounds : mine);
        if (more) fetch(ks + (i + 1) * KS);
        if (KS == 1 || i < mine) {
            const float *as = lds[ks][i & (BUFS - 1)] + (wm + lr) * AP + 4 * lk;
            const float *bs = lds[ks][i & (BUFS - 1)] + TM * AP + 4 * lk * BP + wn + lr;
#pragma unroll
            for (int kk = 0; kk < kGK; kk += 8) {
                f4 av[NB];
                float bv[NB][4];
#pragma unroll
                for (int a = 0; a < NB; ++a) av[a] = *reinterpret_cast<const f4 *>(as + a * 32 * AP + kk);
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int s = 0; s < 4; ++s) bv[b][s] = bs[(kk + s) * BP + b * 32];
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int a = 0; a < NB; ++a)
#pragma unroll
                        for (int b = 0; b < NB; ++b)
                            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[a][s], bv[b][s], acc[a][b], 0, 0, 0);
            }
        }
        if (more) commit((i + 1) & 1);
        __syncthreads();
    }
    if constexpr (KS > 1) {  // the groups' sums, one after the other, through LDS
        float *red = &lds[0][0][0];
        static_assert(KS == 1 || sizeof(float) * KS * TM * TM <= sizeof(lds), "partial tiles fit the staging LDS");
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    red[(((ks * 4 + wave) * NB + a) * NB + b) * 1024 + r * 64 + lane] = acc[a][b][r];
        __syncthreads();
        if (ks > 0) return;
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r)
#pragma unroll
                    for (int g = 1; g < KS; ++g)
                        acc[a][b][r] += red[(((g * 4 + wave) * NB + a) * NB + b) * 1024 + r * 64 + lane];
    }
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = m0 + wm + a * 32 + 8 * (r / 4) + 4 * lk + (r % 4);
                const int col = n0 + wn + b * 32 + lr;
                if (row < ga.M && col < ga.N) ga.C[(int64_t)row * ga.ldc + col] = acc[a][b][r];
            }
}

template <int TM, int KS, int BUFS = 2>
static int launch_gemm(GemmArgs ga, hipStream_t s) {
    ga.tiles_m = (ga.M + TM - 1) / TM;
    ga.tiles_n = (ga.N + TM - 1) / TM;
    const int64_t total = (int64_t)ga.tiles_m * ga.tiles_n;
    WOTK_REQUIRE(total < (1ll << 28), "GEMM output too large");
    gemm_f32_mfma_kernel<TM, KS, BUFS><<<(unsigned)(8 * ((total + 7) / 8)), 256 * KS, 0, s>>>(ga);
    WOTK_LAUNCH_CHECK();
    return WOTK_OK;
}

}  // namespace wotk

using namespace wotk;

extern "C" int wotk_gemm_f32(const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int64_t ldc,
                             int64_t M, int64_t N, int64_t K, void *stream) {
    WOTK_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31),
                 "bad GEMM shape %lld x %lld x %lld", (long long)M, (long long)N, (long long)K);
    WOTK_REQUIRE(lda >= K && ldb >= N && ldc >= N, "leading dimension too small");
    const GemmArgs ga{A, lda, B, ldb, C, ldc, (int)M, (int)N, (int)K, 0, 0};
    hipStream_t s = (hipStream_t)stream;
    const int64_t t128 = ((M + 127) / 128) * ((N + 127) / 128), t64 = ((M + 63) / 64) * ((N + 63) / 64);
    // Rounds of 256 CUs times the tile's area; a 64 x 64 tile's products cost 1.3 times a
    // 128 x 128 tile's (97 against 130 TFLOP/s on full rounds).  Up to one round of 64 x 64
    // tiles, 16 waves on each instead of 4 (700 x 5000 x 700: 103 against 134 us).
    if (t64 <= 256) return launch_gemm<64, 4>(ga, s);
    // one chunk of K: bound by the product's own bytes, small tiles in flight on them (us, 128 x 128 with
    // two buffers / this: 5000 x 5000 x 16 52 / 46, 12000 x 12000 x 1 159 / 145)
    if (K <= kGK) return launch_gemm<64, 1, 1>(ga, s);
    const double c128 = 4.0 * (double)((t128 + 255) / 256), c64 = 1.3 * (double)((t64 + 255) / 256);
    return c128 <= c64 ? launch_gemm<128, 1>(ga, s) : launch_gemm<64, 1>(ga, s);
}
