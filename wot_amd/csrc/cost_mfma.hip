// Squared-Euclidean cost with the cross term on the matrix cores:
//   D_ij = |x_i|^2 + |y_j|^2 - 2 x_i . y_j
// Coordinates are centred on the mean of both days (distances are
// translation invariant; centring shrinks the norms that cancel), norms are
// FP64, and the cross term is a split-BF16 product: x = x_hi + x_mid + x_lo
// with x_hi = bf16(x), x_mid = bf16(x - x_hi), x_lo = bf16(x - x_hi - x_mid),
// accumulated in FP32 as
//   3 terms: x_hi.y_hi + x_hi.y_mid + x_mid.y_hi
//   6 terms: the 3 above + x_hi.y_lo + x_lo.y_hi + x_mid.y_mid
// (every product of combined weight 2^-16 or larger; ~2^-16 and ~2^-24
// relative error of the cross term).
// The products are formed where the distances are used (distance.hip, Bf16Tile);
// here: the mean, the norms and the split.
#include "common.h"
#include "distance.h"

namespace wotk {

// mean of the stacked coordinates: block k reduces column k over both days
__global__ __launch_bounds__(256) void coord_mean_kernel(const double *__restrict__ X, int n_i,
                                                         const double *__restrict__ Y, int n_j, int d,
                                                         double *__restrict__ mean) {
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

// centred FP64 norms and the bf16 hi/mid/lo split, K padded to kp with zeros
__global__ __launch_bounds__(256) void split_bf16_kernel(const double *__restrict__ X, int n, int d, int kp,
                                                         const double *__restrict__ mean, __bf16 *__restrict__ hi,
                                                         __bf16 *__restrict__ mid, __bf16 *__restrict__ lo,
                                                         double *__restrict__ norm) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double acc = 0.0;
    for (int k = 0; k < kp; ++k) {
        const double v = k < d ? X[(int64_t)i * d + k] - mean[k] : 0.0;
        acc = fma(v, v, acc);
        const __bf16 h = (__bf16)(float)v;
        const double r1 = v - (double)(float)h;
        const __bf16 m = (__bf16)(float)r1;
        const __bf16 l = (__bf16)(float)(r1 - (double)(float)m);
        hi[(int64_t)i * kp + k] = h;
        mid[(int64_t)i * kp + k] = m;
        lo[(int64_t)i * kp + k] = l;
    }
    norm[i] = acc;
}

static int64_t padded_k(int64_t d) { return round_up(d, 16); }

size_t cost_bf16_scratch(int64_t I, int64_t J, int64_t d) {
    Arena ar(nullptr, 0);
    const int64_t kp = padded_k(d);
    ar.take<double>(d);
    for (int p = 0; p < 3; ++p) ar.take<__bf16>((size_t)I * kp);
    for (int p = 0; p < 3; ++p) ar.take<__bf16>((size_t)J * kp);
    ar.take<double>(I);
    ar.take<double>(J);
    return ar.off + 256;
}

int prepare_split(DistanceProblem *pb, void *scratch, hipStream_t s) {
    const int64_t I = pb->n_i, J = pb->n_j, d = pb->d;
    WOTK_REQUIRE(d <= 4096, "split-BF16 cost supports d <= 4096");
    const int64_t kp = padded_k(d);
    Arena ar(scratch, cost_bf16_scratch(I, J, d));
    double *mean = ar.take<double>(d);
    __bf16 *xp[3], *yp[3];
    for (int p = 0; p < 3; ++p) xp[p] = ar.take<__bf16>((size_t)I * kp);
    for (int p = 0; p < 3; ++p) yp[p] = ar.take<__bf16>((size_t)J * kp);
    double *nx = ar.take<double>(I);
    double *ny = ar.take<double>(J);
    coord_mean_kernel<<<(unsigned)d, 256, 0, s>>>(pb->X, (int)I, pb->Y, (int)J, (int)d, mean);
    split_bf16_kernel<<<(unsigned)((I + 255) / 256), 256, 0, s>>>(pb->X, (int)I, (int)d, (int)kp, mean, xp[0], xp[1],
                                                                   xp[2], nx);
    split_bf16_kernel<<<(unsigned)((J + 255) / 256), 256, 0, s>>>(pb->Y, (int)J, (int)d, (int)kp, mean, yp[0], yp[1],
                                                                   yp[2], ny);
    WOTK_LAUNCH_CHECK();
    pb->kp = (int)kp;
    pb->xs = SplitCoords{xp[0], xp[1], xp[2], nx};
    pb->ys = SplitCoords{yp[0], yp[1], yp[2], ny};
    return WOTK_OK;
}

}  // namespace wotk
