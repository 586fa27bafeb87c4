// Squared distances of a day pair regenerated tile by tile (distance.hip), for
// the stored cost (cost.hip) and the never-stored solver (fused.hip).  Not part
// of the C ABI.
#pragma once
#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "common.h"

namespace wotk {

// hi / mid / lo bf16 parts of the centred coordinates (n x kp, zero-padded)
// and their FP64 squared norms
struct SplitCoords {
    const __bf16 *h, *m, *l;
    const double *norm;
};

// The distances of one day pair.  terms = 0: FP64 direct differences
// sum_k (x_k - y_k)^2, k ascending; 3 or 6: |x|^2 + |y|^2 - 2 x.y with the
// cross term from split-BF16 MFMA products of the centred coordinates.
struct DistanceProblem {
    const double *X, *Y;
    int n_i, n_j, d;
    int terms;
    int kp;
    SplitCoords xs, ys;
    const double *D = nullptr;  // stored (I x J, contiguous): read instead of formed
};

// split-BF16 preparation of pb (terms 3 or 6) into scratch (cost_mfma.hip)
size_t cost_bf16_scratch(int64_t I, int64_t J, int64_t d);
int prepare_split(DistanceProblem *pb, void *scratch, hipStream_t s);

// workspace of distance_median; lean: a fixed few MB, for one more pass over the distances
size_t distance_median_bytes(int64_t I, int64_t J, bool lean);

// exact numpy-style median of the I x J distances (and, if index_out is not
// null, the smallest flat indices holding the lower / upper middle value)
int distance_median(const DistanceProblem &pb, bool lean, void *workspace, int64_t *index_out,
                    const double **median, hipStream_t s);

// FP32 C (I x J) and C^T (J x I) = distance / *median; padding columns up to
// the next multiple of 4 are written as 0
int launch_cost_write(const DistanceProblem &pb, const double *median, float *C, int64_t ldc, float *CT,
                      int64_t ldct, hipStream_t s);

// whether pb's distances are formed once and stored in FP64 for the median and the cost
bool distances_stored(const DistanceProblem &pb);

// the FP64 distances themselves to D (I x J, ld)
int launch_distances(const DistanceProblem &pb, double *D, int64_t ld, hipStream_t s);
int launch_sqeuclid_f64(const double *X, const double *Y, int64_t I, int64_t J, int64_t d, double *C64, int64_t ld,
                        hipStream_t s);

}  // namespace wotk
