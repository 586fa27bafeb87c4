// One Sinkhorn iteration over one read of the stored cost (onepass.hip), for the
// schedules in sinkhorn.hip.  Not part of the C ABI.
#pragma once
#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "common.h"

namespace wotk {

// whether pairs of this shape take the one-read iteration
bool one_pass_fits(int64_t I, int64_t J);

// floats of the column partials (workgroups x J rounded up to 4)
size_t one_pass_partials(int64_t I, int64_t J);

struct OnePass {
    const float *C;   // I x J, ldc
    int64_t ldc;
    const float *CT;  // J x I, ldct: columns whose one-read sum left the safe range
    int64_t ldct;
    int n_i, n_j;
    double *f, *g;           // potentials, updated in place
    const double *logp;      // log G_i
    const double *logq_dev;  // device scalar log mean G
    float *part;             // one_pass_partials floats
};

// f from g, then g from f, at eps
int one_pass_iterate(const OnePass &op, double lambda1, double lambda2, double eps, hipStream_t s);

}  // namespace wotk
