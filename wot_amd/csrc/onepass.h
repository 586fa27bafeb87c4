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

// The tau check (optimal_transport.py:137-141) inside the iteration: the largest growth
// max((f - u)/eps, (g - v)/eps) of an iteration goes to *cur as an ordered key; the next
// iteration (prev = this cur) sees whether it exceeded tau and absorbs u = f, v = g of the
// iteration before while it updates them.
struct TauTrack {
    const unsigned long long *prev;  // null: no tracking
    unsigned long long *cur;
    double tau, inv_eps;
    double *u, *v;
    long long *counter;              // absorptions
};

// double <-> ordered unsigned key
__host__ __device__ inline unsigned long long tau_key(double m) {
    union { double d; unsigned long long b; } x{m};
    return x.b >> 63 ? ~x.b : x.b | (1ull << 63);
}
__host__ __device__ inline double tau_value(unsigned long long k) {
    union { unsigned long long b; double d; } x{k >> 63 ? k & ~(1ull << 63) : ~k};
    return x.d;
}
// whether the iteration that left this key exceeded tau (no iteration yet: no)
__device__ inline bool tau_fired(unsigned long long key, double tau) {
    const double m = tau_value(key);
    return m > -INFINITY && exp(m) > tau;
}

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
    TauTrack tau;
    const int *skip;         // device flag: the launches do nothing when it is set (null: never)
};

// f from g, then g from f, at eps
int one_pass_iterate(const OnePass &op, double lambda1, double lambda2, double eps, hipStream_t s);

}  // namespace wotk
