// Whole solves of small pairs in one persistent launch (resident.hip), for the
// entry points in sinkhorn.hip.  Not part of the C ABI.
#pragma once
#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "common.h"

namespace wotk {

// how long a workgroup waits for a value and how much one launch does
struct ResidentLimits {
    // 0.1 s of the 100 MHz clock, looked at every 256 polls: a value takes some us, so a longer wait is
    // for workgroups without CUs, and sweeps get on beside whatever has them
    long long wait_ticks = 10000000ll;
    unsigned look_mask = 255;
    // 10 to 30 ms, so that no launch holds the chip, or a hardware queue that other streams share, for
    // long; the next launch costs about 40 us
    long long launch_iters = 2048;
};

// whether pairs of this shape take the resident solver
bool resident_fits(int64_t I, int64_t J);

// bytes of its exchange buffers
size_t resident_bytes(int64_t I, int64_t J);

struct ResidentProblem {
    const float *C;   // I x J, ldc
    int64_t ldc;
    const float *CT;  // J x I, ldct
    int64_t ldct;
    int n_i, n_j;
    const double *G;
    const double *logp;  // log G_i
    const double *misc;  // [0] log mean G, [1] mean G
    double *f, *g;       // potentials: start values in, results out
    double *u, *v;       // absorbed potentials where a launch of the duality-gap schedule stopped
    void *exchange;      // resident_bytes
};

// outcome of a resident solve (device side, copied back by the caller)
struct ResidentResult {
    int aborted;          // a wait ran out: nothing else is valid, solve again by launches
    int max_iter_reached;
    long long launches;   // of this solve, all ended but the last when aborted
    long long iterations, stabilisations, checks;
    double gap, primal, dual, eps;
    // duality-gap schedule: the launch has done its iterations and the next one goes on from f, g, u,
    // v, this scaling, so many iterations into its batch
    int stopped, scaling;
    long long in_batch;
    double sum_ktilde;
};

// The fixed-iteration schedule (optimal_transport.py:167-236).  *launched is 0 when the
// device cannot hold all workgroups at once: nothing ran.
int resident_fixed(const ResidentProblem &rp, double lambda1, double lambda2, double epsilon, double epsilon0,
                   int64_t scaling_iter, int64_t inner_iter_max, int64_t extra_iter, const ResidentLimits &lim,
                   int *launched, hipStream_t s);

// the duality-gap schedule (optimal_transport.py:67-164) up to its last iteration; *out is its
// outcome when *launched (waits for it)
int resident_gap(const ResidentProblem &rp, double lambda1, double lambda2, double epsilon, long long batch_size,
                 double tolerance, double tau, double epsilon0, long long max_iter, const ResidentLimits &lim,
                 int *launched, ResidentResult *out, hipStream_t s);

// leaves the result of no launch on rp, for a solve that does not take the resident solver
int resident_pass_by(const ResidentProblem &rp, hipStream_t s);

// the result of the last resident launch on rp (waits for it)
int resident_result(const ResidentProblem &rp, ResidentResult *out, hipStream_t s);

}  // namespace wotk
