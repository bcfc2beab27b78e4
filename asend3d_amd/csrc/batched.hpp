// Batched multi-right-hand-side solver over many design variants (definitions
// in batched.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <vector>

#include "kernels.hpp"

namespace asend {

constexpr int kNrhs = 16;  // right-hand sides per variant advanced together

// Device view of one assembled variant (owned by its context).
struct OperatorView {
    int n_rows = 0;                 // block rows (nodes)
    int n_slices = 0;
    const int32_t* order = nullptr;   // batch_row_order (host)
    const int32_t* h_rp = nullptr;    // block-row pointers (host)
    const int32_t* sptr = nullptr;
    const int32_t* scol = nullptr;
    const float* K32 = nullptr;
    const double* K64 = nullptr;
    const float* dinv32 = nullptr;
};

struct BatchStats {
    int64_t outer_iterations;
    int64_t lockstep_iterations;    // inner iterations of the slowest system, summed over refinements
    int64_t system_iterations;      // inner iterations summed over all systems
    int64_t unconverged;
    double max_rel_residual;
    double device_ms;
};

struct Batch;
// Order of a variant's rows in a batch: order[i] is the row that stands i-th.
std::vector<int32_t> batch_row_order(int64_t n, const int32_t* rp, const int32_t* bc, const double* xyz);
int batch_create(Batch** out, const std::vector<OperatorView>& ops);
void batch_destroy(Batch* b);
const char* batch_error(const Batch* b);
// rhs / x: per variant nrhs vectors of its DOFs, one after another (FP64, host);
// zero right-hand sides are skipped.
// verbose != 0 prints one progress line per refinement to stderr.
int batch_solve(Batch* b, const double* const* rhs, double* const* x, int nrhs, double tol, double inner_tol, int64_t max_it,
                int check_every, int verbose, BatchStats* stats);

}  // namespace asend
