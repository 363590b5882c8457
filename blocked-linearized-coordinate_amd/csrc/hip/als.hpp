// als.hpp -- launchers of als.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "blco_host.h"

namespace blco {

struct GramSet {
    const double* g[BLCO_MAX_MODES];
};

constexpr int GRAM_MAX_PARTS = 2048;  // partial Gram blocks (workgroups) at most
int gram_parts(uint64_t rows, int* nparts, uint64_t* rows_per_wg);
// G = U^T U (f64, R x R) from dtype U; with M, ip[col] = sum_i U_ic M_ic.
// part needs gram_parts(rows) * (R*R + R) doubles.
int launch_gram(const void* U, int dtype, uint64_t rows, int R, const void* M,
                double* part, double* G, double* ip, hipStream_t st);
// Machine epsilon of the precision the Grams of factor_dtype factors are
// accumulated in (f64 for f64 factors, f32 for f32 and bf16 ones).
double gram_eps(int factor_dtype);
// fac: R x R (V^{-1}, or V^+ with status 1); work: 2 R^2 + R doubles.  eps
// scales the Cholesky pivot floor and the pseudo-inverse tolerance.
int launch_factorize(const GramSet& gs, int nmodes, int mode, int R, double eps, double* fac,
                     double* work, int* status, hipStream_t st);
// In-place pseudo-inverse of a general n x n matrix (n <= 64); info
// (device, may be null): 0 converged, else the sweep count.
int launch_pinv_general(double* A, int n, int* info, hipStream_t st);
// U = M F^T row by row.
int launch_solve_rows(const void* M, void* U, int dtype, uint64_t rows, int R, const double* fac, hipStream_t st);

// One mode's ALS update of one tensor, after its MTTKRP is in M (an array of
// these in device memory, one for each tensor of a launch): U = M diag(c) F^T,
// lambda and dinv[mode] from U's column statistics, G[mode] = the Gram of the
// normalised factor, with `last` the fit, and F = fac and c = colscale for
// mode `next`.  M is left cleared.
struct AlsTask {
    void *M, *U;
    uint64_t rows;
    double *fac, *colscale, *work;     // R x R; R; 2 R^2 + R
    double *stats, *part;              // parts x R; parts x (R^2 + R)
    double *lambda, *dinv;             // R; nmodes x R
    double* G[BLCO_MAX_MODES];
    double* fit;                       // fit, inner product, ||model||^2
    const double* normX2;
    int* status;
    int nmodes, mode, next, last;
    uint32_t parts, first;             // workgroups, and the first one's index in the launch
};
struct AlsLaunch {
    const AlsTask* d_tasks = nullptr;
    int ntasks = 0;
    uint32_t blocks = 0, most_parts = 0;  // of all tasks; of the largest
};
uint32_t solve_gram_parts(uint64_t rows);  // parts of a task
int launch_als_update(const AlsLaunch& l, int dtype, int R, int which, double eps, hipStream_t st);
// fac and colscale of the tasks' `next` modes from the Grams and dinv alone.
int launch_als_begin(const AlsLaunch& l, int R, double eps, hipStream_t st);
// lambda, 1/lambda from column statistics (folded in place).
int launch_lambda(double* stats, int nparts, int R, int which, double* lambda, double* inv, hipStream_t st);
// out[0] = fit, out[1] = inner product, out[2] = ||M||^2.
int launch_fit(const GramSet& gs, int nmodes, int R, const double* lambda, const double* ip,
               double normX2, double* out, hipStream_t st);
int launch_sumsq(const void* x, int dtype, uint64_t n, double* part, int nparts, double* out,
                 hipStream_t st);
int launch_hadamard(double* x, const double* y, uint64_t n, hipStream_t st);

int launch_colstats(const void* U, int dtype, uint64_t rows, int R, int which, double* stats,
                    int nparts, hipStream_t st);
int launch_scale(void* U, int dtype, uint64_t rows, int R, const double* inv, hipStream_t st);
// out (f64) = U diag(inv).
int launch_export(const void* U, int dtype, uint64_t rows, int R, const double* inv, double* out, hipStream_t st);
int launch_vecsum(double* x, uint64_t n, hipStream_t st);

}  // namespace blco
