// als.hip -- the ALS step of CP-ALS on gfx950 (src/cpd_gpu.cu:21-242 of the
// reference does it with cuBLAS / cuSOLVER; the semantics kept here are the
// CPU reference's, include/cpd.hpp:44-272).
//
//   gram       G = U^T U on MFMA: v_mfma_f64_16x16x4f64 for f64 factors,
//              v_mfma_f32_16x16x4f32 for f32/bf16 factors.  One wave walks
//              4-row steps of U; lane l holds U[r0 + l/16][16 t + l%16], which
//              is both the A operand (A[i][k] = U[r0+k][16 ti + i]) and the B
//              operand of tile (ti, tj).  The accumulator layouts differ: the
//              f32 form leaves D[4*(l/16) + v][l%16] in register v of lane l,
//              the f64 form D[l/16 + 4*v][l%16] (checked on the hardware).  Per-workgroup partial Grams are
//              summed in a fixed order (deterministic).  Optionally the same
//              pass forms the fit inner products sum_i U_ir M_ir.
//   factorize  one workgroup: V = prod_{m != n} G_m (Hadamard), for R <= 32
//              V = L D L^T and L^{-1} in one wave's registers, else lower
//              Cholesky in LAPACK dpotf2 order in LDS; when a pivot falls to
//              R * eps * max V_ii or below, cyclic Jacobi eigendecomposition
//              of V and the pseudo-inverse V^+ = Q diag(1/w) Q^T with
//              tolerance R * ulp(max |w|) (src/cpd_gpu.cu:487-489), where eps
//              and ulp are those of the precision the Grams were accumulated
//              in (f64, or f32 for the f32 / bf16 factor forms).
//              On success the explicit inverse V^{-1} = L^{-T} L^{-1} is
//              formed (so both outcomes leave one R x R matrix F).
//   solve rows U = M F on f64 MFMA, a wave per 16 rows.
//   als update the CP-ALS update of a mode in one pass on MFMA (k_als_update):
//              the solve's result registers feed the Gram tiles directly, with
//              the column statistics for the norm beside; k_als_finish turns
//              the partial sums into lambda, Gram and fit and factors the next
//              mode's V.
//   lambda     lambda_r = sqrt(sum) (L2) or max(1, max) (max norm,
//              src/kruskal_model.cpp:183-223), and 1/lambda (0 for a zero
//              column).
//   fit        one workgroup: fit = 1 - r / ||X|| with
//              r^2 = ||X||^2 + |sum_ij l_i l_j prod_n G_n(i,j)| - 2 sum_r l_r ip_r
//              (include/cpd.hpp:190-272).
#include "als.hpp"
#include "devcommon.hpp"

namespace blco {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T> __device__ __forceinline__ float as_f32(T x) { return (float)x; }
template <> __device__ __forceinline__ float as_f32<bf16>(bf16 x) { return bf16_to_f32(x.bits); }
template <typename T> __device__ __forceinline__ double as_f64(T x) { return (double)x; }
template <> __device__ __forceinline__ double as_f64<bf16>(bf16 x) { return (double)bf16_to_f32(x.bits); }
template <typename T> __device__ __forceinline__ bool is_zero(T x) { return x == (T)0; }

// ------------------------------------------------------------------ gram

// Partial Gram (and optional scaling / inner products) of rows
// [g * rows_per_wg, ...) for workgroup g.  T tiles of 16 columns.
template <typename UT, int T>
__global__ __launch_bounds__(WG) void k_gram(const UT* __restrict__ U, uint64_t rows, int R,
                                             uint64_t rows_per_wg,
                                             const void* __restrict__ M,
                                             double* __restrict__ part)
{
    constexpr bool F64 = std::is_same<UT, double>::value;
    using AT = typename std::conditional<F64, double, float>::type;
    using VT = typename std::conditional<F64, d4, f4>::type;
    constexpr int NT = T * (T + 1) / 2;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i16 = lane & 15, k4 = lane >> 4;
    const uint64_t rb = (uint64_t)blockIdx.x * rows_per_wg;
    const uint64_t re = min(rb + rows_per_wg, rows);
    VT acc[NT];
    #pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = VT{0, 0, 0, 0};
    double ip[T];
    #pragma unroll
    for (int t = 0; t < T; ++t) ip[t] = 0.0;
    // UN row steps' loads are issued together (their MFMAs in row order): 1.8M
    // rows at rank 32, FP32, 100 us with one step's loads at a time
    constexpr int UN = 4;
    for (uint64_t r0 = rb + (uint64_t)w * 4; r0 < re; r0 += UN * WAVES_PER_WG * 4) {
        AT a[UN][T];
        #pragma unroll
        for (int u = 0; u < UN; ++u) {
            const uint64_t row = r0 + (uint64_t)u * WAVES_PER_WG * 4 + k4;
            #pragma unroll
            for (int t = 0; t < T; ++t) {
                const int col = t * 16 + i16;
                a[u][t] = (row < re && col < R) ? (AT)as_f64(U[row * (uint64_t)R + col]) : (AT)0;
            }
        }
        if (M) {
            #pragma unroll
            for (int u = 0; u < UN; ++u) {
                const uint64_t row = r0 + (uint64_t)u * WAVES_PER_WG * 4 + k4;
                #pragma unroll
                for (int t = 0; t < T; ++t) {
                    const int col = t * 16 + i16;
                    if (row < re && col < R) {
                        const double mv = F64 ? reinterpret_cast<const double*>(M)[row * (uint64_t)R + col]
                                              : (double)reinterpret_cast<const float*>(M)[row * (uint64_t)R + col];
                        ip[t] += (double)a[u][t] * mv;
                    }
                }
            }
        }
        #pragma unroll
        for (int u = 0; u < UN; ++u) {
            int q = 0;
            #pragma unroll
            for (int ti = 0; ti < T; ++ti)
                #pragma unroll
                for (int tj = ti; tj < T; ++tj) {
                    if constexpr (F64)
                        acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][ti], a[u][tj], acc[q], 0, 0, 0);
                    else
                        acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][ti], a[u][tj], acc[q], 0, 0, 0);
                    ++q;
                }
        }
    }
    // combine the 4 waves in LDS, then write this workgroup's partial
    __shared__ double s_g[WAVES_PER_WG][T * 16][T * 16 + 1];
    __shared__ double s_ip[WAVES_PER_WG][T * 16];
    int q = 0;
    #pragma unroll
    for (int ti = 0; ti < T; ++ti)
        #pragma unroll
        for (int tj = ti; tj < T; ++tj) {
            #pragma unroll
            for (int v = 0; v < 4; ++v) {
                // D register v of lane l holds row 4*(l/16) + v (f32 form) or
                // row l/16 + 4*v (f64 form), column l % 16 of the tile
                int i = ti * 16 + (F64 ? k4 + 4 * v : 4 * k4 + v), j = tj * 16 + i16;
                double x = (double)acc[q][v];
                s_g[w][i][j] = x;
                s_g[w][j][i] = x;
            }
            ++q;
        }
    #pragma unroll
    for (int t = 0; t < T; ++t) {
        // lanes with equal i16 hold partial sums of the same column
        double x = ip[t];
        x += __shfl_xor(x, 16);
        x += __shfl_xor(x, 32);
        if (k4 == 0) s_ip[w][t * 16 + i16] = x;
    }
    __syncthreads();
    double* out = part + (uint64_t)blockIdx.x * (uint64_t)(R * R + R);
    for (int e = threadIdx.x; e < R * R; e += WG) {
        int i = e / R, j = e % R;
        out[e] = ((s_g[0][i][j] + s_g[1][i][j]) + s_g[2][i][j]) + s_g[3][i][j];
    }
    for (int e = threadIdx.x; e < R; e += WG)
        out[R * R + e] = ((s_ip[0][e] + s_ip[1][e]) + s_ip[2][e]) + s_ip[3][e];
}

// Deterministic reduction of nparts rows of W doubles (part[p][e], row
// major) over p, in two passes that both fill the GPU.  Pass 1: workgroup
// (x, y) takes entries [64 x, 64 x + 64) of the rows p = y (mod gridDim.y);
// wave w of it folds the rows y + P2 (w + 4 j), j = 0, 1, ..., with two
// accumulators, the four waves' results are combined in wave order and
// written over row y (only this workgroup reads row y's entries, and it
// has read them all by then).  Pass 2 folds rows 0..P2-1 in order.  which:
// 0 sum (seed 0), 1 max seeded with 1.
constexpr int RED_SPLIT = 16;

__device__ __forceinline__ double fold_op(int which, double a, double b) { return which == 0 ? a + b : fmax(a, b); }

__global__ __launch_bounds__(WG) void k_fold_parts(double* __restrict__ part, int nparts, int W, int which)
{
    __shared__ double s_sum[WAVES_PER_WG][WAVE];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int e = blockIdx.x * WAVE + lane, y = blockIdx.y, P2 = gridDim.y;
    const double seed = which == 0 ? 0.0 : 1.0;
    double a0 = seed, a1 = seed;
    if (e < W) {
        int p = y + P2 * w;
        for (; p + WAVES_PER_WG * P2 < nparts; p += 2 * WAVES_PER_WG * P2) {
            a0 = fold_op(which, a0, part[(uint64_t)p * W + e]);
            a1 = fold_op(which, a1, part[(uint64_t)(p + WAVES_PER_WG * P2) * W + e]);
        }
        if (p < nparts) a0 = fold_op(which, a0, part[(uint64_t)p * W + e]);
    }
    s_sum[w][lane] = fold_op(which, a0, a1);
    __syncthreads();
    if (w == 0 && e < W)
        part[(uint64_t)y * W + e] =
            fold_op(which, fold_op(which, fold_op(which, s_sum[0][lane], s_sum[1][lane]), s_sum[2][lane]), s_sum[3][lane]);
}

static int fold_parts(double* part, int nparts, int W, int which, int* rows_left, hipStream_t st)
{
    const int p2 = nparts < RED_SPLIT ? (nparts < 1 ? 1 : nparts) : RED_SPLIT;
    hipLaunchKernelGGL(k_fold_parts, dim3((W + WAVE - 1) / WAVE, p2), dim3(WG), 0, st, part, nparts, W, which);
    HIP_TRY(hipGetLastError());
    *rows_left = p2;
    return BLCO_OK;
}

// Pass 2 of the Gram reduction: G (R*R) and ip (R) from the P2 folded rows
// of (R*R + R).
__global__ __launch_bounds__(WAVE) void k_gram_finish(const double* __restrict__ part, int p2, int R,
                                                      double* __restrict__ G, double* __restrict__ ip)
{
    const int e = blockIdx.x * WAVE + threadIdx.x, W = R * R + R;
    if (e >= W) return;
    double s = part[e];
    for (int y = 1; y < p2; ++y) s += part[(uint64_t)y * W + e];
    if (e < R * R) G[e] = s;
    else if (ip) ip[e - R * R] = s;
}

// ------------------------------------------------------------- factorize

__device__ __forceinline__ double lane_value(double x, int lane)
{
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

// V = s_a = L D L^T by one wave and in registers (R <= RP): X = L^{-1} (unit
// lower, row-major) into s_x and D^{-1} X into s_a.  Lane i holds row i of
// the matrix while it is factored, then column i of X.  Right-looking, so
// every entry's terms are subtracted in the order of dpotf2's column dot
// products; D_j is the pivot that dpotf2 would take the root of.  One
// reciprocal a column, no root and no barriers: by a workgroup in LDS the
// Cholesky form took 42 us at R = 32 and 16 us at R = 16.  False when a pivot
// falls to `floor_piv` or below (the same for every lane).
template <int RP>
__device__ __forceinline__ bool ldl_inverse_wave(double* s_a, double* s_x, int R, double floor_piv)
{
    const int lane = threadIdx.x & 63;
    double a[RP], rd[RP];
    #pragma unroll
    for (int k = 0; k < RP; ++k) a[k] = (lane < R && k < R) ? s_a[lane * R + k] : (lane == k ? 1.0 : 0.0);
    #pragma unroll
    for (int j = 0; j < RP; ++j) {
        rd[j] = 1.0;
        if (j < R) {
            const double ajj = lane_value(a[j], j);
            if (!(ajj > floor_piv)) return false;
            rd[j] = 1.0 / ajj;
            const double l = lane > j ? a[j] * rd[j] : 0.0;
            #pragma unroll
            for (int k = j + 1; k < RP; ++k) a[k] -= l * lane_value(a[j], k);
            a[j] = l;
        }
    }
    double x[RP];
    #pragma unroll
    for (int k = 0; k < RP; ++k) x[k] = lane == k ? 1.0 : 0.0;
    #pragma unroll
    for (int k = 0; k < RP; ++k) {
        if (k < R) {
            #pragma unroll
            for (int i = k + 1; i < RP; ++i) x[i] -= lane_value(a[k], i) * x[k];
            if (lane < R) {
                s_x[k * R + lane] = x[k];
                s_a[k * R + lane] = x[k] * rd[k];
            }
        }
    }
    return true;
}

// X = L^{-1} of the Cholesky factor of s_a (overwritten) into s_x, by the
// whole workgroup in LDS, for ranks whose rows do not fit a lane's registers.
__device__ __forceinline__ bool chol_inverse_lds(double* s_a, double* s_x, int R, double floor_piv)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int e = tid; e < R * R; e += nt) s_x[e] = (e / R == e % R) ? 1.0 : 0.0;
    __syncthreads();
    for (int j = 0; j < R; ++j) {
        const double ajj = s_a[j * R + j];
        if (!(ajj > floor_piv)) return false;  // every thread reads the same value: a uniform exit
        const double piv = sqrt(ajj);
        __syncthreads();  // all have read a_jj
        for (int i = j + 1 + tid; i < R; i += nt) s_a[i * R + j] /= piv;
        if (tid == 0) s_a[j * R + j] = piv;
        __syncthreads();
        const int n = R - 1 - j;
        for (int t = tid; t < n * n; t += nt) {
            const int i = j + 1 + t / n, k = j + 1 + t % n;
            if (k <= i) s_a[i * R + k] -= s_a[i * R + j] * s_a[k * R + j];
        }
        __syncthreads();
    }
    for (int k = 0; k < R; ++k) {
        const double lkk = s_a[k * R + k];
        for (int c = tid; c <= k; c += nt) s_x[k * R + c] /= lkk;
        __syncthreads();
        const int n = R - 1 - k, w = k + 1;
        for (int t = tid; t < n * w; t += nt) {
            const int i = k + 1 + t / w, c = t % w;
            s_x[i * R + c] -= s_a[i * R + k] * s_x[k * R + c];
        }
        __syncthreads();
    }
    return true;
}

// V^+ of the symmetric V in work (R x R, destroyed) into fac by cyclic Jacobi.
__device__ void jacobi_pinv(int R, double eps, double* __restrict__ work, double* __restrict__ fac)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    // ---- fallback: symmetric pseudo-inverse by cyclic Jacobi
    double* A = work;          // R x R, V (destroyed)
    double* Q = work + R * R;  // R x R eigenvectors (columns)
    double* wv = work + 2 * R * R;
    for (int e = tid; e < R * R; e += nt) Q[e] = (e / R == e % R) ? 1.0 : 0.0;
    // s_done (sweep converged) and s_skip (one pair's rotation skipped) are
    // separate flags, and every thread has read s_done before thread 0 can
    // write either again, so no wave acts on a flag of another step.
    __shared__ int s_done, s_skip;
    __shared__ double s_c, s_s;
    __syncthreads();
    for (int sweep = 0; sweep < 60; ++sweep) {
        if (tid == 0) {
            double off = 0.0, diag = 0.0;
            for (int i = 0; i < R; ++i)
                for (int j = 0; j < R; ++j) {
                    double x = A[i * R + j];
                    if (i != j) off += x * x;
                    else diag += x * x;
                }
            s_done = (off <= 1e-30 * diag || off == 0.0);
        }
        __syncthreads();
        const bool converged = s_done != 0;
        __syncthreads();
        if (converged) break;
        for (int p = 0; p < R - 1; ++p)
            for (int qq = p + 1; qq < R; ++qq) {
                if (tid == 0) {
                    double apq = A[p * R + qq];
                    if (apq == 0.0) {
                        s_c = 1.0; s_s = 0.0; s_skip = 1;
                    } else {
                        double app = A[p * R + p], aqq = A[qq * R + qq];
                        double tau = (aqq - app) / (2.0 * apq);
                        double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
                        double c = 1.0 / sqrt(1.0 + t * t);
                        s_c = c; s_s = t * c; s_skip = 0;
                    }
                }
                __syncthreads();
                if (s_skip) { __syncthreads(); continue; }
                const double c = s_c, s = s_s;
                for (int k = tid; k < R; k += nt) {
                    double akp = A[k * R + p], akq = A[k * R + qq];
                    A[k * R + p] = c * akp - s * akq;
                    A[k * R + qq] = s * akp + c * akq;
                }
                __threadfence_block();
                __syncthreads();
                for (int k = tid; k < R; k += nt) {
                    double apk = A[p * R + k], aqk = A[qq * R + k];
                    A[p * R + k] = c * apk - s * aqk;
                    A[qq * R + k] = s * apk + c * aqk;
                    double qkp = Q[k * R + p], qkq = Q[k * R + qq];
                    Q[k * R + p] = c * qkp - s * qkq;
                    Q[k * R + qq] = s * qkp + c * qkq;
                }
                __threadfence_block();
                __syncthreads();
            }
    }
    if (tid == 0) {
        double emax = 0.0;
        for (int i = 0; i < R; ++i) emax = fmax(emax, fabs(A[i * R + i]));
        // R * ulp(emax) in the Grams' precision; with eps = 2^-52 this is
        // R * (nextafter(emax, +inf) - emax) of src/cpd_gpu.cu:487-489
        double tol = emax > 0.0 ? R * ldexp(eps, ilogb(emax)) : 0.0;
        for (int i = 0; i < R; ++i) {
            double x = A[i * R + i];
            wv[i] = (fabs(x) > tol) ? 1.0 / x : 0.0;
        }
    }
    __threadfence_block();
    __syncthreads();
    for (int e = tid; e < R * R; e += nt) {
        int i = e / R, j = e % R;
        double s = 0.0;
        for (int k = 0; k < R; ++k) s += Q[i * R + k] * wv[k] * Q[j * R + k];
        fac[e] = s;
    }
}

// The whole workgroup: V = s_a (R x R, also kept in work), then fac = V^{-1}
// = X^T D^{-1} X with status 0, or V^+ with status 1.
// A pivot at or below R * eps * max_i V_ii means V is singular to the working
// precision its Grams carry: its Cholesky factor would carry pivots of
// rounding noise (and the solve factors of that size), so the pseudo-inverse
// takes over -- the threshold the Jacobi fallback uses for eigenvalues.  eps
// is that of the Grams' accumulation (2^-52 for f64 factors, 2^-23 for f32 /
// bf16 ones: an f32 V that is singular to f32 precision clears an f64 floor
// or not depending on the summation order).  dpotrf's own test (a pivot <= 0)
// is the special case of an exactly singular V.
__device__ __forceinline__ void factorize_block(double* s_a, double* s_x, int R, double eps, double* fac, double* work,
                                                int* status)
{
    __shared__ int s_ok;
    const int tid = threadIdx.x, nt = blockDim.x;
    __syncthreads();
    double dmax = 0.0;
    for (int i = 0; i < R; ++i) dmax = fmax(dmax, s_a[i * R + i]);
    const double floor_piv = R * eps * dmax;
    bool ok;
    if (R <= 32) {
        if (tid < WAVE) {
            const bool r = R <= 16 ? ldl_inverse_wave<16>(s_a, s_x, R, floor_piv)
                                   : ldl_inverse_wave<32>(s_a, s_x, R, floor_piv);
            if (tid == 0) s_ok = r;
        }
        __syncthreads();
        ok = s_ok != 0;
    } else {
        ok = chol_inverse_lds(s_a, s_x, R, floor_piv);
    }
    if (ok) {
        const double* s_y = R <= 32 ? s_a : s_x;  // D^{-1} X, or X where L holds the roots
        for (int e = tid; e < R * R; e += nt) {
            const int a = e / R, b = e % R;
            double t = 0.0;
            for (int k = a > b ? a : b; k < R; ++k) t += s_x[k * R + a] * s_y[k * R + b];
            fac[e] = t;
        }
        if (tid == 0) *status = 0;
        return;
    }
    __syncthreads();
    jacobi_pinv(R, eps, work, fac);
    if (tid == 0) *status = 1;
}

// status: 0 V^{-1} in fac (by Cholesky), 1 pseudo-inverse in fac.
__global__ __launch_bounds__(WG) void k_factorize(GramSet gs, int nmodes, int mode, int R, double eps,
                                                  double* __restrict__ fac, double* __restrict__ work,
                                                  int* __restrict__ status)
{
    extern __shared__ double s_a[];  // R x R: V, then R x R: L^{-1}
    for (int e = threadIdx.x; e < R * R; e += WG) {
        double v = 1.0;
        for (int m = 0; m < nmodes; ++m)
            if (m != mode) v *= gs.g[m][e];
        s_a[e] = v;
        work[e] = v;  // keep V for the fallback
    }
    factorize_block(s_a, s_a + R * R, R, eps, fac, work, status);
}

// --------------------------------------------------------- pseudo-inverse

// In-place Moore-Penrose pseudo-inverse of a general n x n row-major matrix
// (pseudoinverse_gpu, src/cpd_gpu.cu:452-532, which takes an SVD by gesvdj):
// one-sided Jacobi SVD (Hestenes) in LDS.  W = A is rotated column pair by
// column pair, the rotations accumulated in V, until every pair of columns
// of W is orthogonal to working precision; then sigma_j = ||w_j||,
// A = U diag(sigma) V^T with u_j = w_j / sigma_j, and
// A^+ = V diag(1 / sigma^2) W^T over the sigma_j above the reference's
// cutoff n * (nextafter(sigma_max, +inf) - sigma_max).  A sweep visits all
// pairs as n' - 1 rounds of n' / 2 disjoint pairs (round-robin tournament,
// n' = n rounded up to even), one thread per pair.  *info = 0 when a sweep
// made no rotation, else the sweep count (gesvdj's info > 0: not converged).
__global__ __launch_bounds__(WG) void k_pinv_general(double* __restrict__ A, int n,
                                                     int* __restrict__ info)
{
    extern __shared__ double s_w[];  // W (n x n), then V (n x n), then sigma (n)
    double* s_v = s_w + n * n;
    double* s_sig = s_v + n * n;
    __shared__ int s_rot;
    const int tid = threadIdx.x;
    for (int e = tid; e < n * n; e += WG) {
        s_w[e] = A[e];
        s_v[e] = (e / n == e % n) ? 1.0 : 0.0;
    }
    const int np = (n + 1) & ~1, m = np - 1;
    int sweeps = 0;
    bool converged = false;
    for (; sweeps < 60 && !converged; ++sweeps) {
        if (tid == 0) s_rot = 0;
        __syncthreads();
        for (int r = 0; r < m; ++r) {
            if (tid < np / 2) {
                int p = tid == 0 ? r : (r + tid) % m;
                int q = tid == 0 ? m : (r - tid + m) % m;
                if (p > q) { const int t = p; p = q; q = t; }
                if (q < n) {
                    double a = 0.0, b = 0.0, g = 0.0;
                    for (int i = 0; i < n; ++i) {
                        const double x = s_w[i * n + p], y = s_w[i * n + q];
                        a += x * x;
                        b += y * y;
                        g += x * y;
                    }
                    if (g != 0.0 && fabs(g) > 1e-15 * sqrt(a * b)) {
                        const double z = (b - a) / (2.0 * g);
                        const double t = (z >= 0 ? 1.0 : -1.0) / (fabs(z) + sqrt(1.0 + z * z));
                        const double c = 1.0 / sqrt(1.0 + t * t), s = c * t;
                        for (int i = 0; i < n; ++i) {
                            const double x = s_w[i * n + p], y = s_w[i * n + q];
                            s_w[i * n + p] = c * x - s * y;
                            s_w[i * n + q] = s * x + c * y;
                            const double vx = s_v[i * n + p], vy = s_v[i * n + q];
                            s_v[i * n + p] = c * vx - s * vy;
                            s_v[i * n + q] = s * vx + c * vy;
                        }
                        s_rot = 1;
                    }
                }
            }
            __syncthreads();
        }
        converged = s_rot == 0;  // every thread reads it after the round's barrier
        __syncthreads();
    }
    for (int j = tid; j < n; j += WG) {
        double a = 0.0;
        for (int i = 0; i < n; ++i) a += s_w[i * n + j] * s_w[i * n + j];
        s_sig[j] = sqrt(a);
    }
    __syncthreads();
    double smax = 0.0;
    for (int j = 0; j < n; ++j) smax = fmax(smax, s_sig[j]);
    const double tol = n * (nextafter(smax, INFINITY) - smax);
    for (int e = tid; e < n * n; e += WG) {
        const int i = e / n, k = e % n;
        double t = 0.0;
        for (int j = 0; j < n; ++j) {
            const double sg = s_sig[j];
            if (sg > tol) t += s_v[i * n + j] * s_w[k * n + j] / (sg * sg);
        }
        A[e] = t;
    }
    if (tid == 0 && info) *info = converged ? 0 : sweeps;
}

// ------------------------------------------------------------ solve rows

// U = M F with F = V^{-1} (or V^+), a wave per 16-row tile on f64 MFMA: the
// solve half of k_als_update.  Bound by HBM (M read and U written once): 1.8M
// rows at rank 32, FP32, 327 us with a group of 32 lanes per row and the row
// of M in LDS.
template <typename MT, typename UT, int T>
__global__ __launch_bounds__(WG) void k_solve_rows(const MT* __restrict__ M, UT* __restrict__ U, uint64_t rows, int R,
                                                   const double* __restrict__ fac)
{
    constexpr int KS = 4 * T;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i16 = lane & 15, k4 = lane >> 4;
    double b[T][KS];
    #pragma unroll
    for (int ct = 0; ct < T; ++ct)
        #pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 4 * ks + k4, j = 16 * ct + i16;
            b[ct][ks] = (k < R && j < R) ? fac[j * R + k] : 0.0;
        }
    const uint64_t tiles = (rows + 15) / 16, stride = (uint64_t)gridDim.x * WAVES_PER_WG;
    MT m[KS];  // the next tile's operands, loaded behind this one's MFMAs
    auto load = [&](uint64_t tile) {
        const uint64_t ra = tile * 16 + i16;
        #pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 4 * ks + k4;
            m[ks] = (ra < rows && k < R) ? M[ra * (uint64_t)R + k] : (MT)0;
        }
    };
    uint64_t tile = (uint64_t)blockIdx.x * WAVES_PER_WG + w;
    load(tile);
    for (; tile < tiles; tile += stride) {
        const uint64_t r0 = tile * 16;
        d4 d[T];
        #pragma unroll
        for (int ct = 0; ct < T; ++ct) d[ct] = d4{0, 0, 0, 0};
        double x[KS];
        #pragma unroll
        for (int ks = 0; ks < KS; ++ks) x[ks] = (double)m[ks];
        load(tile + stride);
        #pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            #pragma unroll
            for (int ct = 0; ct < T; ++ct) d[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[ks], b[ct][ks], d[ct], 0, 0, 0);
        #pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint64_t row = r0 + k4 + 4 * v;
            #pragma unroll
            for (int ct = 0; ct < T; ++ct) {
                const int col = 16 * ct + i16;
                if (row < rows && col < R) U[row * (uint64_t)R + col] = from_f64<UT>(d[ct][v]);
            }
        }
    }
}

// ------------------------------------------------------- fused solve + Gram

// One pass of a mode's ALS update on MFMA: U = M diag(c) F^T row tile by row
// tile (16 rows), then, from the same registers, the tile's contribution to
// G = U^T U, the column statistics of U and (with ip) sum_i U_ic M_ic.
//   solve  v_mfma_f64_16x16x4f64 with A[i][k] = M[r0 + i][4 ks + k] (lane l
//          loads M[r0 + l%16][4 ks + l/16]) and B[k][j] = c_k F[16 ct + j][k]
//          (held in registers for the whole launch); the result D[i][j] sits
//          in register v of lane l as U[r0 + l/16 + 4 v][16 ct + l%16].
//   Gram   that register v is, for the row step r0 + 4 v, exactly the A and B
//          operand of the Gram's MFMA (lane l: U[r0 + 4v + l/16][16 t + l%16]),
//          so the stored (rounded) values feed the Gram tiles directly: f64
//          MFMA for f64 factors, f32 for f32 / bf16 ones, as in k_gram.
// Rows past the end load as 0 and give 0 rows of U (not stored).  Each
// workgroup's waves take tiles with a fixed stride; its partial Gram (and
// ip) and column statistics are combined in LDS in wave order and written to
// part[block] (R*R + R) and stats[block] (R): deterministic.  A tile of M is
// cleared once it is used: the next mode's MTTKRP adds into zeros without a
// fill of its own.  One launch updates a mode of every task (the tensors of
// a batch, or one): workgroup b belongs to the last task with first <= b.
template <typename MT, typename UT, int T>
__global__ __launch_bounds__(WG) void k_als_update(const AlsTask* __restrict__ tasks, int ntasks, int R, int which)
{
    int lo = 0;
    for (int hi = ntasks; hi - lo > 1;) {
        const int mid = (lo + hi) >> 1;
        if (tasks[mid].first <= blockIdx.x) lo = mid;
        else hi = mid;
    }
    const AlsTask& tk = tasks[lo];
    MT* __restrict__ M = static_cast<MT*>(tk.M);
    UT* __restrict__ U = static_cast<UT*>(tk.U);
    const uint64_t rows = tk.rows;
    const double* __restrict__ fac = tk.fac;
    const double* __restrict__ colscale = tk.colscale;
    const bool want_ip = tk.last != 0;
    const uint32_t block = blockIdx.x - tk.first, blocks = tk.parts;
    constexpr bool F64 = std::is_same<UT, double>::value;
    using AT = typename std::conditional<F64, double, float>::type;
    using VT = typename std::conditional<F64, d4, f4>::type;
    constexpr int NT = T * (T + 1) / 2;
    constexpr int KS = 4 * T;  // k steps of 4 over the (padded) rank 16 T
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i16 = lane & 15, k4 = lane >> 4;
    // B operands: c_k F[16 ct + j][k] for k = 4 ks + k4, j = i16
    double b[T][KS];
    #pragma unroll
    for (int ct = 0; ct < T; ++ct)
        #pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 4 * ks + k4, j = 16 * ct + i16;
            b[ct][ks] = (k < R && j < R) ? fac[j * R + k] * colscale[k] : 0.0;
        }
    VT g[NT];
    #pragma unroll
    for (int q = 0; q < NT; ++q) g[q] = VT{0, 0, 0, 0};
    double st[T], ipa[T];
    #pragma unroll
    for (int ct = 0; ct < T; ++ct) {
        st[ct] = which == 0 ? 0.0 : 1.0;
        ipa[ct] = 0.0;
    }
    const uint64_t tiles = (rows + 15) / 16;
    const uint64_t stride = (uint64_t)blocks * WAVES_PER_WG;
    for (uint64_t tile = (uint64_t)block * WAVES_PER_WG + w; tile < tiles; tile += stride) {
        const uint64_t r0 = tile * 16;
        d4 d[T];
        #pragma unroll
        for (int ct = 0; ct < T; ++ct) d[ct] = d4{0, 0, 0, 0};
        const uint64_t ra = r0 + i16;
        #pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 4 * ks + k4;
            const double m = (ra < rows && k < R) ? (double)M[ra * (uint64_t)R + k] : 0.0;
            #pragma unroll
            for (int ct = 0; ct < T; ++ct) d[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(m, b[ct][ks], d[ct], 0, 0, 0);
        }
        #pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint64_t row = r0 + k4 + 4 * v;
            AT x[T];
            #pragma unroll
            for (int ct = 0; ct < T; ++ct) {
                const int col = 16 * ct + i16;
                const double t = d[ct][v];
                const bool ok = row < rows && col < R;
                const UT u = from_f64<UT>(t);
                if (ok) {
                    U[row * (uint64_t)R + col] = u;
                    st[ct] = which == 0 ? st[ct] + t * t : fmax(st[ct], t);
                    if (want_ip) {
                        const double mv = (double)M[row * (uint64_t)R + col];
                        ipa[ct] += (double)(AT)as_f64(u) * mv;
                    }
                }
                x[ct] = ok ? (AT)as_f64(u) : (AT)0;
            }
            int q = 0;
            #pragma unroll
            for (int ti = 0; ti < T; ++ti)
                #pragma unroll
                for (int tj = ti; tj < T; ++tj) {
                    if constexpr (F64)
                        g[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[ti], x[tj], g[q], 0, 0, 0);
                    else
                        g[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[ti], x[tj], g[q], 0, 0, 0);
                    ++q;
                }
        }
        const uint64_t e1 = min((r0 + 16) * (uint64_t)R, rows * (uint64_t)R);
        for (uint64_t e = r0 * (uint64_t)R + lane; e < e1; e += WAVE) M[e] = (MT)0;
    }
    // combine the waves: Gram tiles as in k_gram; statistics and ip over the
    // four row groups (k4) of a wave, then over the waves, in order
    __shared__ double s_g[WAVES_PER_WG][T * 16][T * 16 + 1];
    __shared__ double s_v[WAVES_PER_WG][2][T * 16];
    int q = 0;
    #pragma unroll
    for (int ti = 0; ti < T; ++ti)
        #pragma unroll
        for (int tj = ti; tj < T; ++tj) {
            #pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int i = ti * 16 + (F64 ? k4 + 4 * v : 4 * k4 + v), j = tj * 16 + i16;
                const double x = (double)g[q][v];
                s_g[w][i][j] = x;
                s_g[w][j][i] = x;
            }
            ++q;
        }
    #pragma unroll
    for (int ct = 0; ct < T; ++ct) {
        double a = st[ct], c = ipa[ct];
        #pragma unroll
        for (int o = 16; o < 64; o <<= 1) {
            const double y = __shfl_xor(a, o);
            a = which == 0 ? a + y : fmax(a, y);
            c += __shfl_xor(c, o);
        }
        if (k4 == 0) {
            s_v[w][0][ct * 16 + i16] = a;
            s_v[w][1][ct * 16 + i16] = c;
        }
    }
    __syncthreads();
    double* out = tk.part + (uint64_t)block * (uint64_t)(R * R + R);
    for (int e = threadIdx.x; e < R * R; e += WG) {
        const int i = e / R, j = e % R;
        out[e] = ((s_g[0][i][j] + s_g[1][i][j]) + s_g[2][i][j]) + s_g[3][i][j];
    }
    for (int e = threadIdx.x; e < R; e += WG) {
        out[R * R + e] = ((s_v[0][1][e] + s_v[1][1][e]) + s_v[2][1][e]) + s_v[3][1][e];
        double a = s_v[0][0][e];
        for (int x = 1; x < WAVES_PER_WG; ++x) a = which == 0 ? a + s_v[x][0][e] : fmax(a, s_v[x][0][e]);
        tk.stats[(uint64_t)block * R + e] = a;
    }
}

// First fold of the partial rows of tasks with more than FINISH_PARTS of them
// (blockIdx.z: task; as k_fold_parts, sums of part and of stats by `which`).
constexpr int FINISH_PARTS = 32;

__global__ __launch_bounds__(WG) void k_als_fold(const AlsTask* __restrict__ tasks, int R, int which)
{
    const AlsTask& tk = tasks[blockIdx.z];
    const int nparts = (int)tk.parts;
    if (nparts <= FINISH_PARTS) return;
    __shared__ double s_sum[WAVES_PER_WG][WAVE];
    const int W = R * R + R, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int gx = (W + WAVE - 1) / WAVE;  // further columns of blocks fold the statistics
    const bool st = (int)blockIdx.x >= gx;
    const int e = ((int)blockIdx.x - (st ? gx : 0)) * WAVE + lane, width = st ? R : W, y = blockIdx.y, P2 = gridDim.y;
    double* part = st ? tk.stats : tk.part;
    const int op = st ? which : 0;
    const double seed = op == 0 ? 0.0 : 1.0;
    double a0 = seed, a1 = seed;
    if (e < width) {
        int p = y + P2 * w;
        for (; p + WAVES_PER_WG * P2 < nparts; p += 2 * WAVES_PER_WG * P2) {
            a0 = fold_op(op, a0, part[(uint64_t)p * width + e]);
            a1 = fold_op(op, a1, part[(uint64_t)(p + WAVES_PER_WG * P2) * width + e]);
        }
        if (p < nparts) a0 = fold_op(op, a0, part[(uint64_t)p * width + e]);
    }
    s_sum[w][lane] = fold_op(op, a0, a1);
    __syncthreads();
    if (w == 0 && e < width)
        part[(uint64_t)y * width + e] =
            fold_op(op, fold_op(op, fold_op(op, s_sum[0][lane], s_sum[1][lane]), s_sum[2][lane]), s_sum[3][lane]);
}

// The end of a mode's update, one workgroup per task: lambda, 1/lambda and
// the scaled Gram (and ip, and the sweep's fit after its last mode) from the
// partial rows, then the factorisation for the mode that comes next.  One
// launch in place of six and of a factorisation on a side stream: a sweep of
// a small tensor is bound by its launches, and the factorisation takes a few
// microseconds (ldl_inverse_wave).  With nothing to finish (update = 0) only
// the factorisation, for the first mode of the first sweep.
constexpr int FINISH_WG = 512;

__global__ __launch_bounds__(FINISH_WG) void k_als_finish(const AlsTask* __restrict__ tasks, int R, int which,
                                                          double eps, int update)
{
    const AlsTask& tk = tasks[blockIdx.x];
    extern __shared__ double s_dyn[];  // R x R: G, then L^{-1}; R x R: V; lambda, 1/lambda, ip (R each)
    double *s_g = s_dyn, *s_v = s_dyn + R * R, *s_lam = s_v + R * R, *s_inv = s_lam + R, *s_ip = s_inv + R;
    __shared__ double s_red[FINISH_WG / WAVE];
    const int tid = threadIdx.x, W = R * R + R;
    const int np = (int)tk.parts <= FINISH_PARTS ? (int)tk.parts : RED_SPLIT;
    const int mode = tk.mode, nmodes = tk.nmodes, next = tk.next, last = tk.last;
    // the Grams that this update leaves as they are: their product into s_v
    for (int e = tid; e < R * R; e += FINISH_WG) {
        double v = 1.0;
        for (int m = 0; m < nmodes; ++m)
            if (m != next && !(update && m == mode)) v *= tk.G[m][e];
        s_v[e] = v;
    }
    if (update) {
        // sums over the partial rows, eight loads in flight: G and ip, then
        // the statistics
        for (int e = tid; e < W + R; e += FINISH_WG) {
            const bool stat = e >= W;
            const int op = stat ? which : 0;
            const uint64_t width = stat ? R : W;
            const double* q = stat ? tk.stats + (e - W) : tk.part + e;
            double t = q[0];
            int p = 1;
            for (; p + 8 <= np; p += 8) {
                double x[8];
                #pragma unroll
                for (int u = 0; u < 8; ++u) x[u] = q[(p + u) * width];
                #pragma unroll
                for (int u = 0; u < 8; ++u) t = fold_op(op, t, x[u]);
            }
            {
                double x[7];
                #pragma unroll
                for (int u = 0; u < 7; ++u) x[u] = p + u < np ? q[(p + u) * width] : (op == 0 ? 0.0 : t);
                #pragma unroll
                for (int u = 0; u < 7; ++u) t = fold_op(op, t, x[u]);
            }
            if (stat) {
                const int c = e - W;
                if (which == 0) t = sqrt(t);
                const double iv = (t == 0.0) ? 0.0 : 1.0 / t;
                s_lam[c] = t;
                s_inv[c] = iv;
                tk.lambda[c] = t;
                tk.dinv[mode * R + c] = iv;
            } else if (e < R * R) {
                s_g[e] = t;
            } else {
                s_ip[e - R * R] = t * tk.colscale[e - R * R];
            }
        }
        __syncthreads();
        for (int e = tid; e < R * R; e += FINISH_WG) {
            const double g = s_g[e] * (s_inv[e / R] * s_inv[e % R]);
            tk.G[mode][e] = g;
            s_g[e] = g;
        }
        if (last) {
            // fit = 1 - r / ||X||, as k_fit
            double sum = 0.0;
            for (int e = tid; e < R * R; e += FINISH_WG) {  // this thread's own entries of s_g and s_v
                const int i = e / R, j = e % R;
                if (j > i) continue;
                const double t = (s_lam[i] * s_lam[j]) * ((s_v[e] * tk.G[next][e]) * s_g[e]);
                sum += j < i ? 2.0 * t : t;
            }
            #pragma unroll
            for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
            if ((tid & 63) == 0) s_red[tid >> 6] = sum;
            __syncthreads();
            if (tid == 0) {
                double model = 0.0, inner = 0.0;
                for (int i = 0; i < FINISH_WG / WAVE; ++i) model += s_red[i];
                for (int r = 0; r < R; ++r) inner += (s_ip[r] * s_inv[r]) * s_lam[r];
                model = fabs(model);
                const double x2 = *tk.normX2;
                double res = x2 + model - 2.0 * inner;
                if (res > 0.0) res = sqrt(res);
                tk.fit[0] = 1.0 - res / sqrt(x2);
                tk.fit[1] = inner;
                tk.fit[2] = model;
            }
        }
    }
    // the next mode's V, and the column scale its MTTKRP result carries: the
    // product of the other factors' pending inverse scales
    for (int k = tid; k < R; k += FINISH_WG) {
        double c = 1.0;
        for (int m = 0; m < nmodes; ++m)
            if (m != next) c *= update && m == mode ? s_inv[k] : tk.dinv[m * R + k];
        tk.colscale[k] = c;
    }
    for (int e = tid; e < R * R; e += FINISH_WG) {
        const double v = update ? s_v[e] * s_g[e] : s_v[e];
        s_v[e] = v;
        tk.work[e] = v;  // for the fallback
    }
    factorize_block(s_v, s_g, R, eps, tk.fac, tk.work, tk.status);
}

// lambda and 1/lambda (0 for a zero column) from the P2 folded rows of the
// column statistics.
__global__ __launch_bounds__(WAVE) void k_lambda_finish(const double* __restrict__ stats, int p2, int R,
                                                        int which, double* __restrict__ lambda,
                                                        double* __restrict__ inv)
{
    const int c = blockIdx.x * WAVE + threadIdx.x;
    if (c >= R) return;
    double y = stats[c];
    for (int q = 1; q < p2; ++q) y = fold_op(which, y, stats[(uint64_t)q * R + c]);
    if (which == 0) y = sqrt(y);
    const double iv = (y == 0.0) ? 0.0 : 1.0 / y;
    lambda[c] = y;
    inv[c] = iv;
}

// ------------------------------------------------------------------- fit

__global__ __launch_bounds__(WG) void k_fit(GramSet gs, int nmodes, int R,
                                            const double* __restrict__ lambda,
                                            const double* __restrict__ ip, double normX2,
                                            double* __restrict__ out)
{
    __shared__ double s_off[WG], s_diag[WG];
    double off = 0.0, diag = 0.0;
    for (int e = threadIdx.x; e < R * R; e += WG) {
        int i = e / R, j = e % R;
        if (j > i) continue;
        double t = lambda[i] * lambda[j];
        for (int m = 0; m < nmodes; ++m) t *= gs.g[m][e];
        if (j < i) off += 2.0 * t;
        else diag += t;
    }
    s_off[threadIdx.x] = off;
    s_diag[threadIdx.x] = diag;
    __syncthreads();
    if (threadIdx.x == 0) {
        double so = 0.0, sd = 0.0, inner = 0.0;
        for (int t = 0; t < WG; ++t) { so += s_off[t]; sd += s_diag[t]; }
        for (int r = 0; r < R; ++r) inner += ip[r] * lambda[r];
        double normU = fabs(so + sd);
        double res = normX2 + normU - 2.0 * inner;
        if (res > 0.0) res = sqrt(res);
        out[0] = 1.0 - res / sqrt(normX2);
        out[1] = inner;
        out[2] = normU;
    }
}

// Sum of squares of n values (f64 or f32 storage) per workgroup.
template <typename T>
__global__ __launch_bounds__(WG) void k_sumsq(const T* __restrict__ x, uint64_t n,
                                              double* __restrict__ part)
{
    __shared__ double s[WAVES_PER_WG];
    double acc = 0.0;
    for (uint64_t e = (uint64_t)blockIdx.x * WG + threadIdx.x; e < n; e += (uint64_t)gridDim.x * WG) {
        double v = (double)x[e];
        acc += v * v;
    }
    #pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = ((s[0] + s[1]) + s[2]) + s[3];
}

// out[0] = sum of n parts, in a fixed order (61 us for 1024 by one thread).
__global__ __launch_bounds__(WG) void k_sum_parts(const double* __restrict__ part, int n, double* __restrict__ out)
{
    __shared__ double s[WAVES_PER_WG];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += WG) acc += part[i];
    #pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) out[0] = ((s[0] + s[1]) + s[2]) + s[3];
}

// out = U diag(inv) in f64.
template <typename UT>
__global__ __launch_bounds__(WG) void k_export(const UT* __restrict__ U, uint64_t cells, int R,
                                               const double* __restrict__ inv, double* __restrict__ out)
{
    for (uint64_t e = (uint64_t)blockIdx.x * WG + threadIdx.x; e < cells; e += (uint64_t)gridDim.x * WG)
        out[e] = as_f64(U[e]) * inv[e % R];
}

__global__ __launch_bounds__(WG) void k_hadamard(double* __restrict__ x, const double* __restrict__ y,
                                                 uint64_t n)
{
    for (uint64_t e = (uint64_t)blockIdx.x * WG + threadIdx.x; e < n; e += (uint64_t)gridDim.x * WG)
        x[e] *= y[e];
}

// Per-workgroup column statistics of an existing factor (which 0: sum of
// squares, 1: max seeded with 1), for the stand-alone column norm.  A
// workgroup reads WG / R rows at a time, thread t the t-th element of them,
// eight such loads in flight; bound by HBM (1.8M rows at rank 32, FP32: 700
// us with one column's lane walking the rows alone).
template <typename UT>
__global__ __launch_bounds__(WG) void k_colstats(const UT* __restrict__ U, uint64_t rows, int R,
                                                 uint64_t rows_per_wg, int which,
                                                 double* __restrict__ stats)
{
    __shared__ double s_st[WG];
    const uint64_t rb = (uint64_t)blockIdx.x * rows_per_wg;
    const uint64_t re = min(rb + rows_per_wg, rows);
    const double seed = which == 0 ? 0.0 : 1.0;
    for (int c0 = 0; c0 < R; c0 += WG) {  // one pass for R <= WG
        const int width = min(R - c0, WG), groups = WG / width;
        const int t = threadIdx.x, c = t % width, g = t / width;
        double x = seed;
        if (g < groups) {
            uint64_t i = rb + g;
            const uint64_t step = groups;
            for (; i + 7 * step < re; i += 8 * step) {
                double v[8];
                #pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = as_f64(U[(i + u * step) * (uint64_t)R + c0 + c]);
                #pragma unroll
                for (int u = 0; u < 8; ++u) x = (which == 0) ? x + v[u] * v[u] : fmax(x, v[u]);
            }
            for (; i < re; i += step) {
                const double v = as_f64(U[i * (uint64_t)R + c0 + c]);
                x = (which == 0) ? x + v * v : fmax(x, v);
            }
        }
        s_st[t] = x;
        __syncthreads();
        if (t < width) {
            for (int q = 1; q < groups; ++q) x = which == 0 ? x + s_st[q * width + t] : fmax(x, s_st[q * width + t]);
            stats[(uint64_t)blockIdx.x * R + c0 + t] = x;
        }
        __syncthreads();
    }
}

template <typename UT>
__global__ __launch_bounds__(WG) void k_scale(UT* __restrict__ U, uint64_t cells, int R,
                                              const double* __restrict__ inv)
{
    for (uint64_t e = (uint64_t)blockIdx.x * WG + threadIdx.x; e < cells; e += (uint64_t)gridDim.x * WG)
        U[e] = from_f64<UT>(as_f64(U[e]) * inv[e % R]);
}

__global__ void k_vecsum(double* __restrict__ x, uint64_t n)
{
    __shared__ double s[WG];
    double acc = 0.0;
    for (uint64_t e = threadIdx.x; e < n; e += WG) acc += x[e];
    s[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < WG; ++i) t += s[i];
        x[0] = t;
    }
}

// ------------------------------------------------------------ launchers

template <typename UT>
static int gram_t(const UT* U, uint64_t rows, int R, const void* M, double* part,
                  int nparts, uint64_t rpw, hipStream_t st)
{
    int T = (R + 15) / 16;
    switch (T) {
        case 1: hipLaunchKernelGGL((k_gram<UT, 1>), dim3(nparts), dim3(WG), 0, st, U, rows, R, rpw, M, part); break;
        case 2: hipLaunchKernelGGL((k_gram<UT, 2>), dim3(nparts), dim3(WG), 0, st, U, rows, R, rpw, M, part); break;
        case 3: hipLaunchKernelGGL((k_gram<UT, 3>), dim3(nparts), dim3(WG), 0, st, U, rows, R, rpw, M, part); break;
        case 4: hipLaunchKernelGGL((k_gram<UT, 4>), dim3(nparts), dim3(WG), 0, st, U, rows, R, rpw, M, part); break;
        default: return fail(BLCO_EUNSUPPORTED, "rank %d > 64 not supported by the Gram kernel", R);
    }
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int gram_parts(uint64_t rows, int* nparts, uint64_t* rows_per_wg)
{
    uint64_t steps = (rows + 3) / 4;
    uint64_t want = (steps + 63) / 64;  // ~64 row-steps per workgroup (16 per wave)
    if (want < 1) want = 1;
    if (want > GRAM_MAX_PARTS) want = GRAM_MAX_PARTS;  // callers size partial buffers for this
    uint64_t rpw = (rows + want - 1) / want;
    rpw = (rpw + 3) / 4 * 4;
    if (rpw == 0) rpw = 4;
    *rows_per_wg = rpw;
    *nparts = (int)((rows + rpw - 1) / rpw);
    if (*nparts < 1) *nparts = 1;
    return BLCO_OK;
}

int launch_gram(const void* U, int dtype, uint64_t rows, int R, const void* M,
                double* part, double* G, double* ip, hipStream_t st)
{
    if (R < 1 || R > 64) return fail(BLCO_EUNSUPPORTED, "rank %d outside [1, 64] for the Gram kernel", R);
    int nparts;
    uint64_t rpw;
    gram_parts(rows, &nparts, &rpw);
    int rc;
    if (dtype == BLCO_F64) rc = gram_t<double>((const double*)U, rows, R, M, part, nparts, rpw, st);
    else if (dtype == BLCO_F32) rc = gram_t<float>((const float*)U, rows, R, M, part, nparts, rpw, st);
    else rc = gram_t<bf16>((const bf16*)U, rows, R, M, part, nparts, rpw, st);
    if (rc) return rc;
    const int W = R * R + R;
    int p2 = 0;
    rc = fold_parts(part, nparts, W, 0, &p2, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_gram_finish, dim3((W + WAVE - 1) / WAVE), dim3(WAVE), 0, st, part, p2, R, G, ip);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

double gram_eps(int factor_dtype)
{
    return factor_dtype == BLCO_F64 ? 2.220446049250313e-16 : 1.1920928955078125e-07;
}

int launch_factorize(const GramSet& gs, int nmodes, int mode, int R, double eps, double* fac,
                     double* work, int* status, hipStream_t st)
{
    if (R < 1 || R > 64) return fail(BLCO_EUNSUPPORTED, "rank %d outside [1, 64] in the factorisation", R);
    size_t lds = sizeof(double) * 2 * (size_t)R * R;
    if (lds > 64 * 1024) HIP_TRY(hipFuncSetAttribute((const void*)k_factorize,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_factorize, dim3(1), dim3(WG), lds, st, gs, nmodes, mode, R, eps, fac, work, status);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

template <typename MT, typename UT>
static int solve_rows_t(const MT* M, UT* U, uint64_t rows, int R, const double* fac, hipStream_t st)
{
    if (rows == 0) return BLCO_OK;
    const uint32_t grid = solve_gram_parts(rows);
    switch ((R + 15) / 16) {
        case 1: hipLaunchKernelGGL((k_solve_rows<MT, UT, 1>), dim3(grid), dim3(WG), 0, st, M, U, rows, R, fac); break;
        case 2: hipLaunchKernelGGL((k_solve_rows<MT, UT, 2>), dim3(grid), dim3(WG), 0, st, M, U, rows, R, fac); break;
        case 3: hipLaunchKernelGGL((k_solve_rows<MT, UT, 3>), dim3(grid), dim3(WG), 0, st, M, U, rows, R, fac); break;
        case 4: hipLaunchKernelGGL((k_solve_rows<MT, UT, 4>), dim3(grid), dim3(WG), 0, st, M, U, rows, R, fac); break;
        default: return fail(BLCO_EUNSUPPORTED, "rank %d > 64 in the row solve", R);
    }
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_solve_rows(const void* M, void* U, int dtype, uint64_t rows, int R, const double* fac, hipStream_t st)
{
    if (dtype == BLCO_F64) return solve_rows_t<double, double>((const double*)M, (double*)U, rows, R, fac, st);
    if (dtype == BLCO_F32) return solve_rows_t<float, float>((const float*)M, (float*)U, rows, R, fac, st);
    return solve_rows_t<float, bf16>((const float*)M, (bf16*)U, rows, R, fac, st);
}

uint32_t solve_gram_parts(uint64_t rows)
{
    const uint64_t p = (rows + 255) / 256;  // at least 4 row tiles per wave
    return (uint32_t)(p < 1 ? 1 : p > GRAM_MAX_PARTS ? GRAM_MAX_PARTS : p);
}

template <typename MT, typename UT>
static void als_update_t(const AlsTask* tasks, int ntasks, int R, int which, uint32_t grid, hipStream_t st)
{
    switch ((R + 15) / 16) {
        case 1: hipLaunchKernelGGL((k_als_update<MT, UT, 1>), dim3(grid), dim3(WG), 0, st, tasks, ntasks, R, which); break;
        case 2: hipLaunchKernelGGL((k_als_update<MT, UT, 2>), dim3(grid), dim3(WG), 0, st, tasks, ntasks, R, which); break;
        case 3: hipLaunchKernelGGL((k_als_update<MT, UT, 3>), dim3(grid), dim3(WG), 0, st, tasks, ntasks, R, which); break;
        default: hipLaunchKernelGGL((k_als_update<MT, UT, 4>), dim3(grid), dim3(WG), 0, st, tasks, ntasks, R, which); break;
    }
}

static int als_finish(const AlsTask* d_tasks, int ntasks, int R, int which, double eps, int update, hipStream_t st)
{
    const size_t lds = sizeof(double) * (2 * (size_t)R * R + 3 * R);
    if (lds > 64 * 1024) HIP_TRY(hipFuncSetAttribute((const void*)k_als_finish,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_als_finish, dim3(ntasks), dim3(FINISH_WG), lds, st, d_tasks, R, which, eps, update);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_als_update(const AlsLaunch& l, int dtype, int R, int which, double eps, hipStream_t st)
{
    if (R < 1 || R > 64) return fail(BLCO_EUNSUPPORTED, "rank %d outside [1, 64] in the ALS update", R);
    if (!l.ntasks) return BLCO_OK;
    if (dtype == BLCO_F64) als_update_t<double, double>(l.d_tasks, l.ntasks, R, which, l.blocks, st);
    else if (dtype == BLCO_F32) als_update_t<float, float>(l.d_tasks, l.ntasks, R, which, l.blocks, st);
    else als_update_t<float, bf16>(l.d_tasks, l.ntasks, R, which, l.blocks, st);
    HIP_TRY(hipGetLastError());
    if (l.most_parts > (uint32_t)FINISH_PARTS) {
        const int gx = (R * R + R + WAVE - 1) / WAVE + (R + WAVE - 1) / WAVE;
        hipLaunchKernelGGL(k_als_fold, dim3(gx, RED_SPLIT, l.ntasks), dim3(WG), 0, st, l.d_tasks, R, which);
        HIP_TRY(hipGetLastError());
    }
    return als_finish(l.d_tasks, l.ntasks, R, which, eps, 1, st);
}

int launch_als_begin(const AlsLaunch& l, int R, double eps, hipStream_t st)
{
    return l.ntasks ? als_finish(l.d_tasks, l.ntasks, R, 0, eps, 0, st) : BLCO_OK;
}

int launch_pinv_general(double* A, int n, int* info, hipStream_t st)
{
    if (n < 1 || n > 64) return fail(BLCO_EUNSUPPORTED, "pseudo-inverse of order %d outside [1, 64]", n);
    const size_t lds = sizeof(double) * ((size_t)2 * n * n + n);
    hipLaunchKernelGGL(k_pinv_general, dim3(1), dim3(WG), lds, st, A, n, info);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_lambda(double* stats, int nparts, int R, int which, double* lambda, double* inv, hipStream_t st)
{
    int p2 = 0;
    int rc = fold_parts(stats, nparts, R, which, &p2, st);
    if (rc) return rc;
    hipLaunchKernelGGL(k_lambda_finish, dim3((R + WAVE - 1) / WAVE), dim3(WAVE), 0, st, stats, p2, R, which, lambda,
                       inv);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_fit(const GramSet& gs, int nmodes, int R, const double* lambda, const double* ip,
               double normX2, double* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_fit, dim3(1), dim3(WG), 0, st, gs, nmodes, R, lambda, ip, normX2, out);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_sumsq(const void* x, int dtype, uint64_t n, double* part, int nparts, double* out,
                 hipStream_t st)
{
    if (dtype == BLCO_F64)
        hipLaunchKernelGGL(k_sumsq<double>, dim3(nparts), dim3(WG), 0, st, (const double*)x, n, part);
    else
        hipLaunchKernelGGL(k_sumsq<float>, dim3(nparts), dim3(WG), 0, st, (const float*)x, n, part);
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(WG), 0, st, part, nparts, out);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_hadamard(double* x, const double* y, uint64_t n, hipStream_t st)
{
    uint32_t grid = (uint32_t)std::min<uint64_t>((n + WG - 1) / WG, 4096);
    if (grid == 0) return BLCO_OK;
    hipLaunchKernelGGL(k_hadamard, dim3(grid), dim3(WG), 0, st, x, y, n);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

}  // namespace blco

namespace blco {

template <typename UT>
static void colstats_t(const UT* U, uint64_t rows, int R, uint64_t rpw, int nparts, int which,
                       double* stats, hipStream_t st)
{
    hipLaunchKernelGGL(k_colstats<UT>, dim3(nparts), dim3(WG), 0, st, U, rows, R, rpw, which, stats);
}

int launch_colstats(const void* U, int dtype, uint64_t rows, int R, int which, double* stats,
                    int nparts, hipStream_t st)
{
    uint64_t rpw = (rows + nparts - 1) / nparts;
    if (rpw == 0) rpw = 1;
    if (dtype == BLCO_F64) colstats_t((const double*)U, rows, R, rpw, nparts, which, stats, st);
    else if (dtype == BLCO_F32) colstats_t((const float*)U, rows, R, rpw, nparts, which, stats, st);
    else colstats_t((const bf16*)U, rows, R, rpw, nparts, which, stats, st);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_scale(void* U, int dtype, uint64_t rows, int R, const double* inv, hipStream_t st)
{
    uint64_t cells = rows * (uint64_t)R;
    uint32_t grid = (uint32_t)std::min<uint64_t>((cells + WG - 1) / WG, 8192);
    if (grid == 0) return BLCO_OK;
    if (dtype == BLCO_F64) hipLaunchKernelGGL(k_scale<double>, dim3(grid), dim3(WG), 0, st, (double*)U, cells, R, inv);
    else if (dtype == BLCO_F32) hipLaunchKernelGGL(k_scale<float>, dim3(grid), dim3(WG), 0, st, (float*)U, cells, R, inv);
    else hipLaunchKernelGGL(k_scale<bf16>, dim3(grid), dim3(WG), 0, st, (bf16*)U, cells, R, inv);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_export(const void* U, int dtype, uint64_t rows, int R, const double* inv, double* out, hipStream_t st)
{
    const uint64_t cells = rows * (uint64_t)R;
    const uint32_t grid = (uint32_t)std::min<uint64_t>((cells + WG - 1) / WG, 8192);
    if (grid == 0) return BLCO_OK;
    if (dtype == BLCO_F64) hipLaunchKernelGGL(k_export<double>, dim3(grid), dim3(WG), 0, st, (const double*)U, cells, R, inv, out);
    else if (dtype == BLCO_F32) hipLaunchKernelGGL(k_export<float>, dim3(grid), dim3(WG), 0, st, (const float*)U, cells, R, inv, out);
    else hipLaunchKernelGGL(k_export<bf16>, dim3(grid), dim3(WG), 0, st, (const bf16*)U, cells, R, inv, out);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

int launch_vecsum(double* x, uint64_t n, hipStream_t st)
{
    hipLaunchKernelGGL(k_vecsum, dim3(1), dim3(WG), 0, st, x, n);
    HIP_TRY(hipGetLastError());
    return BLCO_OK;
}

}  // namespace blco
