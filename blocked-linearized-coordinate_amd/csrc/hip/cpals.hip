// cpals.hip -- device-resident CP-ALS driver (cpals_blco_dev,
// src/cpd_gpu.cu:21-242) with the CPU reference's iteration semantics
// (cpd_alto, include/cpd.hpp:44-187):
//
//   for it: for each mode n (0..N-1, or longest first):
//       M   = MTTKRP(n)                         (kernel per mode)
//       F   = (prod_{m != n} G_m)^{-1}, or the pseudo-inverse
//       U_n = M F, column statistics
//       lambda = L2 norms at it 0, max(1, max) after; U_n /= lambda
//       G_n = U_n^T U_n (MFMA); for the last mode also sum_i U_n M
//   fit = 1 - ||X - [[lambda; U]]|| / ||X||, stop when it > 0 and
//   |fit - fit_old| < tolerance.
//
// The division by lambda is not written back: each factor is stored as the
// solve leaves it, U_n diag(lambda_n), with 1 / lambda_n kept aside (dinv).
// Its Gram is formed from the stored factor and scaled by 1 / lambda on
// both sides; the MTTKRP of a later mode then carries the product c of the
// other factors' lambdas in its columns, and that mode's solve multiplies
// M by c^{-1} (folded into F); blco_cpals_get applies 1 / lambda.  A mode's
// update is one MFMA kernel that reads M once, writes U_n once, clears M for
// the next MTTKRP and forms the Gram from the solve's registers, and a
// one-workgroup kernel that turns the partial sums into lambda and G_n and
// factors the next mode's V (launch_als_update).
//
// Everything stays on one stream with no host round trip inside a sweep;
// the host reads back the fit (24 bytes) once per iteration.  With use_graph
// one sweep (after iteration 0, whose norm differs) is captured into a
// hipGraph and replayed; the output buffer is cleared by kernels, never by a
// memset node.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "als.hpp"
#include "cpals.hpp"
#include "device.hpp"
#include "devcommon.hpp"
#include "mttkrp.hpp"

using namespace blco;

namespace blco {

static void to_dtype(const double* src, void* dst, uint64_t n, int dt)
{
    if (dt == BLCO_F64) std::memcpy(dst, src, n * 8);
    else if (dt == BLCO_F32) {
        float* f = (float*)dst;
        for (uint64_t i = 0; i < n; ++i) f[i] = (float)src[i];
    } else {
        uint16_t* b = (uint16_t*)dst;
        for (uint64_t i = 0; i < n; ++i) {
            float x = (float)src[i];
            uint32_t u;
            std::memcpy(&u, &x, 4);
            if ((u & 0x7f800000u) == 0x7f800000u) b[i] = (uint16_t)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
            else b[i] = (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
        }
    }
}

// Enqueues one ALS sweep: per mode the MTTKRP and the update, the last one
// with the fit.
static int enqueue_sweep(blco_cpals_state* s, int which_norm, bool timed)
{
    blco_dev* d = s->d;
    for (int k = 0; k < s->N; ++k) {
        const int n = s->order[k];
        if (timed) HIP_TRY(hipEventRecord(s->ev0[n], s->st));
        int rc = mttkrp(d, n, s->R, s->ft, s->U, s->Mbuf, s->o.kernel, s->o.nprtn, s->o.thread_cf, s->st,
                        &s->kern[n]);
        if (rc) return rc;
        if (timed) HIP_TRY(hipEventRecord(s->ev1[n], s->st));
        rc = launch_als_update(s->upd[n], s->ft, s->R, which_norm, s->eps, s->st);
        if (rc) return rc;
    }
    return BLCO_OK;
}

int enqueue_export(blco_cpals_state* s, double* out)
{
    for (int m = 0; m < s->N; ++m) {
        const int rc = launch_export(s->U[m], s->ft, s->d->dims[m], s->R, s->dinv + (size_t)m * s->R, out, s->st);
        if (rc) return rc;
        out += s->d->dims[m] * (uint64_t)s->R;
    }
    return BLCO_OK;
}

int cpals_state_create(blco_dev* d, const blco_cpals_opts* o, const double* const* U, bool own_io,
                       blco_cpals_state** out)
{
    if (!d || !o || !U || !out) return fail(BLCO_EINVAL, "null argument");
    *out = nullptr;
    const int N = d->nmodes, R = o->rank;
    if (R < 1 || R > 64) return fail(BLCO_EUNSUPPORTED, "rank %d outside [1, 64]", R);
    if (N < 2) return fail(BLCO_EUNSUPPORTED, "CP-ALS needs at least 2 modes");
    if (o->precision != BLCO_F64 && o->precision != BLCO_F32 && o->precision != BLCO_BF16)
        return fail(BLCO_EINVAL, "precision %d", o->precision);
    const int need_v = o->precision == BLCO_F64 ? BLCO_F64 : BLCO_F32;
    if (d->vdtype != need_v)
        return fail(BLCO_EINVAL, "precision %d needs %s values on the device", o->precision,
                    need_v == BLCO_F64 ? "f64" : "f32");
    if (o->max_iters < 0) return fail(BLCO_EINVAL, "max_iters %d", o->max_iters);
    for (int m = 0; m < N; ++m)
        if (!U[m]) return fail(BLCO_EINVAL, "initial factor %d is null", m);
    blco_cpals_state* s = new (std::nothrow) blco_cpals_state();
    if (!s) return fail(BLCO_ENOMEM, "out of host memory");
    auto bad = [&](int rc) { blco_cpals_free(s); return rc; };
    s->d = d;
    s->o = *o;
    if (s->o.kernel == 0) s->o.kernel = BLCO_K_AUTO;
    s->N = N;
    s->R = R;
    s->ft = o->precision;
    s->mt = o->precision == BLCO_F64 ? BLCO_F64 : BLCO_F32;
    s->st = d->stream;
    // mode order: natural (CPU reference) or longest first (GPU reference)
    for (int m = 0; m < N; ++m) s->order[m] = m;
    if (o->mode_order == 1)
        for (int i = 1; i < N; ++i)
            for (int j = i; j > 0 && d->dims[s->order[j]] > d->dims[s->order[j - 1]]; --j)
                std::swap(s->order[j], s->order[j - 1]);
    s->eps = o->solve_floor ? gram_eps(s->ft) : gram_eps(BLCO_F64);  // pivot floor: f64's unless asked for
    const int fsz = dtype_size(s->ft), msz = s->mt == BLCO_F64 ? 8 : 4, nnorm = 1024;
    uint64_t maxI = 0, parts = 1;
    for (int m = 0; m < N; ++m) {
        int gp;
        uint64_t rpw;
        gram_parts(d->dims[m], &gp, &rpw);
        maxI = std::max(maxI, d->dims[m]);
        parts = std::max<uint64_t>(parts, std::max<uint64_t>((uint64_t)gp, solve_gram_parts(d->dims[m])));
    }
    // one allocation: offsets first, then the addresses
    uint64_t total = 0;
    auto take = [&](uint64_t bytes) {
        const uint64_t at = total;
        total += (bytes + 255) / 256 * 256;
        return at;
    };
    uint64_t oU[BLCO_MAX_MODES], oG[BLCO_MAX_MODES];
    for (int m = 0; m < N; ++m) oU[m] = take(d->dims[m] * (uint64_t)R * fsz);
    const uint64_t factor_bytes = total;
    for (int m = 0; m < N; ++m) oG[m] = take(sizeof(double) * R * R);
    s->m_bytes = maxI * R * msz;
    const uint64_t oM = take(s->m_bytes), olam = take(8 * R), ofac = take(8 * R * R),
                   owork = take(8 * (2 * R * R + R)), ostat = take(sizeof(int)), opart = take(8 * parts * (R * R + R)),
                   ostats = take(8 * parts * R), ofit = take(8 * 4), onorm = take(8 * (nnorm + 1)),
                   odinv = take(8 * (uint64_t)N * R), ocs = take(8 * R), otask = take(sizeof(AlsTask) * N);
    if (hipMalloc(&s->arena, total) != hipSuccess) return bad(fail(BLCO_ENOMEM, "solver allocation failed (%llu bytes)",
                                                                   (unsigned long long)total));
    char* base = static_cast<char*>(s->arena);
    auto dbl = [&](uint64_t at) { return reinterpret_cast<double*>(base + at); };
    for (int m = 0; m < N; ++m) {
        s->U[m] = base + oU[m];
        s->G[m] = dbl(oG[m]);
    }
    s->Mbuf = base + oM;
    s->lambda = dbl(olam);
    s->fac = dbl(ofac);
    s->work = dbl(owork);
    s->status = reinterpret_cast<int*>(base + ostat);
    s->part = dbl(opart);
    s->stats = dbl(ostats);
    s->fitbuf = dbl(ofit);
    s->norm_part = dbl(onorm);
    s->dinv = dbl(odinv);
    s->colscale = dbl(ocs);
    // the factors in one copy (converted, and laid out as on the device)
    {
        std::vector<char> stage;
        try {
            stage.resize(factor_bytes);
        } catch (const std::bad_alloc&) {
            return bad(fail(BLCO_ENOMEM, "host staging of the factors"));
        }
        for (int m = 0; m < N; ++m) to_dtype(U[m], stage.data() + oU[m], d->dims[m] * (uint64_t)R, s->ft);
        if (hipMemcpy(s->arena, stage.data(), factor_bytes, hipMemcpyHostToDevice) != hipSuccess)
            return bad(fail(BLCO_EHIP, "factor upload failed"));
    }
    if (own_io) {
        for (int m = 0; m < N; ++m)
            if (hipEventCreate(&s->ev0[m]) != hipSuccess || hipEventCreate(&s->ev1[m]) != hipSuccess)
                return bad(fail(BLCO_EHIP, "event creation failed"));
        if (hipHostMalloc((void**)&s->h_fit, sizeof(double) * 4, hipHostMallocDefault) != hipSuccess)
            return bad(fail(BLCO_ENOMEM, "pinned allocation failed"));
        if (hipEventCreate(&s->it0) != hipSuccess || hipEventCreate(&s->it1) != hipSuccess)
            return bad(fail(BLCO_EHIP, "event creation failed"));
    }
    // each mode's task; its successor in the sweep is the mode factored next
    for (int k = 0; k < N; ++k) {
        const int n = s->order[k];
        AlsTask& t = s->tasks[n];
        t.M = s->Mbuf;
        t.U = s->U[n];
        t.rows = d->dims[n];
        t.fac = s->fac;
        t.colscale = s->colscale;
        t.work = s->work;
        t.stats = s->stats;
        t.part = s->part;
        t.lambda = s->lambda;
        t.dinv = s->dinv;
        for (int m = 0; m < N; ++m) t.G[m] = s->G[m];
        t.fit = s->fitbuf;
        t.normX2 = s->norm_part + nnorm;
        t.status = s->status;
        t.nmodes = N;
        t.mode = n;
        t.next = s->order[(k + 1) % N];
        t.last = k == N - 1;
        t.parts = solve_gram_parts(t.rows);
        t.first = 0;
        s->upd[n] = AlsLaunch{reinterpret_cast<AlsTask*>(base + otask) + n, 1, t.parts, t.parts};
    }
    if (hipMemcpy(base + otask, s->tasks, sizeof(AlsTask) * N, hipMemcpyHostToDevice) != hipSuccess)
        return bad(fail(BLCO_EHIP, "task upload failed"));
    // lambda = 1 (KruskalModelRandomInit), ||X||^2, initial Grams
    int rc = launch_fill(s->lambda, R, BLCO_F64, 1.0, s->st);
    if (!rc) rc = launch_fill(s->dinv, (uint64_t)N * R, BLCO_F64, 1.0, s->st);
    if (rc) return bad(rc);
    if (d->nnz && !d->stream_data) {
        rc = launch_sumsq(d->d_vals, d->vdtype, d->nnz, s->norm_part, nnorm, s->norm_part + nnorm, s->st);
        if (rc) return bad(rc);
    } else {
        // streamed tensors: the values are in pinned host memory
        double acc = 0.0;
        if (d->vdtype == BLCO_F64) {
            const double* v = (const double*)d->h_vals;
            for (uint64_t i = 0; i < d->nnz; ++i) acc += v[i] * v[i];
        } else {
            const float* v = (const float*)d->h_vals;
            for (uint64_t i = 0; i < d->nnz; ++i) acc += (double)v[i] * (double)v[i];
        }
        if (hipMemcpy(s->norm_part + nnorm, &acc, sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
            return bad(fail(BLCO_EHIP, "norm upload failed"));
    }
    for (int m = 0; m < N && !rc; ++m)
        rc = launch_gram(s->U[m], s->ft, d->dims[m], R, nullptr, s->part, s->G[m], nullptr, s->st);
    if (rc) return bad(rc);
    *out = s;
    return BLCO_OK;
}

static double now_ms()
{
    return std::chrono::duration<double, std::milli>(
               std::chrono::steady_clock::now().time_since_epoch()).count();
}

}  // namespace blco

extern "C" {

void blco_cpals_free(blco_cpals_state* s)
{
    if (!s) return;
    if (s->st) (void)hipStreamSynchronize(s->st);
    if (s->gexec) (void)hipGraphExecDestroy(s->gexec);
    if (s->graph) (void)hipGraphDestroy(s->graph);
    for (int m = 0; m < BLCO_MAX_MODES; ++m) {
        if (s->ev0[m]) (void)hipEventDestroy(s->ev0[m]);
        if (s->ev1[m]) (void)hipEventDestroy(s->ev1[m]);
    }
    if (s->arena) (void)hipFree(s->arena);
    if (s->h_fit) (void)hipHostFree(s->h_fit);
    if (s->it0) (void)hipEventDestroy(s->it0);
    if (s->it1) (void)hipEventDestroy(s->it1);
    delete s;
}

int blco_cpals_create(blco_dev* d, const blco_cpals_opts* o, const double* const* U,
                      blco_cpals_state** out)
{
    int rc = cpals_state_create(d, o, U, true, out);
    if (rc) return rc;
    if (hipStreamSynchronize((*out)->st) != hipSuccess) {
        blco_cpals_free(*out);
        *out = nullptr;
        return fail(BLCO_EHIP, "setup failed");
    }
    return BLCO_OK;
}

int blco_cpals_iterate(blco_cpals_state* s, int n_iters, double* fits, int* done)
{
    if (!s) return fail(BLCO_EINVAL, "null solver");
    if (done) *done = 0;
    int ran = 0;
    for (int i = 0; i < n_iters && !s->stopped; ++i) {
        const int it = s->iters_done;
        const int which = it == 0 ? 0 : 1;  // L2 at iteration 0, max norm after
        const bool use_graph = s->o.use_graph && it > 0;
        const double t0 = now_ms();
        if (it == 0) {
            // kernel 14's row-ordered copies of every mode, before any MTTKRP
            // of the sweep runs (their construction would share the GPU with it)
            for (int k = 0; k < s->N; ++k) {
                int rc = mttkrp_prepare(s->d, s->order[k], s->R, s->ft, s->o.kernel);
                if (rc) return rc;
            }
        }
        if (it == 0 || s->in_sweep) {
            // F of the first mode; every update factors the next mode's.  After a
            // sweep that ended half-way it is formed anew from the Grams, which
            // are those of the factors as they are.
            AlsLaunch l = s->upd[s->order[s->N - 1]];
            const int rc = launch_als_begin(l, s->R, s->eps, s->st);
            if (rc) return rc;
        }
        HIP_TRY(hipEventRecord(s->it0, s->st));
        if (s->m_dirty) {
            const int rc = launch_fill(s->Mbuf, s->m_bytes / (s->mt == BLCO_F64 ? 8 : 4), s->mt, 0.0, s->st);
            if (rc) return rc;
        }
        s->m_dirty = s->in_sweep = true;  // until the sweep is through
        if (use_graph) {
            if (!s->gexec) {
                HIP_TRY(hipStreamBeginCapture(s->st, hipStreamCaptureModeThreadLocal));
                int rc = enqueue_sweep(s, 1, false);
                hipGraph_t g = nullptr;
                hipError_t e = hipStreamEndCapture(s->st, &g);
                if (rc) { if (g) (void)hipGraphDestroy(g); return rc; }
                HIP_TRY(e);
                s->graph = g;
                HIP_TRY(hipGraphInstantiate(&s->gexec, g, nullptr, nullptr, 0));
            }
            HIP_TRY(hipGraphLaunch(s->gexec, s->st));
        } else {
            int rc = enqueue_sweep(s, which, true);
            if (rc) return rc;
        }
        HIP_TRY(hipMemcpyAsync(s->h_fit, s->fitbuf, sizeof(double) * 3, hipMemcpyDeviceToHost, s->st));
        HIP_TRY(hipEventRecord(s->it1, s->st));
        HIP_TRY(hipStreamSynchronize(s->st));
        s->m_dirty = s->in_sweep = false;
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, s->it0, s->it1));
        s->iter_ms += ms;
        if (!use_graph)
            for (int m = 0; m < s->N; ++m) {
                float mm = 0.f;
                HIP_TRY(hipEventElapsedTime(&mm, s->ev0[m], s->ev1[m]));
                s->mttkrp_ms[m] += mm;
            }
        s->iters_timed++;
        const double fit = s->h_fit[0];
        if (fits) fits[i] = fit;
        if (s->o.verbose)
            printf("--> Iter %3d: f = %0.6f f-delta = %0.6f time = %0.6f, (s)\n", it, fit,
                   fit - s->fit_old, (now_ms() - t0) / 1000.0);
        s->iters_done++;
        ++ran;
        // stop rule of cpd_alto (include/cpd.hpp:158-163); NaN also stops
        // (src/cpd_gpu.cu:195)
        if ((it > 0 && std::fabs(s->fit_old - fit) < s->o.tolerance) || std::isnan(fit)) s->stopped = true;
        s->fit_old = fit;
    }
    if (done) *done = ran;
    return BLCO_OK;
}

int blco_cpals_get(blco_cpals_state* s, double* const* U, double* lambda)
{
    if (!s) return fail(BLCO_EINVAL, "null solver");
    HIP_TRY(hipStreamSynchronize(s->st));
    const int R = s->R;
    // the stored factor carries lambda_m in its columns: scaled (and widened)
    // on the GPU into the MTTKRP buffer, piece by piece
    const uint64_t piece = std::max<uint64_t>(1, s->m_bytes / (8 * (uint64_t)R));
    for (int m = 0; m < s->N; ++m) {
        if (!U || !U[m]) continue;
        if (s->m_bytes < 8 * (uint64_t)R) {  // one float row: no room for a row of doubles
            double* t = nullptr;
            HIP_TRY(hipMalloc((void**)&t, 8 * (uint64_t)R * s->d->dims[m]));
            const int rc = launch_export(s->U[m], s->ft, s->d->dims[m], R, s->dinv + (size_t)m * R, t, s->st);
            hipError_t e = hipStreamSynchronize(s->st);
            if (e == hipSuccess) e = hipMemcpy(U[m], t, 8 * (uint64_t)R * s->d->dims[m], hipMemcpyDeviceToHost);
            (void)hipFree(t);
            if (rc) return rc;
            HIP_TRY(e);
            continue;
        }
        s->m_dirty = true;
        for (uint64_t r = 0; r < s->d->dims[m]; r += piece) {
            const uint64_t rows = std::min(piece, s->d->dims[m] - r);
            const char* from = static_cast<const char*>(s->U[m]) + r * R * dtype_size(s->ft);
            const int rc = launch_export(from, s->ft, rows, R, s->dinv + (size_t)m * R, (double*)s->Mbuf, s->st);
            if (rc) return rc;
            HIP_TRY(hipStreamSynchronize(s->st));
            HIP_TRY(hipMemcpy(U[m] + r * R, s->Mbuf, rows * R * 8, hipMemcpyDeviceToHost));
        }
    }
    if (lambda) HIP_TRY(hipMemcpy(lambda, s->lambda, sizeof(double) * s->R, hipMemcpyDeviceToHost));
    return BLCO_OK;
}

int blco_cpals_times(const blco_cpals_state* s, double* mttkrp_ms, double* iter_ms, int* iters,
                     int* kernels)
{
    if (!s) return fail(BLCO_EINVAL, "null solver");
    for (int m = 0; m < s->N; ++m) {
        if (mttkrp_ms) mttkrp_ms[m] = s->mttkrp_ms[m];
        if (kernels) kernels[m] = s->kern[m];
    }
    if (iter_ms) *iter_ms = s->iter_ms;
    if (iters) *iters = s->iters_timed;
    return BLCO_OK;
}

void blco_cpals_reset_times(blco_cpals_state* s)
{
    if (!s) return;
    for (int m = 0; m < BLCO_MAX_MODES; ++m) s->mttkrp_ms[m] = 0.0;
    s->iter_ms = 0.0;
    s->iters_timed = 0;
}

int blco_cpals(blco_dev* d, const blco_cpals_opts* o, double* const* U, double* lambda,
               double* fit_trace, int* iters, double* final_fit)
{
    blco_cpals_state* s = nullptr;
    int rc = blco_cpals_create(d, o, (const double* const*)U, &s);
    if (rc) return rc;
    if (o->verbose)
        printf("Begin CP-ALS decomposition, rank=%d maxiter=%d tolerance=%f\n", o->rank, o->max_iters,
               o->tolerance);
    int done = 0;
    rc = blco_cpals_iterate(s, o->max_iters, fit_trace, &done);
    if (!rc) rc = blco_cpals_get(s, U, lambda);
    if (!rc) {
        if (iters) *iters = done;
        if (final_fit) *final_fit = s->fit_old;
        if (o->verbose) printf("Final fit: %0.9f\n", s->fit_old);
    }
    blco_cpals_free(s);
    return rc;
}

}  // extern "C"
