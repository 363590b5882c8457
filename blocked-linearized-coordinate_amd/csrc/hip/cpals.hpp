// cpals.hpp -- the CP-ALS solver state of one tensor and the pieces of a
// sweep, shared by the single-tensor driver (cpals.hip) and the batched
// driver (batch.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "als.hpp"
#include "blco_hip.h"
#include "device.hpp"

struct blco_cpals_state {
    blco_dev* d = nullptr;
    blco_cpals_opts o{};
    int N = 0, R = 0, ft = BLCO_F64, mt = BLCO_F64;
    hipStream_t st = nullptr;
    void* arena = nullptr;  // one device allocation for everything below
    void* U[BLCO_MAX_MODES] = {};
    double* G[BLCO_MAX_MODES] = {};
    // F (fac, colscale) belongs to the sweep's first mode between sweeps, and to
    // a later one after a sweep that an error ended
    bool in_sweep = false;
    // the MTTKRP's output, all zeros between a mode's update and the next
    // MTTKRP; m_dirty: an error or an export left something in it
    void* Mbuf = nullptr;
    uint64_t m_bytes = 0;
    bool m_dirty = true;
    double *lambda = nullptr, *fac = nullptr, *work = nullptr;
    int* status = nullptr;
    double *part = nullptr, *stats = nullptr, *fitbuf = nullptr;
    // the factors are stored unnormalised: U[m] = (normalised factor) diag(lambda_m);
    // dinv[m * R + r] = 1 / lambda_m[r] (0 for a zero column; 1 before mode m's
    // first update), and colscale the product of the other modes' dinv for
    // the mode being updated
    double *dinv = nullptr, *colscale = nullptr;
    blco::AlsTask tasks[BLCO_MAX_MODES] = {};  // by mode; the device copies behind `upd`
    blco::AlsLaunch upd[BLCO_MAX_MODES];
    double eps = 0.0;
    double* norm_part = nullptr;
    double* h_fit = nullptr;  // pinned
    int order[BLCO_MAX_MODES] = {};
    int kern[BLCO_MAX_MODES] = {};
    hipEvent_t ev0[BLCO_MAX_MODES] = {}, ev1[BLCO_MAX_MODES] = {};
    hipEvent_t it0 = nullptr, it1 = nullptr;
    double mttkrp_ms[BLCO_MAX_MODES] = {};
    double iter_ms = 0.0;
    int iters_timed = 0;
    int iters_done = 0;
    double fit_old = 0.0;
    bool stopped = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
};

namespace blco {

// The solver state of d: initial factors U (host f64), Grams, ||X||^2 and the
// tasks of every mode, all enqueued on d's stream.  The timing events and the
// pinned fit of blco_cpals_iterate come only with own_io.
int cpals_state_create(blco_dev* d, const blco_cpals_opts* o, const double* const* U, bool own_io,
                       blco_cpals_state** out);
// Factors (f64, dims x R each, one mode after the other) into out, a device
// array, on the state's stream.
int enqueue_export(blco_cpals_state* s, double* out);

}  // namespace blco
