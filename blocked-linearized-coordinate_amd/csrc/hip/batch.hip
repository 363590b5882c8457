// batch.hip -- many small tensors decomposed together.
//
// One persistent kernel per mode runs the MTTKRP of every tensor of the batch
// that has that mode: the work list holds chunks (64 x tpw nonzeros of one
// BLCO block of one tensor), each workgroup walks a contiguous range of it
// (XCD-aware), each wave one chunk at a time with the segmented tile
// reduction of the lvl1 kernel, reading its tensor's masks, positions,
// factors and output from a per-tensor descriptor.  The chunk size (tpw),
// waves per workgroup and workgroups per CU are picked per (mode, rank,
// factor type) by timing the candidates on the batch itself.
//
// The CP-ALS driver keeps one solver state per tensor (cpals.hpp) and runs a
// sweep on one stream, per mode: the MTTKRP of all tensors of each order in
// one launch of kernel 14 over their row-ordered copies (k_mttkrp_rows_batch;
// the persistent kernel where a copy does not fit), then the ALS update of
// all tensors in two or three launches (launch_als_update), the fits among
// them.  After iteration 0 the sweep is captured once into a hipGraph and
// replayed.  32 tensors of 14.4M nonzeros in all, FP64, rank 16: one stream
// and seven launches per tensor and mode took 75 ms for six sweeps and their
// set-up.  The reference
// decomposes one tensor per run (src/main.cpp:322-390); this has no
// counterpart there.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <list>
#include <new>
#include <vector>

#include "als.hpp"
#include "cpals.hpp"
#include "devcommon.hpp"
#include "device.hpp"
#include "mttkrp_kern.hpp"

namespace blco {

struct BatchTensor {
    const uint64_t* coords;
    const void* vals;
    const uint64_t* bcoords;
    uint64_t mask[BLCO_MAX_MODES];
    int pos[BLCO_MAX_MODES];
    const void* f[BLCO_MAX_MODES];
    void* out;
    int nmodes;
};

constexpr int BATCH_MAX_WAVES = 8;

namespace {

template <int L>
constexpr size_t wave_lds_bytes(size_t acc)
{
    return (size_t)BLCO_MAX_MODES * (WAVE + WAVE / L) * 8 + (WAVE + WAVE / L) * acc;
}

template <int N, typename FT, typename VT, int C, int L, bool EXACT>
__device__ __forceinline__ void batch_chunk(const MttkrpArgs& a, const BatchChunk& ch, int lane,
                                            uint64_t (*s_idx)[WAVE + WAVE / L],
                                            typename Acc<FT>::type* s_val)
{
    using AT = typename Acc<FT>::type;
    uint64_t bc[N];
    #pragma unroll
    for (int m = 0; m < N; ++m) bc[m] = a.bcoords[(uint64_t)ch.block * N + m];
    const int slot = lane / L, sub = lane % L;
    AT* out = reinterpret_cast<AT*>(a.out);
    const int R = a.rank;
    for (uint32_t t0 = 0; t0 < ch.len; t0 += WAVE) {
        const uint32_t nvalid = min((uint32_t)WAVE, ch.len - t0);
        stage_tile<N, L, VT, AT>(a, bc, ch.begin + t0, nvalid, lane, s_idx, s_val);
        for (int cb = 0; cb < (EXACT ? 1 : R); cb += C * L) {
            const int col = cb + sub * C;
            segment_tile<N, FT, C, L, EXACT>(a, nvalid, slot, col, s_idx, s_val,
                [&](uint64_t row, const AT (&acc)[C]) {
                    AT* o = out + row * (uint64_t)R + col;
                    #pragma unroll
                    for (int cc = 0; cc < C; ++cc)
                        if (EXACT || col + cc < R) atomic_add_global(o + cc, acc[cc]);
                });
        }
        wave_lds_sync();
    }
}

// blockDim.x = 64 * waves; dynamic LDS = waves * wave_lds_bytes<L>.
template <typename FT, typename VT, int C, int L, bool EXACT>
__global__ __launch_bounds__(BATCH_MAX_WAVES * WAVE) void k_mttkrp_batch(
    const BatchTensor* __restrict__ tens, const BatchChunk* __restrict__ chunks, uint32_t nchunks,
    uint32_t per_wg, int mode, int rank)
{
    using AT = typename Acc<FT>::type;
    extern __shared__ __align__(16) unsigned char s_dyn[];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, waves = blockDim.x >> 6;
    unsigned char* mine = s_dyn + (size_t)w * wave_lds_bytes<L>(sizeof(AT));
    auto s_idx = reinterpret_cast<uint64_t (*)[WAVE + WAVE / L]>(mine);
    AT* s_val = reinterpret_cast<AT*>(mine + (size_t)BLCO_MAX_MODES * (WAVE + WAVE / L) * 8);
    const uint32_t g = xcd_remap(blockIdx.x, gridDim.x);
    const uint64_t c0 = (uint64_t)g * per_wg;
    const uint64_t c1 = min(c0 + per_wg, (uint64_t)nchunks);
    for (uint64_t c = c0 + w; c < c1; c += waves) {  // whole waves; no block barriers
        const BatchChunk ch = chunks[c];
        const BatchTensor& td = tens[ch.tensor];
        MttkrpArgs a;  // the fields the tile helpers read
        a.coords = td.coords;
        a.vals = td.vals;
        a.coord_base = 0;
        a.bcoords = td.bcoords;
        #pragma unroll
        for (int m = 0; m < BLCO_MAX_MODES; ++m) {
            a.mask[m] = td.mask[m];
            a.pos[m] = td.pos[m];
            a.f[m] = td.f[m];
        }
        a.nmodes = td.nmodes;
        a.mode = mode;
        a.rank = rank;
        a.out = td.out;
        switch (td.nmodes) {
            case 2: batch_chunk<2, FT, VT, C, L, EXACT>(a, ch, lane, s_idx, s_val); break;
            case 3: batch_chunk<3, FT, VT, C, L, EXACT>(a, ch, lane, s_idx, s_val); break;
            case 4: batch_chunk<4, FT, VT, C, L, EXACT>(a, ch, lane, s_idx, s_val); break;
            default: batch_chunk<5, FT, VT, C, L, EXACT>(a, ch, lane, s_idx, s_val); break;
        }
    }
}

template <typename FT, typename VT>
const void* batch_kernel(const Shape& s, size_t* per_wave)
{
    using AT = typename Acc<FT>::type;
#define BK(C_, L_, EX_)                                         \
    do {                                                        \
        *per_wave = wave_lds_bytes<L_>(sizeof(AT));             \
        return (const void*)&k_mttkrp_batch<FT, VT, C_, L_, EX_>; \
    } while (0)
    if (s.exact) {
        if (s.C == 1 && s.L == 8) BK(1, 8, true);
        if (s.C == 2 && s.L == 8) BK(2, 8, true);
        if constexpr (sizeof(FT) == 8) {
            if (s.C == 4 && s.L == 8) BK(4, 8, true);
            if (s.C == 4 && s.L == 16) BK(4, 16, true);
        } else if constexpr (sizeof(FT) == 4) {
            if (s.C == 4 && s.L == 8) BK(4, 8, true);
            if (s.C == 4 && s.L == 16) BK(4, 16, true);
        } else {
            if (s.C == 4 && s.L == 8) BK(4, 8, true);
            if (s.C == 8 && s.L == 8) BK(8, 8, true);
        }
        return nullptr;
    }
    if (s.L == 8) BK(1, 8, false);
    if (s.L == 16) BK(1, 16, false);
    if (s.L == 32) BK(1, 32, false);
    BK(1, 64, false);
#undef BK
}

struct ChunkList {
    int tpw = 0, mode = 0;
    BatchChunk* d = nullptr;
    uint32_t n = 0;
};

struct Tuned {
    int mode, rank, ftype;
    int tpw, waves, wpc;
    float ms;
};

int num_cus()
{
    static int n = 0;
    if (!n) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            n = v;
        else
            n = 256;
    }
    return n;
}

}  // namespace
}  // namespace blco

using namespace blco;

namespace blco {
// The chunks of the tensors of one order for a mode of kernel 14, valid for
// the copies named by `copies`.
struct RowsList {
    int mode, order;
    std::vector<uint64_t> copies;
    BatchChunk* d = nullptr;
    uint32_t n = 0;
};
}  // namespace blco

struct blco_batch {
    std::vector<blco_dev*> devs;
    int maxN = 0;
    int device = 0;
    hipStream_t st = nullptr;
    std::list<ChunkList> lists;
    std::list<RowsList> rows_lists;
    bool no_rows[BLCO_MAX_MODES][3] = {};  // no device memory for the copies of a mode (and factor type)
    std::vector<Tuned> tuned;
    BatchTensor* d_tens = nullptr;  // descriptors of blco_batch_mttkrp calls
    size_t tens_cap = 0;
};

namespace blco {
namespace {

// Tensors that have mode `mode`, in batch order (the descriptor order).
std::vector<int> members(const blco_batch* b, int mode)
{
    std::vector<int> t;
    for (size_t i = 0; i < b->devs.size(); ++i)
        if (b->devs[i]->nmodes > mode) t.push_back((int)i);
    return t;
}

const ChunkList* chunk_list(blco_batch* b, int tpw, int mode)
{
    for (auto& l : b->lists)
        if (l.tpw == tpw && l.mode == mode) return &l;
    ChunkList l;
    l.tpw = tpw;
    l.mode = mode;
    std::vector<BatchChunk> h;
    const uint64_t span = (uint64_t)WAVE * tpw;
    const std::vector<int> mem = members(b, mode);
    for (size_t k = 0; k < mem.size(); ++k) {
        const blco_dev* d = b->devs[mem[k]];
        for (uint64_t blk = 0; blk < d->nblocks; ++blk)
            for (uint64_t s0 = 0; s0 < d->bnnz[blk]; s0 += span) {
                BatchChunk c;
                c.begin = d->bstart[blk] + s0;
                c.len = (uint32_t)std::min<uint64_t>(span, d->bnnz[blk] - s0);
                c.block = (uint32_t)blk;
                c.tensor = (uint32_t)k;
                c.pad = 0;
                h.push_back(c);
            }
    }
    l.n = (uint32_t)h.size();
    if (l.n) {
        if (hipMalloc(&l.d, sizeof(BatchChunk) * l.n) != hipSuccess) {
            fail(BLCO_ENOMEM, "device allocation of the batch work list failed");
            return nullptr;
        }
        if (hipMemcpy(l.d, h.data(), sizeof(BatchChunk) * l.n, hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(l.d);
            fail(BLCO_EHIP, "upload of the batch work list failed");
            return nullptr;
        }
    }
    b->lists.push_back(l);
    return &b->lists.back();
}

// Descriptors of the members of `mode` (host), factors F[t * MAX_MODES + m]
// and outputs O[t] indexed by batch position.
std::vector<BatchTensor> descriptors(const blco_batch* b, int mode, void* const* F, void* const* O)
{
    std::vector<BatchTensor> v;
    for (int t : members(b, mode)) {
        const blco_dev* d = b->devs[t];
        BatchTensor x{};
        x.coords = d->d_coords;
        x.vals = d->d_vals;
        x.bcoords = d->d_bcoords;
        for (int m = 0; m < d->nmodes; ++m) {
            x.mask[m] = d->masks[m];
            x.pos[m] = d->pos[m];
            x.f[m] = F[(size_t)t * BLCO_MAX_MODES + m];
        }
        x.out = O[t];
        x.nmodes = d->nmodes;
        v.push_back(x);
    }
    return v;
}

int launch_batch(blco_batch* b, const BatchTensor* d_tens, int mode, int rank, int ftype, int tpw, int waves,
                 int wpc, hipStream_t st)
{
    const ChunkList* l = chunk_list(b, tpw, mode);
    if (!l) return BLCO_ENOMEM;
    if (!l->n) return BLCO_OK;
    const Shape s = pick_shape(rank, dtype_size(ftype));
    size_t per_wave = 0;
    const void* k = ftype == BLCO_F64   ? batch_kernel<double, double>(s, &per_wave)
                    : ftype == BLCO_F32 ? batch_kernel<float, float>(s, &per_wave)
                                        : batch_kernel<bf16, float>(s, &per_wave);
    if (!k) return fail(BLCO_EUNSUPPORTED, "no batch MTTKRP kernel for rank %d", rank);
    const uint64_t wgs_needed = (l->n + waves - 1) / waves;
    const uint32_t grid = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(wgs_needed, (uint64_t)wpc * num_cus()));
    uint32_t per_wg = (uint32_t)((l->n + grid - 1) / grid);
    const size_t lds = per_wave * waves;
    uint32_t nchunks = l->n;
    const BatchChunk* chunks = l->d;
    void* params[] = {(void*)&d_tens, (void*)&chunks, &nchunks, &per_wg, &mode, &rank};
    if (lds > 64 * 1024) HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    HIP_TRY(hipLaunchKernel(k, dim3(grid), dim3(waves * WAVE), params, lds, st));
    return BLCO_OK;
}

const int TPW_SET[] = {1, 2, 4, 8};
const int WAVES_SET[] = {1, 2, 4, 8};
const int WPC_SET[] = {1, 2, 4, 8};

// Times every (tpw, waves, workgroups per CU) on the batch (outputs are
// overwritten) and keeps the fastest.
int tune(blco_batch* b, const BatchTensor* d_tens, int mode, int rank, int ftype, Tuned* out)
{
    for (const Tuned& t : b->tuned)
        if (t.mode == mode && t.rank == rank && t.ftype == ftype) {
            *out = t;
            return BLCO_OK;
        }
    hipEvent_t e0, e1;
    HIP_TRY(hipEventCreate(&e0));
    HIP_TRY(hipEventCreate(&e1));
    Tuned best{mode, rank, ftype, 4, 4, 4, -1.f};
    int rc = BLCO_OK;
    for (int tpw : TPW_SET)
        for (int waves : WAVES_SET)
            for (int wpc : WPC_SET) {
                if (waves * wpc > 32) continue;  // beyond the waves a CU holds
                rc = launch_batch(b, d_tens, mode, rank, ftype, tpw, waves, wpc, b->st);  // warm
                if (rc) break;
                (void)hipEventRecord(e0, b->st);
                for (int r = 0; r < 2 && !rc; ++r) rc = launch_batch(b, d_tens, mode, rank, ftype, tpw, waves, wpc, b->st);
                (void)hipEventRecord(e1, b->st);
                if (hipEventSynchronize(e1) != hipSuccess) rc = fail(BLCO_EHIP, "tuning run failed");
                if (rc) break;
                float ms = 0.f;
                (void)hipEventElapsedTime(&ms, e0, e1);
                ms /= 2.f;
                if (best.ms < 0 || ms < best.ms) best = Tuned{mode, rank, ftype, tpw, waves, wpc, ms};
            }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    b->tuned.push_back(best);
    *out = best;
    return BLCO_OK;
}

// The chunk list of the tensors `who` (all of one order) for kernel 14.
const RowsList* rows_list(blco_batch* b, int mode, int order, const std::vector<int>& who)
{
    constexpr int TPW = 2;  // as for single tensors of these sizes
    std::vector<uint64_t> copies;
    for (int t : who) copies.push_back(b->devs[t]->copy_id[mode]);
    for (auto it = b->rows_lists.begin(); it != b->rows_lists.end(); ++it)
        if (it->mode == mode && it->order == order) {
            if (it->copies == copies) return &*it;
            if (it->d) (void)hipFree(it->d);  // a copy was rebuilt
            b->rows_lists.erase(it);
            break;
        }
    RowsList l{mode, order, copies};
    std::vector<BatchChunk> h;
    for (size_t k = 0; k < who.size(); ++k)
        for (const Chunk& c : rows_batch_chunks(b->devs[who[k]], mode, TPW))
            if (c.len) h.push_back(BatchChunk{c.begin, c.len, c.block, (uint32_t)k, 0});
    l.n = (uint32_t)h.size();
    if (l.n) {
        if (hipMalloc(&l.d, sizeof(BatchChunk) * l.n) != hipSuccess) {
            fail(BLCO_ENOMEM, "device allocation of the batch chunk list failed");
            return nullptr;
        }
        if (hipMemcpy(l.d, h.data(), sizeof(BatchChunk) * l.n, hipMemcpyHostToDevice) != hipSuccess) {
            (void)hipFree(l.d);
            fail(BLCO_EHIP, "upload of the batch chunk list failed");
            return nullptr;
        }
    }
    b->rows_lists.push_back(l);
    return &b->rows_lists.back();
}

int launch_rows_batch(const RowsList* l, const MttkrpArgs* d_args, int rank, int ftype, hipStream_t st)
{
    if (!l->n) return BLCO_OK;
    int C, L;
    const void* k = mttkrp_kernel(W_ROWS_BATCH, l->order, ftype, rank, &C, &L);
    if (!k) return fail(BLCO_EUNSUPPORTED, "no batch MTTKRP kernel for %d modes, rank %d", l->order, rank);
    const BatchChunk* chunks = l->d;
    uint32_t n = l->n;
    void* params[] = {(void*)&d_args, (void*)&chunks, &n};
    HIP_TRY(hipLaunchKernel(k, dim3((n + WAVES_PER_WG - 1) / WAVES_PER_WG), dim3(WG), params, 0, st));
    return BLCO_OK;
}

int check_call(const blco_batch* b, int mode, int rank, int ftype)
{
    if (!b) return fail(BLCO_EINVAL, "null batch");
    if (mode < 0 || mode >= b->maxN) return fail(BLCO_EINVAL, "mode %d: no tensor of the batch has it", mode);
    if (rank < 1 || rank > 64) return fail(BLCO_EUNSUPPORTED, "rank %d outside [1, 64]", rank);
    if (ftype < BLCO_F64 || ftype > BLCO_BF16) return fail(BLCO_EINVAL, "factor dtype %d", ftype);
    const int need_v = ftype == BLCO_F64 ? BLCO_F64 : BLCO_F32;
    for (const blco_dev* d : b->devs)
        if (d->vdtype != need_v) return fail(BLCO_EINVAL, "factor dtype %d needs %s values in every tensor",
                                             ftype, need_v == BLCO_F64 ? "f64" : "f32");
    return BLCO_OK;
}

int upload_descriptors(blco_batch* b, const std::vector<BatchTensor>& v)
{
    if (b->tens_cap < v.size()) {
        if (b->d_tens) (void)hipFree(b->d_tens);
        b->d_tens = nullptr;
        b->tens_cap = 0;
        HIP_TRY(hipMalloc(&b->d_tens, sizeof(BatchTensor) * v.size()));
        b->tens_cap = v.size();
    }
    if (!v.empty()) HIP_TRY(hipMemcpy(b->d_tens, v.data(), sizeof(BatchTensor) * v.size(), hipMemcpyHostToDevice));
    return BLCO_OK;
}

// What a blco_batch_cpals call holds, given back however it ends.
struct BatchRun {
    blco_batch* b;
    std::vector<blco_cpals_state*> S;
    std::vector<BatchTensor*> d_desc;
    char* d_pack = nullptr;  // kernel arguments and ALS tasks of every mode
    double *d_fits = nullptr, *h_fits = nullptr;
    double* d_export = nullptr;  // every tensor's factors and lambda, f64
    hipEvent_t it0 = nullptr, it1 = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;

    BatchRun(blco_batch* batch, int T) : b(batch), S(T, nullptr), d_desc(batch->maxN, nullptr) {}
    ~BatchRun()
    {
        if (b->st) (void)hipStreamSynchronize(b->st);
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        for (blco_cpals_state* s : S)
            if (s) blco_cpals_free(s);
        for (BatchTensor* p : d_desc)
            if (p) (void)hipFree(p);
        if (d_pack) (void)hipFree(d_pack);
        if (d_fits) (void)hipFree(d_fits);
        if (d_export) (void)hipFree(d_export);
        if (h_fits) (void)hipHostFree(h_fits);
        for (hipEvent_t e : {it0, it1})
            if (e) (void)hipEventDestroy(e);
    }
};

}  // namespace
}  // namespace blco

extern "C" {

int blco_batch_create(int ntensors, blco_dev* const* devs, blco_batch** out)
{
    if (!out) return fail(BLCO_EINVAL, "null output handle");
    *out = nullptr;
    if (ntensors < 1 || !devs) return fail(BLCO_EINVAL, "empty batch");
    for (int t = 0; t < ntensors; ++t) {
        if (!devs[t]) return fail(BLCO_EINVAL, "tensor %d is null", t);
        if (devs[t]->stream_data) return fail(BLCO_EUNSUPPORTED, "tensor %d is streamed; a batch needs resident tensors", t);
        if (devs[t]->nnz >= (1ull << 40)) return fail(BLCO_EUNSUPPORTED, "tensor %d is too large for a batch", t);
    }
    blco_batch* b = new (std::nothrow) blco_batch();
    if (!b) return fail(BLCO_ENOMEM, "out of host memory");
    b->devs.assign(devs, devs + ntensors);
    for (blco_dev* d : b->devs) b->maxN = std::max(b->maxN, d->nmodes);
    if (hipGetDevice(&b->device) != hipSuccess || hipStreamCreateWithFlags(&b->st, hipStreamNonBlocking) != hipSuccess) {
        delete b;
        return fail(BLCO_EHIP, "stream creation failed");
    }
    *out = b;
    return BLCO_OK;
}

void blco_batch_free(blco_batch* b)
{
    if (!b) return;
    if (b->st) (void)hipStreamSynchronize(b->st);
    for (auto& l : b->lists)
        if (l.d) (void)hipFree(l.d);
    for (auto& l : b->rows_lists)
        if (l.d) (void)hipFree(l.d);
    if (b->d_tens) (void)hipFree(b->d_tens);
    if (b->st) (void)hipStreamDestroy(b->st);
    delete b;
}

int blco_batch_tune(blco_batch* b, int mode, int rank, int factor_dtype, void* const* factors,
                    void* const* outs, int* tpw, int* waves, int* wgs_per_cu, float* ms)
{
    int rc = check_call(b, mode, rank, factor_dtype);
    if (rc) return rc;
    if (!factors || !outs) return fail(BLCO_EINVAL, "null factor or output table");
    rc = upload_descriptors(b, descriptors(b, mode, factors, outs));
    if (rc) return rc;
    Tuned t;
    rc = tune(b, b->d_tens, mode, rank, factor_dtype, &t);
    if (rc) return rc;
    if (tpw) *tpw = t.tpw;
    if (waves) *waves = t.waves;
    if (wgs_per_cu) *wgs_per_cu = t.wpc;
    if (ms) *ms = t.ms;
    HIP_TRY(hipStreamSynchronize(b->st));
    return BLCO_OK;
}

int blco_batch_mttkrp(blco_batch* b, int mode, int rank, int factor_dtype, void* const* factors,
                      void* const* outs, int tpw, int waves, int wgs_per_cu)
{
    int rc = check_call(b, mode, rank, factor_dtype);
    if (rc) return rc;
    if (!factors || !outs) return fail(BLCO_EINVAL, "null factor or output table");
    for (int t : members(b, mode)) {
        if (!outs[t]) return fail(BLCO_EINVAL, "output of tensor %d is null", t);
        for (int m = 0; m < b->devs[t]->nmodes; ++m)
            if (!factors[(size_t)t * BLCO_MAX_MODES + m])
                return fail(BLCO_EINVAL, "factor %d of tensor %d is null", m, t);
    }
    if (tpw < 0 || tpw > 64 || waves < 0 || waves > BATCH_MAX_WAVES || wgs_per_cu < 0 || wgs_per_cu > 32)
        return fail(BLCO_EINVAL, "bad launch shape (%d, %d, %d)", tpw, waves, wgs_per_cu);
    rc = upload_descriptors(b, descriptors(b, mode, factors, outs));
    if (rc) return rc;
    if (!tpw || !waves || !wgs_per_cu) {  // the tuned shape, else a default
        tpw = 4;
        waves = 4;
        wgs_per_cu = 4;
        for (const Tuned& t : b->tuned)
            if (t.mode == mode && t.rank == rank && t.ftype == factor_dtype) {
                tpw = t.tpw;
                waves = t.waves;
                wgs_per_cu = t.wpc;
            }
    }
    rc = launch_batch(b, b->d_tens, mode, rank, factor_dtype, tpw, waves, wgs_per_cu, b->st);
    if (rc) return rc;
    HIP_TRY(hipStreamSynchronize(b->st));
    return BLCO_OK;
}

static int batch_cpals(blco_batch* b, const blco_cpals_opts* o, double* const* U, double* lambda, double* fits,
                       int* iters, double* iter_ms)
{
    if (!b || !o || !U) return fail(BLCO_EINVAL, "null argument");
    const int T = (int)b->devs.size(), R = o->rank;
    const int ft = o->precision;
    int rc = check_call(b, 0, R, ft);
    if (rc) return rc;
    blco_cpals_opts o2 = *o;
    o2.use_graph = 0;
    o2.mode_order = 0;  // modes 0..N-1 in every tensor
    o2.verbose = 0;
    BatchRun run(b, T);
    std::vector<blco_cpals_state*>& S = run.S;
    std::vector<BatchTensor*>& d_desc = run.d_desc;
    char*& d_pack = run.d_pack;
    double *&d_fits = run.d_fits, *&h_fits = run.h_fits, *&d_export = run.d_export;
    hipEvent_t &it0 = run.it0, &it1 = run.it1;
    hipGraph_t& graph = run.graph;
    hipGraphExec_t& gexec = run.gexec;
    for (int t = 0; t < T; ++t) {
        rc = cpals_state_create(b->devs[t], &o2, (const double* const*)(U + (size_t)t * BLCO_MAX_MODES), false, &S[t]);
        if (rc) return rc;
        rc = launch_fill(S[t]->Mbuf, S[t]->m_bytes / (S[t]->mt == BLCO_F64 ? 8 : 4), S[t]->mt, 0.0, S[t]->st);
        if (rc) return rc;
    }
    // every tensor's fit lands in one array: one read-back per iteration
    std::vector<uint64_t> export_at(T + 1, 0);
    for (int t = 0; t < T; ++t) {
        export_at[t + 1] = export_at[t] + R;
        for (int m = 0; m < S[t]->N; ++m) export_at[t + 1] += S[t]->d->dims[m] * (uint64_t)R;
    }
    if (hipMalloc((void**)&d_fits, sizeof(double) * 4 * T) != hipSuccess ||
        hipMalloc((void**)&d_export, sizeof(double) * export_at[T]) != hipSuccess ||
        hipHostMalloc((void**)&h_fits, sizeof(double) * 4 * T, hipHostMallocDefault) != hipSuccess)
        return fail(BLCO_ENOMEM, "batch result buffers");
    if (hipEventCreate(&it0) != hipSuccess || hipEventCreate(&it1) != hipSuccess)
        return fail(BLCO_EHIP, "event creation failed");
    // per mode: the tensors of each order through kernel 14 over their copies,
    // or the mode's members through the tuned persistent kernel when a copy
    // cannot be had; then the members' update tasks
    struct Group { const RowsList* list; size_t args; };
    std::vector<std::vector<Group>> groups;
    std::vector<bool> by_rows;
    std::vector<Tuned> shape(b->maxN);
    std::vector<AlsLaunch> upd;
    AlsLaunch begin;
    std::vector<std::pair<int, int>> built;  // (tensor, mode) of the copies that this call built
    // drops the copies built since there were `keep` of them
    auto drop_built = [&](size_t keep) {
        for (; built.size() > keep; built.pop_back()) drop_row_copy(b->devs[built.back().first], built.back().second);
    };
    auto plan = [&](bool rows) -> int {
        groups.assign(b->maxN, {});
        by_rows.assign(b->maxN, rows);
        upd.assign(b->maxN, AlsLaunch());
        std::vector<char> pack;
        auto append = [&](const void* p, size_t bytes) {
            const size_t at = (pack.size() + 63) / 64 * 64;
            pack.resize(at + bytes);
            std::memcpy(pack.data() + at, p, bytes);
            return at;
        };
        std::vector<size_t> task_at(b->maxN + 1);
        for (int n = 0; n < b->maxN; ++n) {
            const std::vector<int> mem = members(b, n);
            if (b->no_rows[n][ft]) by_rows[n] = false;
            const size_t before = built.size();
            for (size_t i = 0; i < mem.size() && by_rows[n]; ++i) {
                blco_dev* d = b->devs[mem[i]];
                const bool had = d->d_scoords[n] != nullptr;
                const int r = rows_batch_prepare(d, n, R, ft);
                if (!had && d->d_scoords[n]) built.emplace_back(mem[i], n);
                if (r == BLCO_ENOMEM || r == BLCO_EUNSUPPORTED) {
                    // this mode's copies of the other tensors would only take room
                    by_rows[n] = false;
                    b->no_rows[n][ft] = r == BLCO_ENOMEM;
                    drop_built(before);
                } else if (r) {
                    return r;
                }
            }
            std::vector<AlsTask> tasks;
            for (int t : mem) {
                AlsTask k = S[t]->tasks[n];
                k.fit = d_fits + 4 * t;
                k.first = upd[n].blocks;
                upd[n].blocks += k.parts;
                upd[n].most_parts = std::max(upd[n].most_parts, k.parts);
                tasks.push_back(k);
            }
            upd[n].ntasks = (int)tasks.size();
            task_at[n] = append(tasks.data(), sizeof(AlsTask) * tasks.size());
            if (!by_rows[n]) continue;
            for (int order = 2; order <= BLCO_MAX_MODES; ++order) {
                std::vector<int> who;
                for (int t : mem)
                    if (b->devs[t]->nmodes == order) who.push_back(t);
                if (who.empty()) continue;
                std::vector<MttkrpArgs> args;
                for (int t : who) {
                    MttkrpArgs a = rows_batch_args(b->devs[t], n, R);
                    for (int m = 0; m < order; ++m) a.f[m] = S[t]->U[m];
                    a.out = S[t]->Mbuf;
                    args.push_back(a);
                }
                const RowsList* l = rows_list(b, n, order, who);
                if (!l) return BLCO_ENOMEM;
                groups[n].push_back(Group{l, append(args.data(), sizeof(MttkrpArgs) * args.size())});
            }
        }
        // the tasks of every tensor's last mode, whose successor is mode 0
        {
            std::vector<AlsTask> tasks;
            for (int t = 0; t < T; ++t) tasks.push_back(S[t]->tasks[S[t]->N - 1]);
            begin.ntasks = T;
            task_at[b->maxN] = append(tasks.data(), sizeof(AlsTask) * tasks.size());
        }
        if (d_pack) (void)hipFree(d_pack);
        d_pack = nullptr;
        if (hipMalloc((void**)&d_pack, pack.size()) != hipSuccess) return fail(BLCO_ENOMEM, "batch descriptors");
        if (hipMemcpy(d_pack, pack.data(), pack.size(), hipMemcpyHostToDevice) != hipSuccess)
            return fail(BLCO_EHIP, "descriptor upload failed");
        for (int n = 0; n < b->maxN; ++n) upd[n].d_tasks = reinterpret_cast<const AlsTask*>(d_pack + task_at[n]);
        begin.d_tasks = reinterpret_cast<const AlsTask*>(d_pack + task_at[b->maxN]);
        for (int t = 0; t < T; ++t)
            if (hipStreamSynchronize(S[t]->st) != hipSuccess) return fail(BLCO_EHIP, "setup failed");
        for (int n = 0; n < b->maxN; ++n) {
            if (by_rows[n]) continue;
            std::vector<void*> F((size_t)T * BLCO_MAX_MODES, nullptr), O(T, nullptr);
            for (int t = 0; t < T; ++t) {
                for (int m = 0; m < S[t]->N; ++m) F[(size_t)t * BLCO_MAX_MODES + m] = S[t]->U[m];
                O[t] = S[t]->Mbuf;
            }
            const std::vector<BatchTensor> v = descriptors(b, n, F.data(), O.data());
            if (!d_desc[n] && hipMalloc(&d_desc[n], sizeof(BatchTensor) * std::max<size_t>(1, v.size())) != hipSuccess) {
                d_desc[n] = nullptr;
                return fail(BLCO_ENOMEM, "descriptor allocation failed");
            }
            if (!v.empty() && hipMemcpy(d_desc[n], v.data(), sizeof(BatchTensor) * v.size(), hipMemcpyHostToDevice) != hipSuccess)
                return fail(BLCO_EHIP, "descriptor upload failed");
            int r = tune(b, d_desc[n], n, R, ft, &shape[n]);
            for (int t : members(b, n))  // the tuning runs left their sums there
                if (!r) r = launch_fill(S[t]->Mbuf, S[t]->m_bytes / (S[t]->mt == BLCO_F64 ? 8 : 4), S[t]->mt, 0.0, b->st);
            if (r) return r;
        }
        return BLCO_OK;
    };
    rc = plan(true);
    if (rc == BLCO_ENOMEM && !built.empty()) {  // everything else fits without the copies
        (void)hipStreamSynchronize(b->st);
        drop_built(0);
        rc = plan(false);
    }
    if (rc) return rc;
    const double eps = S[0]->eps;
    auto sweep = [&](int which_norm) -> int {
        for (int n = 0; n < b->maxN; ++n) {
            int r = BLCO_OK;
            for (const Group& g : groups[n]) {
                r = launch_rows_batch(g.list, reinterpret_cast<const MttkrpArgs*>(d_pack + g.args), R, ft, b->st);
                if (r) return r;
            }
            if (!by_rows[n]) r = launch_batch(b, d_desc[n], n, R, ft, shape[n].tpw, shape[n].waves, shape[n].wpc, b->st);
            if (!r) r = launch_als_update(upd[n], ft, R, which_norm, eps, b->st);
            if (r) return r;
        }
        return BLCO_OK;
    };
    // results of the tensors `who` (every sweep so far is done) to the caller
    std::vector<double> host;
    auto fetch = [&](const std::vector<int>& who) -> int {
        if (who.empty()) return BLCO_OK;
        try {
            host.resize(export_at[T]);
        } catch (const std::bad_alloc&) {
            return fail(BLCO_ENOMEM, "host copy of the factors");
        }
        for (int t : who) {
            int r = enqueue_export(S[t], d_export + export_at[t]);
            if (r) return r;
            HIP_TRY(hipMemcpyAsync(d_export + export_at[t + 1] - R, S[t]->lambda, sizeof(double) * R,
                                   hipMemcpyDeviceToDevice, S[t]->st));
        }
        for (int t : who) HIP_TRY(hipStreamSynchronize(S[t]->st));
        // neighbouring tensors in one copy
        for (size_t i = 0; i < who.size();) {
            size_t j = i + 1;
            while (j < who.size() && who[j] == who[j - 1] + 1) ++j;
            const uint64_t lo = export_at[who[i]], hi = export_at[who[j - 1] + 1];
            HIP_TRY(hipMemcpy(host.data() + lo, d_export + lo, sizeof(double) * (hi - lo), hipMemcpyDeviceToHost));
            i = j;
        }
        for (int t : who) {
            const double* from = host.data() + export_at[t];
            for (int m = 0; m < S[t]->N; ++m) {
                const uint64_t n = S[t]->d->dims[m] * (uint64_t)R;
                if (double* to = U[(size_t)t * BLCO_MAX_MODES + m]) std::memcpy(to, from, sizeof(double) * n);
                from += n;
            }
            if (lambda) std::memcpy(lambda + (size_t)t * R, from, sizeof(double) * R);
        }
        return BLCO_OK;
    };

    std::vector<double> fit_old(T, 0.0);
    std::vector<int> stopped_at(T, 0);
    int alive = T, it = 0;
    double ms_sum = 0.0;
    int ms_n = 0;
    for (; it < o->max_iters && alive > 0; ++it) {
        HIP_TRY(hipEventRecord(it0, b->st));
        if (it == 0) {
            rc = launch_als_begin(begin, R, eps, b->st);
            if (!rc) rc = sweep(0);
            if (rc) return rc;
        } else {
            if (!gexec) {
                HIP_TRY(hipStreamBeginCapture(b->st, hipStreamCaptureModeThreadLocal));
                rc = sweep(1);
                hipError_t e = hipStreamEndCapture(b->st, &graph);
                if (rc) return rc;
                if (e != hipSuccess) return fail(BLCO_EHIP, "sweep capture failed: %s", hipGetErrorString(e));
                if (hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0) != hipSuccess)
                    return fail(BLCO_EHIP, "graph instantiation failed");
            }
            HIP_TRY(hipGraphLaunch(gexec, b->st));
        }
        HIP_TRY(hipEventRecord(it1, b->st));
        HIP_TRY(hipMemcpyAsync(h_fits, d_fits, sizeof(double) * 4 * T, hipMemcpyDeviceToHost, b->st));
        HIP_TRY(hipStreamSynchronize(b->st));
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, it0, it1));
        if (it > 0 || o->max_iters == 1) {
            ms_sum += ms;
            ++ms_n;
        }
        std::vector<int> done;
        for (int t = 0; t < T; ++t) {
            if (stopped_at[t]) continue;
            const double f = h_fits[4 * t];
            const bool stop = (it > 0 && std::fabs(fit_old[t] - f) < o->tolerance) || std::isnan(f) ||
                              it + 1 == o->max_iters;
            fit_old[t] = f;
            if (stop) {
                // this tensor's result is final: keep it before later sweeps move it
                stopped_at[t] = it + 1;
                --alive;
                done.push_back(t);
            }
        }
        rc = fetch(done);
        if (rc) return rc;
    }
    std::vector<int> never;  // max_iters == 0
    for (int t = 0; t < T; ++t)
        if (!stopped_at[t]) never.push_back(t);
    rc = fetch(never);
    if (rc) return rc;
    for (int t = 0; t < T; ++t) {
        if (fits) fits[t] = fit_old[t];
        if (iters) iters[t] = stopped_at[t];
    }
    if (iter_ms) *iter_ms = ms_n ? ms_sum / ms_n : 0.0;
    return BLCO_OK;
}

int blco_batch_cpals(blco_batch* b, const blco_cpals_opts* o, double* const* U, double* lambda, double* fits,
                     int* iters, double* iter_ms)
{
    try {
        return batch_cpals(b, o, U, lambda, fits, iters, iter_ms);
    } catch (const std::bad_alloc&) {
        return fail(BLCO_ENOMEM, "out of host memory");
    }
}

}  // extern "C"
