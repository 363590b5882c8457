// mttkrp.hpp -- kernel arguments and launchers of mttkrp.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "blco_host.h"

namespace blco {

// A run of nonzeros of one block handled by one wave (begin is the global
// nonzero offset in ALTO order).
struct Chunk {
    uint64_t begin;
    uint32_t len;
    uint32_t block;
};

// A workgroup's share of a block: a run of nonzeros whose output rows, for
// each mode, lie in a known [lo, hi] (the row window).
struct SuperChunk {
    uint64_t begin;
    uint32_t len;
    uint32_t block;
};

// A chunk of a tensor of a batch (an index into the launch's tensors).
struct BatchChunk {
    uint64_t begin;
    uint32_t len;
    uint32_t block;
    uint32_t tensor;
    uint32_t pad;
};

struct MttkrpArgs {
    const uint64_t* coords;  // element e lives at coords[e - coord_base]
    const void* vals;        // same indexing, f64 or f32
    uint64_t coord_base;
    const Chunk* chunks;
    uint32_t chunk0;         // first chunk of this launch
    uint32_t nchunks;        // chunks in this launch
    const uint64_t* bcoords; // block coordinates, nblocks x nmodes
    uint64_t mask[BLCO_MAX_MODES];
    int pos[BLCO_MAX_MODES];
    int nmodes;
    int mode;
    int rank;
    const void* f[BLCO_MAX_MODES];
    void* out;
    // lvl3 only
    uint64_t out_rows;
    int nprtn;
    void* partials;
    uint32_t chunks_per_wg;
    // row-window kernel only
    const SuperChunk* sc;
    const uint64_t* sc_range;  // [entry][2]: lo, hi of the output mode (non-hot rows)
    uint32_t lds_rows;         // rows the LDS window holds
    const int32_t* hot_rank;   // output mode: frequency rank of a row, -1 if not a candidate
    uint32_t hot_rows;         // ranks < hot_rows are accumulated in the LDS hot area
    const uint64_t* sc_poff;   // [entry + 1]: the entry's window is partial rows [poff[e], poff[e+1])
    uint64_t hot_poff;         // first partial row of the hot areas (entry e: + e * hot_rows)
    void* part;                // partial rows (rank wide), reduced by k_window_reduce
    // fiber-ordered copies: the mode that varies within a fiber
    int inner;
    // k_mttkrp_rows: the input modes in gather order, then the output mode
    int order[BLCO_MAX_MODES];
    // k_mttkrp_lvl3_rows: copies of the output in LDS, slot s adds to s mod this
    uint32_t lvl3_copies;
    // row-ordered kernels: chunks per wave (consecutive, or with
    // cpw_interleave one grid width apart), and for the first two input
    // modes (the inner and first outer mode with fibers) a window of rows
    // [hot_lo, hot_lo + hot_n) kept in LDS (hot_n = 0: none)
    uint32_t cpw;
    uint32_t cpw_interleave;
    uint32_t hot_lo[2];
    uint32_t hot_n[2];
};

// Launch plan of a row-ordered kernel for one (rank, factor type, windows,
// chunk count) of a mode: chunks per wave and the hot-row windows.
struct RowsPlan {
    int rank, ftype;
    bool windows;  // planned with windows, if any pay
    uint32_t nchunks, cpw, interleave, hot_lo[2], hot_n[2];
    size_t lds;
};

enum { W_LVL1 = 0, W_LVL3 = 1, W_ATOMIC = 2, W_WINDOW = 3, W_WINDOW64 = 4, W_SORTED64 = 5, W_FIBER64 = 6,
       W_SORTED_LDS = 7, W_FIBER_LDS = 8, W_ROWS = 9, W_ROWS_SHORT = 10, W_ROWS_BATCH = 11,
       W_LVL3_ROWS = 12 };

// Threads of a workgroup of k_mttkrp_lvl3_rows.  Every workgroup ends in one
// add to each output element, and in FP32 each of those rounds: with floats in
// the output a workgroup takes 64 chunks (16384 nonzeros, as many adds as the
// tile-sorting kernel), and 16 waves to run them.  Workgroups of 1024 nonzeros
// ran 300k nonzeros into 24 rows with an error of 2.6e-7 against 64 bits,
// these 18 run it with 6.9e-8 (8.2e-8 with sorted tiles and sums in floats).
constexpr int lvl3_wg(bool f64) { return f64 ? 4 * 64 : 16 * 64; }

// Doubles from row to row and from copy to copy of k_mttkrp_lvl3_rows' output in
// LDS: odd, so that the slots of a wave, which add to different rows, spread
// over the banks (at rank 32 and a stride of 32 all of them met in 16 of 64).
constexpr __host__ __device__ uint32_t lvl3_row_stride(int rank) { return (uint32_t)rank | 1; }
constexpr __host__ __device__ uint32_t lvl3_copy_stride(uint32_t rows, int rank)
{
    return rows * lvl3_row_stride(rank) | 1;
}

// The row-ordered and fiber kernels take 31-bit byte offsets into factors
// of fewer bytes than this (bit 31 marks an offset into an LDS window).
constexpr uint32_t FACTOR_BYTES_MAX = 0x80000000u;
// LDS for the hot-row windows of the row-ordered kernels (per workgroup)
constexpr uint32_t HOT_TABLE_BYTES = 24 * 1024;
constexpr uint32_t FINE_CHUNK = 1024;        // nonzeros per range-table entry
constexpr uint32_t WINDOW_LDS_BYTES = 40 * 1024;  // hot area + row window per workgroup
constexpr int WIN_WAVES = 8;                      // waves per row-window workgroup
constexpr int WIN_BATCH = 4;                      // positions whose gathers are issued together

// Field positions of a tensor's words, as a kernel argument.
struct BlcoPos {
    int p[BLCO_MAX_MODES];
};

// Marks a reduce segment whose output row is split over several segments.
constexpr uint64_t REDUCE_SHARED = 1ull << 63;

// out[rows[u]][:] += sum of the partial rows idx[ptr[u] .. ptr[u+1]), with
// an atomic add when rows[u] carries REDUCE_SHARED.
int launch_window_reduce(void* out, const void* part, const uint64_t* rows, const uint64_t* ptr,
                         const uint32_t* idx, uint64_t nrows, int rank, int otype, hipStream_t st);

const void* mttkrp_kernel(int which, int nmodes, int ftype, int rank, int* C, int* L);
int launch_mttkrp(int which, const MttkrpArgs& a, int ftype, uint32_t grid, size_t dyn_lds,
                  hipStream_t st);
int launch_reduce_partials(void* out, const void* part, uint64_t cells, int nprtn, int otype,
                           hipStream_t st);
int launch_fill(void* x, uint64_t n, int dtype, double v, hipStream_t st);

}  // namespace blco
