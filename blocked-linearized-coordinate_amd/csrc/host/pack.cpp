// pack.cpp -- the words of a streamed tensor packed for the host link, chunk by
// chunk (no reference counterpart: the reference streams its 8-byte words,
// src/alto_dev.cu:1869-1874).  Unpacked on the GPU by k_unpack (device.hip).
#include <algorithm>

#include "internal.hpp"

namespace blco {

bool pack_words(int nmodes, const uint64_t* masks, const int* pos, uint64_t nnz, const uint64_t* coords,
                const std::vector<uint64_t>& fbeg, const std::vector<uint32_t>& flen, std::vector<PackChunk>* chunks,
                uint64_t* dwords, uint32_t* widest)
{
    uint64_t used = 0;
    for (int m = 0; m < nmodes; ++m) {
        const uint64_t f = masks[m] << pos[m];
        if ((f & used) || (f >> pos[m]) != masks[m]) return false;
        used |= f;
    }
    const uint64_t nf = fbeg.size();
    chunks->assign(nf + 1, PackChunk{});
    #pragma omp parallel for schedule(static)
    for (uint64_t f = 0; f < nf; ++f) {
        PackChunk& pc = (*chunks)[f];
        pc.begin = fbeg[f];
        pc.len = flen[f];
        uint64_t lo[BLCO_MAX_MODES], hi[BLCO_MAX_MODES];
        std::fill(lo, lo + nmodes, ~0ull);
        std::fill(hi, hi + nmodes, 0);
        for (uint64_t i = pc.begin; i < pc.begin + pc.len; ++i)
            for (int m = 0; m < nmodes; ++m) {
                const uint64_t v = (coords[i] >> pos[m]) & masks[m];
                lo[m] = std::min(lo[m], v);
                hi[m] = std::max(hi[m], v);
            }
        for (int m = 0; m < nmodes; ++m) {
            pc.bits[m] = (uint8_t)(hi[m] > lo[m] ? 64 - __builtin_clzll(hi[m] - lo[m]) : 0);
            pc.base += lo[m] << pos[m];
            pc.width += pc.bits[m];
        }
    }
    uint64_t at = 0, bits = 0;
    *widest = 0;
    for (uint64_t f = 0; f <= nf; ++f) {
        PackChunk& pc = (*chunks)[f];
        pc.at = at;
        if (f == nf) break;
        at += ((uint64_t)pc.len * pc.width + 31) / 32;
        bits += (uint64_t)pc.len * pc.width;
        *widest = std::max<uint32_t>(*widest, pc.width);
    }
    *dwords = at;
    return *widest <= 60 && bits <= nnz * 48;
}

void write_packed(int nmodes, const uint64_t* masks, const int* pos, const uint64_t* coords,
                  const std::vector<PackChunk>& chunks, uint32_t* out)
{
    const uint64_t nf = chunks.size() - 1;
    #pragma omp parallel for schedule(static)
    for (uint64_t f = 0; f < nf; ++f) {
        const PackChunk& pc = chunks[f];
        uint32_t* q = out + pc.at;
        unsigned __int128 acc = 0;
        int have = 0;
        for (uint64_t i = pc.begin; i < pc.begin + pc.len; ++i) {
            int sh = have;
            for (int m = 0; m < nmodes; ++m) {
                const uint64_t lo = (pc.base >> pos[m]) & masks[m];
                acc |= (unsigned __int128)(((coords[i] >> pos[m]) & masks[m]) - lo) << sh;
                sh += pc.bits[m];
            }
            have += pc.width;
            for (; have >= 32; have -= 32, acc >>= 32) *q++ = (uint32_t)acc;
        }
        if (have > 0) *q = (uint32_t)acc;
    }
}

}  // namespace blco
