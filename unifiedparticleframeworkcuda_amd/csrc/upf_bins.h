// upf_bins.h -- particles into key order through the cell table.
//
// A particle's cell is the high part of its key, so counting the particles of
// every cell gives the cell table by a scan and every particle its cell's slots;
// within a cell (about nine particles of a fluid) a particle's slot is its rank
// by (key, previous slot).  The result is the stable sort by key, and the cell
// table with it, in four or five launches where the radix sort, the gather and
// the table took twelve.
#ifndef UPF_BINS_H_
#define UPF_BINS_H_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "upf_kernels.h"

namespace upf {

// The cell of a key: one grid, or a grid per scene (doms, scene_of; scenes keep
// their slot ranges, and their tables follow each other in the same order).
struct CellMap {
    uint32_t shift3;  // 3 block_shift
    const Dom* doms;
    const int* scene_of;
    __device__ uint32_t operator()(uint32_t key, int slot) const {
        if (!scene_of) return key >> shift3;
        const Dom& d = doms[scene_of[slot]];
        return d.cell_off + (key >> (3u * d.block_shift));
    }
};

struct Bins {
    uint2* cells;     // [first, end) of every cell; empty cells have first == end
    uint32_t ncells;
    uint32_t* count;  // ncells zeros, before and after
    uint32_t* at;     // n: place within the cell, in order of arrival
    uint64_t* place;  // n: key << 32 | previous slot, cell by cell
    uint32_t* sums;   // BIN_BLOCKS
};
constexpr int BIN_BLOCKS = 1024;

// Whether the counting pays: it reads and writes 16 bytes per cell of the table
// where the radix path clears 8 (about 3 us more per million cells), and saves
// 15 us at 3,080 particles and 59 at 1,132,556.
inline bool bins_apply(int n, uint32_t ncells) { return (uint64_t)ncells <= (1ull << 22) + 8ull * (uint64_t)n; }

// Fills B.cells and B.place for keys[0..n).  B.place[t] then goes to slot
// bin_slot(B.place, B.place[t], B.cells[its cell]).
hipError_t cell_bins(const uint32_t* keys, int n, const CellMap& map, const Bins& B, hipStream_t st);

// Slot of entry v of the cell whose entries are place[r.x .. r.y).
__device__ inline uint32_t bin_slot(const uint64_t* __restrict__ place, uint64_t v, uint2 r) {
    uint32_t rank = 0;
    for (uint32_t u = r.x; u < r.y; u += 4) {
        uint64_t w[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) w[q] = place[min(u + q, r.y - 1u)];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) rank += u + q < r.y && w[q] < v ? 1u : 0u;
    }
    return r.x + rank;
}

}  // namespace upf

#endif
