// upf_bins.h -- particles into key order through the cell table.
//
// A particle's cell is the high part of its key, so counting the particles of
// every cell gives the cell table by a scan and every particle its cell's slots;
// within a cell (about nine particles of a fluid) a particle's slot is its rank
// by (key, previous slot).  The result is the stable sort by key, and the cell
// table with it, in four or five launches where the radix sort, the gather and
// the table took twelve.  A slot's rank costs a read of its cell; cells with more
// than BIN_CROWD particles (piles, a state of NaNs) are ranked by blocks.
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
// 15 us at 3,080 particles and 59 at 1,132,556.  How full the cells are shows only
// when they have been counted: see BIN_CROWD.
inline bool bins_apply(int n, uint32_t ncells) { return (uint64_t)ncells <= (1ull << 22) + 8ull * (uint64_t)n; }

// Fills B.cells and B.place for keys[0..n); move_ranked gives the slots.
// pub: the first kernel publishes the failures so far (ctl).
hipError_t cell_bins(const uint32_t* keys, int n, const CellMap& map, const Bins& B, hipStream_t st,
                     const Ctl* ctl = nullptr, const Publish& pub = Publish{});

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

// A thread passes 4 entries in 0.15 us, so that a pile takes its square.  A block
// ranks BIN_CHUNK entries of a crowded cell: it finds the smallest and the largest
// of them by their digits, collects what lies between and ranks that in LDS.  A
// sort with all particles in one cell, by threads and by blocks: 4,096 0.21 and
// 0.31 ms, 8,192 0.38 and 0.32, 100,000 5.5 and 0.6, 1,000,000 465 and 12 (the
// radix sort: 0.24, which a simulation takes once it has met such a cell).
constexpr uint32_t BIN_CROWD = 6144, BIN_CHUNK = 2048;
constexpr int BIN_DIGIT = 11;

struct CrowdLds {
    union {
        uint32_t hist[2][1 << BIN_DIGIT];
        uint64_t chunk[BIN_CHUNK];
    };
    uint64_t vary, bound[2];  // bits in which the cell's entries differ; smallest and largest of the chunk
    uint32_t rank[2], n, starts, start[2];
    uint2 cell[2];
};

// f(entry) over the cell's entries, spread over the block, eight loads in flight
template <class F>
__device__ __forceinline__ void for_each_entry(const uint64_t* __restrict__ place, uint2 r, F f) {
    for (uint32_t u = r.x + threadIdx.x; u < r.y; u += 8 * BLOCK) {
        uint64_t w[8];
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) w[q] = place[min(u + q * BLOCK, r.y - 1u)];
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q)
            if (u + q * BLOCK < r.y) f(w[q]);
    }
}

// hist[d] += 1 for the wave's active lanes; one addition for those with the first
// lane's digit (neighbours in a pile mostly agree in the upper ones)
__device__ __forceinline__ void count_digit(uint32_t* hist, uint32_t d) {
    const uint64_t same = __builtin_amdgcn_ballot_w64(d == (uint32_t)__builtin_amdgcn_readfirstlane((int)d));
    const int lane = threadIdx.x & 63;
    const bool mine = (same >> lane) & 1;
    if (!mine || lane == __builtin_ctzll(same)) atomicAdd(hist + d, mine ? (uint32_t)__popcll(same) : 1u);
}

// move(v, slot) for the entries of cell r whose ranks are first .. first + BIN_CHUNK - 1
template <class Move>
__device__ __forceinline__ void move_chunk(const uint64_t* __restrict__ place, uint2 r, uint32_t first, CrowdLds& T,
                                           Move move) {
    const uint32_t size = min(BIN_CHUNK, r.y - r.x - first);
    const uint64_t any = place[r.x];
    if (threadIdx.x == 0) {
        T.vary = 0;
        T.n = 0;
    }
    __syncthreads();
    uint64_t x = 0;
    for_each_entry(place, r, [&](uint64_t w) { x |= w ^ any; });
    atomicOr((unsigned long long*)&T.vary, x);
    __syncthreads();
    uint64_t vary = T.vary;  // not 0: the entries differ
    if (threadIdx.x < 2) {
        T.bound[threadIdx.x] = any & ~vary;
        T.rank[threadIdx.x] = threadIdx.x == 0 ? first : first + size - 1u;
    }
    while (vary) {  // both bounds' digits from the top, by the count of the entries that share what is above
        const int top = 64 - __builtin_clzll(vary), shift = max(top - BIN_DIGIT, 0);
        const uint64_t digits = (1ull << (top - shift)) - 1ull;
        vary &= (1ull << shift) - 1ull;
        for (int k = threadIdx.x; k < 2 << BIN_DIGIT; k += BLOCK) T.hist[k >> BIN_DIGIT][k & ((1 << BIN_DIGIT) - 1)] = 0u;
        __syncthreads();
        const uint64_t above = ~((digits << shift) | ((1ull << shift) - 1ull)), b0 = T.bound[0] & above, b1 = T.bound[1] & above;
        for_each_entry(place, r, [&](uint64_t w) {
            const uint32_t d = (uint32_t)((w >> shift) & digits);
            if ((w & above) == b0) count_digit(T.hist[0], d);
            if ((w & above) == b1) count_digit(T.hist[1], d);
        });
        __syncthreads();
        // wave e: bound e, a run of digits per lane
        const int e = threadIdx.x >> 6, lane = threadIdx.x & 63;
        constexpr int RUN = (1 << BIN_DIGIT) / 64;
        if (e < 2) {
            uint32_t own = 0;
            for (int q = 0; q < RUN; ++q) own += T.hist[e][lane * RUN + q];
            uint32_t incl = own;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)incl, o, 64);
                if (lane >= o) incl += y;
            }
            const uint32_t k = T.rank[e];
            uint32_t at = incl - own;
            if (k >= at && k < incl) {  // one lane
                int q = lane * RUN;
                while (k - at >= T.hist[e][q]) at += T.hist[e][q++];
                T.bound[e] = (T.bound[e] & ~(digits << shift)) | (uint64_t)q << shift;
                T.rank[e] = k - at;
            }
        }
        __syncthreads();
    }
    const uint64_t lo = T.bound[0], hi = T.bound[1];
    for_each_entry(place, r, [&](uint64_t w) {
        if (w >= lo && w <= hi) T.chunk[atomicAdd(&T.n, 1u)] = w;
    });
    __syncthreads();
    constexpr int OWN = 4;
    for (uint32_t q0 = 0; q0 < size; q0 += OWN * BLOCK) {
        uint64_t v[OWN];
        uint32_t rank[OWN];
#pragma unroll
        for (int q = 0; q < OWN; ++q) {
            v[q] = T.chunk[min(q0 + (uint32_t)(q * BLOCK) + threadIdx.x, size - 1u)];
            rank[q] = 0;
        }
        for (uint32_t k = 0; k < size; ++k) {
            const uint64_t w = T.chunk[k];
#pragma unroll
            for (int q = 0; q < OWN; ++q) rank[q] += w < v[q] ? 1u : 0u;
        }
#pragma unroll
        for (int q = 0; q < OWN; ++q)
            if (q0 + (uint32_t)(q * BLOCK) + threadIdx.x < size) move(v[q], [&] { return r.x + first + rank[q]; });
    }
    __syncthreads();
}

// move(entry, function that gives its slot) for every entry of place; all threads
// of blocks of BLOCK call it.  *crowded is set when a cell was ranked by blocks.
template <class Move>
__device__ __forceinline__ void move_ranked(int n, const CellMap& map, const uint64_t* __restrict__ place,
                                            const uint2* __restrict__ cells, uint32_t* crowded, Move move) {
    __shared__ CrowdLds T;
    const int t = blockIdx.x * BLOCK + threadIdx.x;
    bool crowd = false;
    uint2 r = make_uint2(0u, 0u);
    if (t < n) {
        const uint64_t v = place[t];
        r = cells[map((uint32_t)(v >> 32), t)];
        crowd = r.y - r.x > BIN_CROWD;
        if (!crowd) move(v, [&] { return bin_slot(place, v, r); });
    }
    if (__syncthreads_or(crowd) == 0) return;
    // chunks start in this block at most twice: a crowded cell is larger than a block
    if (threadIdx.x == 0) T.starts = 0;
    __syncthreads();
    if (crowd && ((uint32_t)t - r.x) % BIN_CHUNK == 0) {
        const uint32_t k = atomicAdd(&T.starts, 1u);
        T.cell[k] = r;
        T.start[k] = (uint32_t)t - r.x;
        *crowded = 1u;
    }
    __syncthreads();
    const uint32_t starts = T.starts;
    for (uint32_t k = 0; k < starts; ++k) move_chunk(place, T.cell[k], T.start[k], T, move);
}

}  // namespace upf

#endif
