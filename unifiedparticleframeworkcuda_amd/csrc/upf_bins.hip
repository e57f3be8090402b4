// upf_bins.hip -- counting, scan and placement of upf_bins.h.
#include "upf_bins.h"

#include <algorithm>

namespace upf {

constexpr int BIN_THREADS = 1024;
constexpr uint32_t BIN_TILE = 4 * BIN_THREADS;  // cells per step of a block

// Arrival places in the cells.  Consecutive particles are mostly in the same
// cell (the previous step's order): one atomic per run of a wave.
__global__ __launch_bounds__(BLOCK) void k_bin_count(const uint32_t* __restrict__ keys, int n, CellMap map,
                                                     uint32_t* __restrict__ count, uint32_t* __restrict__ at,
                                                     const Ctl* ctl, Publish pub) {
    if (pub.m && blockIdx.x == 0 && threadIdx.x == 0) publish_failures(pub, *ctl, true);
    const int i = blockIdx.x * BLOCK + threadIdx.x, lane = threadIdx.x & 63;
    const bool in = i < n;
    const uint32_t c = in ? map(keys[i], i) : 0xFFFFFFFFu;  // no cell has this number
    const uint32_t prev = (uint32_t)__shfl_up((int)c, 1, 64);
    const uint64_t heads = __builtin_amdgcn_ballot_w64(lane == 0 || prev != c);
    const int head = 63 - __builtin_clzll(heads & (~0ull >> (63 - lane)));
    const uint64_t after = lane == 63 ? 0ull : heads >> (lane + 1);
    uint32_t base = 0;
    if (head == lane && in) {
        const int len = after ? __builtin_ctzll(after) + 1 : 64 - lane;
        base = atomicAdd(count + c, (uint32_t)len);
    }
    base = (uint32_t)__shfl((int)base, head, 64);
    if (in) at[i] = base + (uint32_t)(lane - head);
}

// Four cells' counts (grids are powers of two, so tables and spans are multiples of four).
__device__ __forceinline__ uint4 counts4(const uint32_t* __restrict__ count, uint64_t c, uint64_t end) {
    return c < end ? *reinterpret_cast<const uint4*>(count + c) : make_uint4(0u, 0u, 0u, 0u);
}

// Sum over the block, on every thread; part: 16 words of LDS.
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* part) {
    for (int o = 32; o > 0; o >>= 1) v += (uint32_t)__shfl_xor((int)v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    uint32_t s = 0;
    for (int w = 0; w < BIN_THREADS / 64; ++w) s += part[w];
    return s;
}

// Particles in the block's `span` cells.
__global__ __launch_bounds__(BIN_THREADS) void k_bin_sums(const uint32_t* __restrict__ count, uint32_t ncells, uint32_t span,
                                                          uint32_t* __restrict__ sums) {
    __shared__ uint32_t part[BIN_THREADS / 64];
    const uint64_t beg = (uint64_t)blockIdx.x * span, end = min(beg + span, (uint64_t)ncells);
    uint32_t s = 0;
    for (uint64_t c = beg + 4 * threadIdx.x; c < end; c += BIN_TILE) {
        const uint4 k = counts4(count, c, end);
        s += k.x + k.y + k.z + k.w;
    }
    s = block_sum(s, part);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

// The cell table of the block's `span` cells.  sums: the blocks' particles, or
// null: counted here over the cells before the block's (a small table, where
// that costs less than a launch).
__global__ __launch_bounds__(BIN_THREADS) void k_bin_scan(const uint32_t* __restrict__ count, uint32_t ncells, uint32_t span,
                                                          const uint32_t* __restrict__ sums, uint2* __restrict__ cells) {
    __shared__ uint32_t part[BIN_THREADS / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t beg = (uint64_t)blockIdx.x * span, end = min(beg + span, (uint64_t)ncells);
    uint32_t s = 0;
    if (sums) {
        if (threadIdx.x < blockIdx.x) s = sums[threadIdx.x];  // at most BIN_BLOCKS = BIN_THREADS blocks
    } else {
#pragma unroll 8
        for (uint64_t c = 4 * threadIdx.x; c < beg; c += BIN_TILE) {
            const uint4 k = counts4(count, c, beg);
            s += k.x + k.y + k.z + k.w;
        }
    }
    uint32_t run = block_sum(s, part);
    for (uint64_t t0 = beg; t0 < end; t0 += BIN_TILE) {
        const uint64_t c = t0 + 4 * threadIdx.x;
        const uint4 k = counts4(count, c, end);
        const uint32_t own = k.x + k.y + k.z + k.w;
        uint32_t incl = own;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, o, 64);
            if (lane >= o) incl += y;
        }
        __syncthreads();
        if (lane == 63) part[w] = incl;
        __syncthreads();
        uint32_t a = run + incl - own;
        for (int q = 0; q < BIN_THREADS / 64; ++q) {
            a += q < w ? part[q] : 0u;
            run += part[q];
        }
        const uint32_t b = a + k.x, d = b + k.y, e = d + k.z, f = e + k.w;
        if (c < end) {
            uint4* o = reinterpret_cast<uint4*>(cells + c);
            o[0] = make_uint4(a, b, b, d);
            o[1] = make_uint4(d, e, e, f);
        }
    }
}

// Every particle to its cell's slots, in order of arrival; the counts of the
// occupied cells go back to zero.
__global__ __launch_bounds__(BLOCK) void k_bin_place(const uint32_t* __restrict__ keys, int n, CellMap map,
                                                     const uint2* __restrict__ cells, const uint32_t* __restrict__ at,
                                                     uint64_t* __restrict__ place, uint32_t* __restrict__ count) {
    const int i = blockIdx.x * BLOCK + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = keys[i], c = map(k, i);
    place[cells[c].x + at[i]] = (uint64_t)k << 32 | (uint32_t)i;
    count[c] = 0;
}

hipError_t cell_bins(const uint32_t* keys, int n, const CellMap& map, const Bins& B, hipStream_t st, const Ctl* ctl,
                     const Publish& pub) {
    const dim3 g((unsigned)((n + BLOCK - 1) / BLOCK)), b(BLOCK);
    const uint32_t tiles = (B.ncells + BIN_TILE - 1) / BIN_TILE;
    const uint32_t per = (tiles + BIN_BLOCKS - 1) / BIN_BLOCKS, span = per * BIN_TILE;
    const dim3 gt((tiles + per - 1) / per);
    const bool direct = tiles <= 32;
    hipLaunchKernelGGL(k_bin_count, g, b, 0, st, keys, n, map, B.count, B.at, ctl, pub);
    if (!direct) hipLaunchKernelGGL(k_bin_sums, gt, dim3(BIN_THREADS), 0, st, B.count, B.ncells, span, B.sums);
    hipLaunchKernelGGL(k_bin_scan, gt, dim3(BIN_THREADS), 0, st, B.count, B.ncells, span, direct ? nullptr : B.sums, B.cells);
    hipLaunchKernelGGL(k_bin_place, g, b, 0, st, keys, n, map, B.cells, B.at, B.place, B.count);
    return hipGetLastError();
}

}  // namespace upf
