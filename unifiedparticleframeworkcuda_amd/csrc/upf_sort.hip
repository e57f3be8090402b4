// upf_sort.hip -- stable LSD radix sort of (32-bit key, 32-bit value) pairs
// for gfx950 wave64.  Replaces the reference's RadixSort
// (src/gpu/particles.cu:31-60, kernels RadixSum / RadixPrefixSum /
// RadixAddOffsetsAndShuffle in src/gpu/radixsort_kernel.cu:64,216,339) with a
// design of its own:
//   * digits of 10 bits where that saves a pass, else of 8;
//   * a tile is one workgroup's keys; each wave ranks 64 consecutive keys per
//     round with one ballot per digit bit (lanes with equal digits form a peer
//     mask), so the rank of a key is the number of equal digits before it ->
//     stable;
//   * up to 8,192 keys: one workgroup, all passes in LDS, one launch;
//   * more: per pass a launch that counts the tiles' digits and one that
//     scatters; up to RS_FUSED_TILES tiles the scatter sums the counts of the
//     tiles before its own, beyond that a launch between them scans the counts.
//     The scatter orders its tile by digit in LDS first, so that the keys of
//     one digit leave as one contiguous run at digit base + tile offset.
#include <hip/hip_runtime.h>

#include "upf_sort.h"

namespace upf {

constexpr int RS_ONE_THREADS = 1024;
constexpr int RS_FUSED_TILES = 32;
constexpr int RS_SCAN_WAVES = 16;

__device__ __forceinline__ uint32_t rs_wave_scan(uint32_t v, int lane) {  // inclusive
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)v, o, 64);
        if (lane >= o) v += y;
    }
    return v;
}

// exclusive scan over the block's threads of one value each; part: WAVES
// words.  The caller synchronises before part is used again.
template <int WAVES>
__device__ __forceinline__ uint32_t rs_block_scan(uint32_t v, uint32_t* part, int lane, int w) {
    const uint32_t incl = rs_wave_scan(v, lane);
    if (lane == 63) part[w] = incl;
    __syncthreads();
    uint32_t before = 0;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) before += k < w ? part[k] : 0u;
    return before + incl - v;
}

// LDS of a tile: per wave the digit counts (then their starts within the
// digit), the tile's digit starts, and the tile in digit order
template <int DB, int TH, int IPT>
struct RsTile {
    uint16_t wcnt[(TH / 64)][1 << DB];
    uint32_t start[1 << DB];
    uint32_t part[(TH / 64)];
    uint32_t skey[TH * IPT], sval[TH * IPT];
};

// Digits per thread in the per-digit steps (thread t: digits t * DPT ...)
template <int DB, int TH>
constexpr int rs_dpt = (1 << DB) > TH ? (1 << DB) / TH : 1;

// Places the tile's keys (thread's key r is number (w * IPT + r) * 64 + lane of
// the tile, valid below cnt) into skey / sval in digit order; dcnt gets the
// counts of this thread's digits, start[] the digits' first places.
template <int DB, int TH, int IPT>
__device__ __forceinline__ void rs_place(RsTile<DB, TH, IPT>& T, const uint32_t (&key)[IPT], const uint32_t (&val)[IPT],
                                         int cnt, int shift, uint32_t (&dcnt)[rs_dpt<DB, TH>]) {
    constexpr int ND = 1 << DB, DPT = rs_dpt<DB, TH>;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint64_t lt = (1ull << lane) - 1ull;
    for (int k = t; k < (TH / 64) * ND / 2; k += TH) reinterpret_cast<uint32_t*>(T.wcnt)[k] = 0u;
    __syncthreads();
    uint32_t rank[IPT];
    uint16_t* mine = T.wcnt[w];
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const bool valid = (w * IPT + r) * 64 + lane < cnt;
        const uint32_t d = (key[r] >> shift) & (ND - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t before = (uint32_t)__popcll(peers & lt);
        const uint32_t cur = mine[d];
        rank[r] = cur + before;
        // all lanes of the wave have read the count before the leaders write it
        __builtin_amdgcn_wave_barrier();
        if (valid && before == 0) mine[d] = (uint16_t)(cur + (uint32_t)__popcll(peers));
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // per digit: exclusive prefix over the waves, and the tile's count
    uint32_t own = 0;
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
        const int d = t * DPT + q;
        dcnt[q] = 0;
        if (d < ND) {
#pragma unroll
            for (int k = 0; k < (TH / 64); ++k) {
                const uint32_t c = T.wcnt[k][d];
                T.wcnt[k][d] = (uint16_t)dcnt[q];
                dcnt[q] += c;
            }
        }
        own += dcnt[q];
    }
    uint32_t at = rs_block_scan<TH / 64>(own, T.part, lane, w);
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
        if (t * DPT + q < ND) T.start[t * DPT + q] = at;
        at += dcnt[q];
    }
    __syncthreads();
    // stable: wave, round, lane order within a digit
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        if ((w * IPT + r) * 64 + lane < cnt) {
            const uint32_t d = (key[r] >> shift) & (ND - 1);
            const uint32_t p = T.start[d] + mine[d] + rank[r];
            T.skey[p] = key[r];
            T.sval[p] = val[r];
        }
    }
    __syncthreads();
}

// up to TH * IPT keys in one workgroup
template <int DB, int TH, int IPT>
__global__ __launch_bounds__(TH) void rs_one(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                     uint32_t* __restrict__ kout, uint32_t* __restrict__ vout, int n,
                                                     int passes) {
    __shared__ RsTile<DB, TH, IPT> T;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t key[IPT], val[IPT], dcnt[rs_dpt<DB, TH>];
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int idx = (w * IPT + r) * 64 + lane;
        key[r] = idx < n ? kin[idx] : 0u;
        val[r] = idx < n ? (vin ? vin[idx] : (uint32_t)idx) : 0u;
    }
    for (int p = 0; p < passes; ++p) {
        if (p) {
#pragma unroll
            for (int r = 0; r < IPT; ++r) {
                const int idx = (w * IPT + r) * 64 + lane;
                key[r] = T.skey[idx];  // beyond n: not used
                val[r] = T.sval[idx];
            }
            // rs_place synchronises before it writes skey / sval
        }
        rs_place<DB, TH, IPT>(T, key, val, n, DB * p, dcnt);
    }
    for (int q = threadIdx.x; q < n; q += TH) {
        kout[q] = T.skey[q];
        vout[q] = T.sval[q];
    }
}

// digit counts of every tile: hist[tile][digit]
template <int DB, int TH, int IPT>
__global__ __launch_bounds__(TH) void rs_hist(const uint32_t* __restrict__ keys, int n, int shift,
                                                      uint32_t* __restrict__ hist) {
    constexpr int ND = 1 << DB;
    __shared__ uint32_t cnt[ND];
    for (int d = threadIdx.x; d < ND; d += TH) cnt[d] = 0;
    __syncthreads();
    const int base = blockIdx.x * (TH * IPT);
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int idx = base + r * TH + (int)threadIdx.x;
        if (idx < n) atomicAdd(&cnt[(keys[idx] >> shift) & (ND - 1)], 1u);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < ND; d += TH) hist[(size_t)blockIdx.x * ND + d] = cnt[d];
}

// 64 digits per workgroup: the tile counts of each digit become exclusive
// prefixes over the tiles, the totals go to totals[digit].  Each wave sums a
// run of tiles (rows of 64 counts), then walks it again from its start.
template <int DB>
__global__ __launch_bounds__(64 * RS_SCAN_WAVES) void rs_scan(uint32_t* __restrict__ hist, int ntiles,
                                                      uint32_t* __restrict__ totals) {
    constexpr int ND = 1 << DB;
    __shared__ uint32_t sum[RS_SCAN_WAVES][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t* col = hist + blockIdx.x * 64 + lane;
    const int per = (ntiles + RS_SCAN_WAVES - 1) / RS_SCAN_WAVES;
    const int beg = min(w * per, ntiles), end = min(beg + per, ntiles);
    uint32_t s = 0;
#pragma unroll 8
    for (int i = beg; i < end; ++i) s += col[(size_t)i * ND];
    sum[w][lane] = s;
    __syncthreads();
    uint32_t run = 0, all = 0;
#pragma unroll
    for (int k = 0; k < RS_SCAN_WAVES; ++k) {
        run += k < w ? sum[k][lane] : 0u;
        all += sum[k][lane];
    }
    if (w == 0) totals[blockIdx.x * 64 + lane] = all;
#pragma unroll 8
    for (int i = beg; i < end; ++i) {
        const uint32_t c = col[(size_t)i * ND];
        col[(size_t)i * ND] = run;
        run += c;
    }
}

// FUSED: hist holds counts, summed here over the tiles before this one and
// over all; else hist holds prefixes and totals the digit totals (rs_scan)
template <int DB, int TH, int IPT, bool FUSED>
__global__ __launch_bounds__(TH) void rs_scatter(const uint32_t* __restrict__ kin,
                                                         const uint32_t* __restrict__ vin,
                                                         uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                         int n, int shift, const uint32_t* __restrict__ hist,
                                                         int ntiles, const uint32_t* __restrict__ totals) {
    constexpr int ND = 1 << DB, DPT = rs_dpt<DB, TH>, TILE = TH * IPT;
    __shared__ RsTile<DB, TH, IPT> T;
    __shared__ uint32_t dst[ND];  // where a digit's run goes, minus its start in the tile
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int tile0 = blockIdx.x * TILE, cnt = min(TILE, n - tile0);
    uint32_t key[IPT], val[IPT], dcnt[DPT];
#pragma unroll
    for (int r = 0; r < IPT; ++r) {
        const int idx = tile0 + (w * IPT + r) * 64 + lane;
        key[r] = idx < n ? kin[idx] : 0u;
        val[r] = idx < n ? (vin ? vin[idx] : (uint32_t)idx) : 0u;
    }
    // this thread's digits: keys in tiles before this one, keys in all
    uint32_t pre[DPT], all[DPT], own = 0;
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
        const int d = t * DPT + q;
        pre[q] = all[q] = 0;
        if (d < ND) {
            if constexpr (FUSED) {
#pragma unroll 8
                for (int i = 0; i < ntiles; ++i) {
                    const uint32_t c = hist[(size_t)i * ND + d];
                    pre[q] += i < (int)blockIdx.x ? c : 0u;
                    all[q] += c;
                }
            } else {
                pre[q] = hist[(size_t)blockIdx.x * ND + d];
                all[q] = totals[d];
            }
        }
        own += all[q];
    }
    uint32_t base = rs_block_scan<TH / 64>(own, T.part, lane, w);
    rs_place<DB, TH, IPT>(T, key, val, cnt, shift, dcnt);  // synchronises before it uses part
#pragma unroll
    for (int q = 0; q < DPT; ++q) {
        const int d = t * DPT + q;
        if (d < ND) dst[d] = base + pre[q] - T.start[d];
        base += all[q];
    }
    __syncthreads();
    for (int q = t; q < cnt; q += TH) {
        const uint32_t k = T.skey[q];
        const uint32_t at = dst[(k >> shift) & (ND - 1)] + (uint32_t)q;
        kout[at] = k;
        vout[at] = T.sval[q];
    }
}

template <int DB, int TH, int IPT>
static void rs_tiles(const uint32_t* keys, const uint32_t* vals, uint32_t* keys_out, uint32_t* vals_out, int n,
                     int passes, void* temp, hipStream_t st) {
    constexpr int ND = 1 << DB;
    const int ntiles = (n + TH * IPT - 1) / (TH * IPT);
    const dim3 g(ntiles), b(TH);
    uint32_t* hist = (uint32_t*)temp;
    uint32_t* totals = hist + (size_t)ND * ntiles;
    uint32_t* kbuf = totals + ND;
    uint32_t* vbuf = kbuf + n;
    const uint32_t* kin = keys;
    const uint32_t* vin = vals;
    for (int p = 0; p < passes; ++p) {
        // passes alternate between (kbuf, vbuf) and (keys_out, vals_out), the last writes the latter
        const bool to_out = ((passes - 1 - p) % 2) == 0;
        uint32_t* ko = to_out ? keys_out : kbuf;
        uint32_t* vo = to_out ? vals_out : vbuf;
        hipLaunchKernelGGL((rs_hist<DB, TH, IPT>), g, b, 0, st, kin, n, DB * p, hist);
        if (ntiles <= RS_FUSED_TILES) {
            hipLaunchKernelGGL((rs_scatter<DB, TH, IPT, true>), g, b, 0, st, kin, vin, ko, vo, n, DB * p, hist, ntiles, totals);
        } else {
            hipLaunchKernelGGL(rs_scan<DB>, dim3(ND / 64), dim3(64 * RS_SCAN_WAVES), 0, st, hist, ntiles, totals);
            hipLaunchKernelGGL((rs_scatter<DB, TH, IPT, false>), g, b, 0, st, kin, vin, ko, vo, n, DB * p, hist, ntiles, totals);
        }
        kin = ko;
        vin = vo;
    }
}

// One workgroup sorts 3,080 keys in 16 us and 8,192 in 28 (30 bits); tiles take
// 27 and 29 at 8,193 and 19,209 keys, and one tile's ranking is then most of a
// pass.  Tiles of 2,048 keys as long as they are no more than the CUs, which
// then hold one each; twice that beyond (1,048,576 keys: 62 us, 69 with 2,048;
// 524,288 keys: 53 and 49).  Three passes of 10 bits beat four of 8 at every
// size (1,132,556 keys: 74 us against 91); three of 11 bits scatter in runs of
// two keys and lose to four of 8 for full 32-bit keys (104 against 88).
// Sums of up to 32 tiles' counts by the scatter cost less than a launch.
// With four passes, 256-thread tiles and a scan launch in each pass the sort
// took 44 us at 3,080 keys, 49 at 80,648 (now 40), 92 at 1,132,556 (now 74).
template <int DB>
static void rs_sort(const uint32_t* keys, const uint32_t* vals, uint32_t* keys_out, uint32_t* vals_out, int n,
                    int bits, void* temp, hipStream_t st) {
    const int passes = (bits + DB - 1) / DB;
    const dim3 one(1), b(RS_ONE_THREADS);
    if (n <= RS_ONE_THREADS * 4)
        hipLaunchKernelGGL((rs_one<DB, RS_ONE_THREADS, 4>), one, b, 0, st, keys, vals, keys_out, vals_out, n, passes);
    else if (n <= RS_ONE_THREADS * 8)
        hipLaunchKernelGGL((rs_one<DB, RS_ONE_THREADS, 8>), one, b, 0, st, keys, vals, keys_out, vals_out, n, passes);
    else if (n <= 256 * RS_THREADS * RS_IPT_MIN)
        rs_tiles<DB, RS_THREADS, RS_IPT_MIN>(keys, vals, keys_out, vals_out, n, passes, temp, st);
    else
        rs_tiles<DB, RS_THREADS, 2 * RS_IPT_MIN>(keys, vals, keys_out, vals_out, n, passes, temp, st);
}

// Sorts keys[0..n) with values; vals == nullptr means values = index.  The
// result lands in keys_out / vals_out.  `bits` = number of key bits in use.
hipError_t radix_sort(const uint32_t* keys, const uint32_t* vals, uint32_t* keys_out, uint32_t* vals_out, int n,
                      int bits, void* temp, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    if ((bits + 9) / 10 < (bits + 7) / 8) rs_sort<10>(keys, vals, keys_out, vals_out, n, bits, temp, st);
    else rs_sort<8>(keys, vals, keys_out, vals_out, n, bits, temp, st);
    return hipGetLastError();
}

}  // namespace upf
