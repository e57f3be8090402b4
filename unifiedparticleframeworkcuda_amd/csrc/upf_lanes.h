// upf_lanes.h -- pair sums with several lanes per particle.
//
// Each lane of a particle's group of LANES takes every LANES-th neighbour of
// its list row; the lanes' terms are then added in list order (DPP broadcasts,
// one addition per neighbour, the same on every lane of the group), so a sum
// has the bits of one lane's loop over the list while its gathers and terms run
// side by side.  A lane without a neighbour gives a term that leaves any sum as
// it is: +0 to be subtracted, -0 to be added.
#ifndef UPF_LANES_H_
#define UPF_LANES_H_

#include <hip/hip_runtime.h>

#include <cstdint>

#include "upf_device.h"

namespace upf {

// v of lane U of this lane's group of LANES (4: the quad, 16: the DPP row)
template <int LANES, int U>
__device__ __forceinline__ float lane_of(float v) {
    static_assert(LANES == 4 || LANES == 16, "a quad or a row");
    constexpr int ctrl = LANES == 4 ? U * 0x55 : 0x150 + U;  // quad_perm [U U U U] : row_newbcast U
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true));
}
// acc -/+ the group's terms, lane 0's first
template <int LANES, int U = 0>
__device__ __forceinline__ float sub_terms(float acc, float t) {
    if constexpr (U < LANES) return sub_terms<LANES, U + 1>(acc - lane_of<LANES, U>(t), t);
    else return acc;
}
template <int LANES, int U = 0>
__device__ __forceinline__ float add_terms(float acc, float t) {
    if constexpr (U < LANES) return add_terms<LANES, U + 1>(acc + lane_of<LANES, U>(t), t);
    else return acc;
}

// acc - t - u per lane of the group, lane 0's first
template <int LANES, int U = 0>
__device__ __forceinline__ float sub_terms2(float acc, float t, float u) {
    if constexpr (U < LANES)
        return sub_terms2<LANES, U + 1>((acc - lane_of<LANES, U>(t)) - lane_of<LANES, U>(u), t, u);
    else return acc;
}

// Entry k of the list row (0 past its end).
__device__ __forceinline__ uint32_t entry_at(const uint32_t* __restrict__ row, int cnt, int k) {
    return k < cnt ? row[k] : 0u;
}

// A list's length and this lane's first two entries, which do not wait for the
// length: rows of ld words are there whole, and for_pairs ignores what lies past
// the list's end.  Loaded with the particle's own records, so that the first
// gathers come one trip to memory after a pass starts, not three or four.
struct RowHead {
    int cnt;
    uint32_t e, f;
};
template <int LANES>
__device__ __forceinline__ RowHead row_head(const uint32_t* __restrict__ row, int ld, const int* __restrict__ cnt, int sub) {
    return RowHead{*cnt, row[min(sub, ld - 1)], row[min(sub + LANES, ld - 1)]};
}
// Values that are to be on their way together: the compiler moves no load of
// theirs past this, where the first use of any of them waits.
__device__ __forceinline__ void together(int& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void together(uint32_t& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void together(float& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void together(float4& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }
__device__ __forceinline__ void together(RowHead& v) { asm volatile("" : "+v"(v.cnt), "+v"(v.e), "+v"(v.f)); }
template <class T, class... More>
__device__ __forceinline__ void together(T& v, More&... more) {
    together(v);
    together(more...);
}

// Walks this lane's entries of the list row: load(entry) for the lane's next
// two, then for each term(record, whether the lane has that entry) and, per
// LANES neighbours, add(the lane's term).  An entry past the list's end reads
// slot 0's records, for a term that changes no sum.  The next entries are
// loaded ahead of the gathers of this round.
template <int LANES, class Load, class Term, class Add>
__device__ __forceinline__ void for_pairs(const uint32_t* __restrict__ row, const RowHead& head, int sub, Load load,
                                          Term term, Add add) {
    const int cnt = head.cnt;
    uint32_t e = sub < cnt ? head.e : 0u, f = sub + LANES < cnt ? head.f : 0u;
    for (int k = sub; k - sub < cnt; k += 2 * LANES) {
        const auto r = load(e);
        const auto s = load(f);
        e = entry_at(row, cnt, k + 2 * LANES);
        f = entry_at(row, cnt, k + 3 * LANES);
        add(term(r, k < cnt));
        if (k - sub + LANES < cnt) add(term(s, k + LANES < cnt));
    }
}

// three sums' terms, and their subtraction or addition
struct Term3 {
    float x, y, z;
};
template <int LANES>
__device__ __forceinline__ void sub_terms(float& x, float& y, float& z, const Term3& t) {
    x = sub_terms<LANES>(x, t.x);
    y = sub_terms<LANES>(y, t.y);
    z = sub_terms<LANES>(z, t.z);
}
template <int LANES>
__device__ __forceinline__ void add_terms(float& x, float& y, float& z, const Term3& t) {
    x = add_terms<LANES>(x, t.x);
    y = add_terms<LANES>(y, t.y);
    z = add_terms<LANES>(z, t.z);
}
// two 16-byte records of a neighbour
struct Pair4 {
    float4 a, b;
};

// Visits the candidates of the query box of (x, y, z) (the reference's BoxQuery)
// in ascending slot order with BOX_LANES lanes (lane sub of them): per round,
// load(slot) and then test(whether the lane has a candidate, slot, record).
// Each lane finds cells of its own, their slots go to a candidate table in LDS
// (tab, BOX_CAND entries per group), and four rounds' records are loaded
// together.  BOX_CAND slots hold any query box of a fluid; a denser one is
// walked cell by cell.
constexpr int BOX_LANES = 16;
constexpr int BOX_CAND = 384;
template <class Load, class Test>
__device__ __forceinline__ void for_each_in_box(float x, float y, float z, float h, const float* scales,
                                                uint32_t block_shift, uint32_t grid_dim,
                                                const uint2* __restrict__ cells, int sub, uint32_t* tab, Load load,
                                                Test test) {
    using V = decltype(load(0u));
    // This lane's cells: numbers sub, sub + 16, ... of the 3x3x3 stencil around
    // (x, y, z) in Morton order.  Of an axis' three coordinates two share all but
    // the lowest bit, the third differs from them first at bit key of the cell code;
    // the numbers count through three high bits, the axes' keys in order, then the
    // lowest bits.  The box reaches at most one cell either way (a cell is wider
    // than h).
    bool in_grid;
    const uint32_t c = dkey(x, y, z, scales, in_grid) >> (3u * block_shift);
    uint32_t key[3], v0[3], v1[3];  // the axis' part of the code for a high bit of 0 / 1
    bool ok0[3], ok1[3];
    const float xv[3] = {x, y, z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const uint32_t ma = 0x09249249u << a, ca = c & ma;
        const bool odd = (c >> a) & 1u, lb = (sub >> a) & 1;
        const uint32_t dn = (ca - 1u) & ma, up = ((ca | ~ma) + 1u) & ma, third = odd ? up : ca;
        key[a] = third ? (uint32_t)__ffs((int)third) : 33u + a;
        v0[a] = lb && odd ? ca : dn;
        v1[a] = lb || odd ? up : ca;
        // BoxQuery along the axis
        bool in;
        const uint32_t own = dgrid(scales[a] * xv[a], in) >> block_shift;
        const float lo_f = scales[a] * (xv[a] - h), hi_f = scales[a] * (xv[a] + h);
        const uint32_t l = ((uint32_t)(unsigned short)(lo_f >= 0.0f ? lo_f : 0.0f)) >> block_shift;
        const uint32_t u = ((uint32_t)(unsigned short)(hi_f <= 1024.0f ? hi_f : 1024.0f)) >> block_shift;
        const bool below = l < own, above = u > own && own + 1 < grid_dim;
        ok0[a] = odd ? lb || below : !lb && below;
        ok1[a] = odd ? !lb && above : !lb || above;
    }
    uint2 r[4];
    uint32_t before[4];  // candidates of the box in earlier cells
    uint32_t total = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t code = 0;
        bool ok = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int b = (a + 1) % 3, d = (a + 2) % 3;
            const int sh = (key[b] < key[a] ? 1 : 0) + (key[d] < key[a] ? 1 : 0);  // the axis' high bit
            const bool hb = sh == 0 ? (sub >> 3) & 1 : (sh == 1 ? q & 1 : q >> 1);
            code |= hb ? v1[a] : v0[a];
            ok = ok && (hb ? ok1[a] : ok0[a]);
        }
        r[q] = make_uint2(0u, 0u);
        if (ok) r[q] = cells[code];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t incl = r[q].y - r[q].x;
#pragma unroll
        for (int o = 1; o < BOX_LANES; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, o, BOX_LANES);
            if (sub >= o) incl += y;
        }
        before[q] = total + incl - (r[q].y - r[q].x);
        total += (uint32_t)__shfl((int)incl, BOX_LANES - 1, BOX_LANES);
    }
    if (total <= BOX_CAND) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            for (uint32_t s = r[q].x; s < r[q].y; ++s) tab[before[q] + (s - r[q].x)] = s;
        // the group's lanes are in one wave: its LDS writes are in order before its reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (uint32_t t = (uint32_t)sub; t - (uint32_t)sub < total; t += 4 * BOX_LANES) {
            uint32_t s[4];
            V v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                s[q] = tab[min(t + q * BOX_LANES, total - 1u)];
                v[q] = load(s[q]);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) test(t + q * BOX_LANES < total, s[q], v[q]);
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            for (int u = 0; u < BOX_LANES; ++u) {
                const uint32_t s0 = (uint32_t)__shfl((int)r[q].x, u, BOX_LANES);
                const uint32_t s1 = (uint32_t)__shfl((int)r[q].y, u, BOX_LANES);
                for (uint32_t t = s0; t < s1; t += BOX_LANES) {
                    const uint32_t s = min(t + (uint32_t)sub, s1 - 1u);
                    test(t + sub < s1, s, load(s));
                }
            }
    }
}

}  // namespace upf

#endif
