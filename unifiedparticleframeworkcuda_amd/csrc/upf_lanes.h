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

// Walks this lane's entries of the list row: load(entry) for the lane's next
// two, then for each term(record, whether the lane has that entry) and, per
// LANES neighbours, add(the lane's term).  An entry past the list's end reads
// slot 0's records, for a term that changes no sum.  The next entries are
// loaded ahead of the gathers of this round.  e: entry_at().
template <int LANES, class Load, class Term, class Add>
__device__ __forceinline__ void for_pairs(const uint32_t* __restrict__ row, int cnt, int sub, uint32_t e, Load load,
                                          Term term, Add add) {
    uint32_t f = entry_at(row, cnt, sub + LANES);
    for (int k = sub; k - sub < cnt; k += 2 * LANES) {
        const auto r = load(e);
        const auto s = load(f);
        e = entry_at(row, cnt, k + 2 * LANES);
        f = entry_at(row, cnt, k + 3 * LANES);
        add(term(r, k < cnt));
        if (k - sub + LANES < cnt) add(term(s, k + LANES < cnt));
    }
}
template <int LANES, class Load, class Term, class Add>
__device__ __forceinline__ void for_pairs(const uint32_t* __restrict__ row, int cnt, int sub, Load load, Term term,
                                          Add add) {
    for_pairs<LANES>(row, cnt, sub, entry_at(row, cnt, sub), load, term, add);
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

}  // namespace upf

#endif
