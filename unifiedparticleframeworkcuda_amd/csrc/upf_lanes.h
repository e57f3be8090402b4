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

// This lane's first entry of the list row (0 past its end).
__device__ __forceinline__ uint32_t first_entry(const uint32_t* __restrict__ row, int cnt, int sub) {
    return sub < cnt ? row[sub] : 0u;
}

// term(entry) for this lane's entries of the list (none(): it has no entry in
// this round), then add() for the group's LANES terms; the next round's entry
// is loaded ahead of this round's gathers.  e: first_entry().
template <int LANES, class Term, class None, class Add>
__device__ __forceinline__ void for_pairs(const uint32_t* __restrict__ row, int cnt, int sub, uint32_t e, Term term,
                                          None none, Add add) {
    for (int k = 0; k < cnt; k += LANES) {
        const int next = k + LANES + sub;
        const uint32_t en = next < cnt ? row[next] : 0u;
        if (k + sub < cnt) term(e);
        else none();
        add();
        e = en;
    }
}
template <int LANES, class Term, class None, class Add>
__device__ __forceinline__ void for_pairs(const uint32_t* __restrict__ row, int cnt, int sub, Term term, None none,
                                          Add add) {
    for_pairs<LANES>(row, cnt, sub, first_entry(row, cnt, sub), term, none, add);
}

}  // namespace upf

#endif
