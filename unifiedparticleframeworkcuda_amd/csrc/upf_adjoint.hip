// upf_adjoint.hip -- differentiable PCISPH rollout and its adjoint on gfx950.
//
// The step is the static-boundary PCISPH step (CpuParticlePhysicsStaticBoundariesPCISPH,
// src/cpu/UnifiedPhysics.cpp:4220-4238, CPU boundary mode) with a fixed number
// of correction iterations and the kernels in closed form (KernelM4
// src/cpu/WeightingKernel.cpp:75-97, kernelPressureGrad :165-180,
// kernelViscosityLaplacian :190-200) rather than through the 300-entry tables,
// whose step values have no useful derivative:
//   F_i   = -sum_j (v_i - v_j) V0^2 mu L(r_ij) - m g e_y + B(x_i)  (fluid j)
//   with B the wall penalty force (CalculateBoundaryForcePerLiquidParticleHost,
//   src/cpu/UnifiedPhysics.cpp:2032-2069), k_b = 2 F_max / d_f per unit depth
//   within d_f of a face of the collision box;
//   iteration k (Fp = 0 before the first):
//     v*_i = v_i + (F_i + Fp_i) dt/m;  z_i = x_i + v*_i dt;  x*_i = clamp(z_i)
//     rho_i = m W(0) + sum_j [r*_ij < h] m W(r*_ij)
//     p_i  += delta sp(rho_i - rho0),  sp(s) = tau log(1 + exp(s / tau))
//     Fp_i  = -(m^2/rho0^2) sum_j (p_i + p_j) G(r_ij) (x_i - x_j)   (p_wall = 0)
//   v'_i = v_i + (F_i + Fp_i) dt/m;  y_i = x_i + v'_i dt;  x'_i = clamp(y_i).
// sp with tau = 1 kg/m^3 (0.1 % of rho0) is a smooth form of the CPU path's
// max(s, 0) (:5477-5478): a settling fluid keeps many particles at the kink,
// where rounding alone decides the branch and FP32 and FP64 gradients of a
// 64-step rollout differ by O(1).
// The CPU path's velocity reflection at the box (:4000-4044) jumps when a
// particle crosses a face; here the position clamp stays, the reflection is
// dropped and the penalty force pushes particles back, so that the rollout is
// a continuous function of its inputs.
// Particles keep their upload order; each step sorts z-index keys only to
// build the cell table and neighbour lists (ascending sorted order, so every
// sum runs in the order of the CPU restatement).
//
// The backward pass is the exact reverse of these passes with the neighbour
// sets held fixed, in gather form over the symmetric lists (no atomics):
//   dL/dp_i  += -(m^2/rho0^2) sum_j G (x_ij . (gFp_i - gFp_j))
//   dL/dx_i  += -(m^2/rho0^2) sum_j (p_i + p_j) H(x_ij) (gFp_i - gFp_j),
//               H(d) = G I + (G'/r) d d^T
//   dL/drho_i = delta sp'(rho_i - rho0) dL/dp_i
//   dL/dx*_i  = sum_j m W'(r*)/r* x*_ij (dL/drho_i + dL/drho_j)
// and the elementwise reverses of the prediction, the clamps and the
// integration.  Memory: the state every `ckpt` steps is kept; the backward
// pass recomputes one segment at a time, keeping its steps' lists and
// iteration states, then runs the segment in reverse.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "upf.h"
#include "upf_bins.h"
#include "upf_device.h"
#include "upf_internal.h"
#include "upf_kernels.h"
#include "upf_lanes.h"
#include "upf_sort.h"

namespace upf {
namespace ad {

constexpr int AB = 256;  // threads per block

// Pair passes run LANES lanes per particle (upf_lanes.h).  One lane per particle
// was one serial chain of gathers per wave and about one wave per SIMD at
// 65,536 particles (density 16.7 us, pressure force 15.6, their reverses 27 and
// 29; 8.9, 8.7, 10 and 14 now); see lanes() for the choice.

struct Kern {  // closed-form kernels and their radial derivatives, FP32
    float h, a, ah, cs, cv;
    explicit Kern(float sr) : h(sr) {
        a = 2.546479089470325472f / (sr * sr * sr);  // 8 / (pi h^3)
        ah = a / h;
        cs = -45.0f / (3.1415926535897932384626f * sr * sr * sr * sr * sr * sr);
        cv = 45.0f / (3.1415926535897932384626f * sr * sr * sr * sr * sr * sr);
    }
    __device__ float W(float r) const {
        if (!(r < h)) return 0.0f;
        const float s = r / h;
        if (s < 0.5f) return a * (1.0f - 6.0f * s * s + 6.0f * s * s * s);
        const float t = 1.0f - s;
        return a * (2.0f * t * t * t);
    }
    __device__ float dW(float r) const {
        if (!(r < h)) return 0.0f;
        const float s = r / h;
        if (s < 0.5f) return ah * (-12.0f * s + 18.0f * s * s);
        const float t = 1.0f - s;
        return ah * (-6.0f * t * t);
    }
    __device__ float G(float r) const {
        if (!(r < h) || r == 0.0f) return 0.0f;
        const float t = h - r;
        return cs * t * t / r;
    }
    __device__ float dG(float r) const {
        if (!(r < h) || r == 0.0f) return 0.0f;
        const float t = h - r;
        return cs * (-2.0f * t / r - t * t / (r * r));
    }
    __device__ float L(float r) const { return r < h ? cv * (h - r) : 0.0f; }
    __device__ float dL(float r) const { return r < h ? -cv : 0.0f; }
};

constexpr float kTau = 1.0f;  // width of the smooth pressure clamp, kg/m^3

__device__ inline float softplus(float s) {
    const float sx = s / kTau;
    return sx > 30.0f ? s : kTau * log1pf(expf(sx));
}
__device__ inline float softplus_grad(float s) { return 1.0f / (1.0f + expf(-s / kTau)); }

struct Consts {
    Kern kn;
    float m, rho0, dt, q, cvis, cp, delta, g;
    float fd, kb;  // wall penalty: depth and stiffness 2 F_max / d_f
    float cmin[3], cmax[3];
    explicit Consts(float sr) : kn(sr) {}
};

// wall penalty force on a liquid particle at (x, y, z) and its diagonal derivative
__device__ inline void wall_force(const Consts& C, float x, float y, float z, float* f, float* g) {
    const float c[3] = {x, y, z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        f[a] = 0.0f;
        g[a] = 0.0f;
        if (c[a] < C.cmin[a] + C.fd) { f[a] = f[a] + (C.cmin[a] + C.fd - c[a]) * C.kb; g[a] = g[a] - C.kb; }
        if (c[a] > C.cmax[a] - C.fd) { f[a] = f[a] - (c[a] + C.fd - C.cmax[a]) * C.kb; g[a] = g[a] - C.kb; }
    }
}

__device__ inline bool is_fluid(const float4& x) { return __float_as_int(x.w) == UPF_LIQUID; }
__device__ inline float len3(float dx, float dy, float dz) { return sqrtf(dx * dx + dy * dy + dz * dz); }
__device__ inline float dot3(const float4& a, const float4& b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline float ax(const float4& v, int a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }

// ---------------------------------------------------------- neighbour search
__device__ inline void put_key(const upf_params& P, float x, float y, float z, uint32_t* key, Ctl* ctl) {
    bool ok;
    *key = dkey(x, y, z, P.scales, ok);
    if (!ok) atomicOr(&ctl->err, 1u << UPF_ERR_RANGE);
}

__global__ void k_keys(int n, const float4* __restrict__ x, upf_params P, uint32_t* __restrict__ keys, Ctl* ctl) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 p = x[i];
    put_key(P, p.x, p.y, p.z, keys + i, ctl);
}

__global__ void k_clear_cells(uint2* __restrict__ cells, uint32_t nc) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < nc) cells[c] = make_uint2(0u, 0u);
}

// the cell table, and the positions in sorted order with their particle in w:
// the lists read a cell's candidates as one run
__global__ void k_cell_bounds(int n, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ perm,
                              const float4* __restrict__ x, uint32_t shift3, uint2* __restrict__ cells,
                              float4* __restrict__ cand) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t c = keys[i] >> shift3;
    if (i == 0 || (keys[i - 1] >> shift3) != c) cells[c].x = (uint32_t)i;
    if (i == n - 1 || (keys[i + 1] >> shift3) != c) cells[c].y = (uint32_t)(i + 1);
    const uint32_t j = perm[i];
    const float4 p = x[j];
    cand[i] = make_float4(p.x, p.y, p.z, __uint_as_float(j));
}

// the same positions from the particles' places cell by cell (upf_bins.h)
__global__ __launch_bounds__(AB, 8) void k_rank_cand(int n, CellMap map, const uint64_t* __restrict__ place,
                                                  const uint2* __restrict__ cells, const float4* __restrict__ x,
                                                  float4* __restrict__ cand, Ctl* ctl) {
    static_assert(AB == BLOCK, "move_ranked");
    move_ranked(n, map, place, cells, &ctl->crowded, [&](uint64_t v, auto slot) __attribute__((always_inline)) {
        const uint32_t j = (uint32_t)v;
        const float4 p = x[j];
        cand[slot()] = make_float4(p.x, p.y, p.z, __uint_as_float(j));
    });
}

// neighbour ids of every fluid particle: the cells of its query box (the
// reference's BoxQuery) in Morton order, candidates in sorted order, r < h.
// Sixteen lanes per particle test sixteen candidates at a time, the passing ones
// appended in order through the group's ballot.  Bound by the latency of table
// and candidate reads (267 us at 80,648 particles with one lane walking the cells
// of each, 37 with BoxCells' enumeration per lane, now 32).
constexpr int LIST_LANES = BOX_LANES;
__global__ __launch_bounds__(AB) void k_lists(int n, const float4* __restrict__ x, const float4* __restrict__ cand,
                                              const uint2* __restrict__ cells, upf_params P,
                                              uint32_t* __restrict__ nb, int* __restrict__ cnt, Ctl* ctl) {
    __shared__ uint32_t table[AB / LIST_LANES][BOX_CAND];
    const int i = (int)((blockIdx.x * AB + threadIdx.x) / LIST_LANES);
    const int sub = threadIdx.x % LIST_LANES;
    if (i >= n) return;
    const float4 xi = x[i];
    if (!is_fluid(xi)) {
        if (sub == 0) cnt[i] = 0;
        return;
    }
    const float h = P.support_radius, hh = h * h;
    const int cap = P.max_neighbors;
    uint32_t* row = nb + (size_t)i * cap;
    const int shift = (threadIdx.x & 63) & ~(LIST_LANES - 1);  // the group's bits of the wave's ballot
    int c = 0;
    // tests one candidate per lane (if any) and appends the passing ones
    auto test = [&](bool have, uint32_t, const float4& xj) __attribute__((always_inline)) {
        const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
        const uint32_t j = __float_as_uint(xj.w);
        const bool pass = have && j != (uint32_t)i && dx * dx + dy * dy + dz * dz < hh;
        const uint32_t m = (uint32_t)(__ballot(pass) >> shift) & 0xFFFFu;
        const int at = c + __popc(m & ((1u << sub) - 1u));
        if (pass && at < cap) row[at] = j;
        c += __popc(m);
    };
    for_each_in_box(xi.x, xi.y, xi.z, h, P.scales, P.block_shift, P.grid_dim, cells, sub,
                    table[threadIdx.x / LIST_LANES], [&](uint32_t s) { return cand[s]; }, test);
    if (sub == 0) {
        cnt[i] = c < cap ? c : cap;
        if (c > cap) atomicOr(&ctl->err, 1u << UPF_ERR_NBR_OVERFLOW);
    }
}

// --------------------------------------------------------------- forward
__device__ inline float clampc(float c, float mn, float mx) {
    if (c < mn) c = mn;
    if (c > mx) c = mx;
    return c;
}
__device__ inline bool outside(float c, int a, const Consts& C) { return c < C.cmin[a] || c > C.cmax[a]; }

// type bits of a predicted or new position, with the axes that the clamp moved
// above them (the reverse passes' derivative of the clamp)
constexpr int OUT_SHIFT = 8;
__device__ inline float type_and_out(float tw, float x, float y, float z, const Consts& C) {
    const int out = (outside(x, 0, C) ? 1 : 0) | (outside(y, 1, C) ? 2 : 0) | (outside(z, 2, C) ? 4 : 0);
    return __int_as_float(__float_as_int(tw) | out << OUT_SHIFT);
}
__device__ inline bool moved(float w, int a) { return (__float_as_int(w) >> (OUT_SHIFT + a)) & 1; }
__device__ inline bool is_fluid_w(float w) { return (__float_as_int(w) & ((1 << OUT_SHIFT) - 1)) == UPF_LIQUID; }

// prediction of an iteration: x* = clamp(z)
__device__ inline float4 predict(const float4& xi, const float4& vi, float fx, float fy, float fz, const float4& f,
                                 const Consts& C, Ctl* ctl) {
    const float vx = vi.x + (f.x + fx) * C.q, vy = vi.y + (f.y + fy) * C.q, vz = vi.z + (f.z + fz) * C.q;
    const float zx = xi.x + vx * C.dt, zy = xi.y + vy * C.dt, zz = xi.z + vz * C.dt;
    if (!(zx == zx) || !(zy == zy) || !(zz == zz)) atomicOr(&ctl->err, 1u << UPF_ERR_NAN);
    return make_float4(clampc(zx, C.cmin[0], C.cmax[0]), clampc(zy, C.cmin[1], C.cmax[1]),
                       clampc(zz, C.cmin[2], C.cmax[2]), type_and_out(xi.w, zx, zy, zz, C));
}

// external force, and the first iteration's prediction.  Clears nc cells of the
// table for the next step: the lists of this one are built.
template <int LANES>
__global__ __launch_bounds__(AB) void k_ext(int n, const float4* __restrict__ x, const float4* __restrict__ v,
                                            const uint32_t* __restrict__ nb, const int* __restrict__ cnt, int ld,
                                            Consts C, float4* __restrict__ F, float* __restrict__ p,
                                            float4* __restrict__ xs, uint2* __restrict__ cells, uint32_t nc, Ctl* ctl) {
    const unsigned id = blockIdx.x * AB + threadIdx.x;
    for (uint32_t c = id; c < nc; c += gridDim.x * AB) cells[c] = make_uint2(0u, 0u);
    const int i = (int)(id / LANES), sub = (int)(id % LANES);
    if (i >= n) return;
    float4 xi = x[i], vi = v[i];
    const uint32_t* row = nb + (size_t)i * ld;
    RowHead head = row_head<LANES>(row, ld, cnt + i, sub);
    together(xi, vi, head);
    if (!is_fluid(xi)) {
        if (sub == 0) {
            F[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            p[i] = 0.0f;
            xs[i] = xi;
        }
        return;
    }
    float fx = 0.0f, fy = 0.0f, fz = 0.0f;
    for_pairs<LANES>(
        row, head, sub, [&](uint32_t j) { return Pair4{x[j], v[j]}; },
        [&](const Pair4& q, bool have) {
            if (!have || !is_fluid(q.a)) return Term3{0.0f, 0.0f, 0.0f};
            const float r = len3(xi.x - q.a.x, xi.y - q.a.y, xi.z - q.a.z);
            const float s = C.cvis * C.kn.L(r);
            return Term3{(vi.x - q.b.x) * s, (vi.y - q.b.y) * s, (vi.z - q.b.z) * s};
        },
        [&](const Term3& t) { sub_terms<LANES>(fx, fy, fz, t); });
    if (sub != 0) return;
    fy = fy - C.m * C.g;
    float wf[3], wg[3];
    wall_force(C, xi.x, xi.y, xi.z, wf, wg);
    const float4 f = make_float4(fx + wf[0], fy + wf[1], fz + wf[2], 0.0f);
    F[i] = f;
    p[i] = 0.0f;
    xs[i] = predict(xi, vi, 0.0f, 0.0f, 0.0f, f, C, ctl);
}

// density and pressure of an iteration; rec: position and pressure, the
// pressure force's one gather per neighbour
template <int LANES>
__global__ __launch_bounds__(AB) void k_density(int n, const float4* __restrict__ x, const float4* __restrict__ xs,
                                                const uint32_t* __restrict__ nb, const int* __restrict__ cnt, int ld,
                                                Consts C, float* __restrict__ p, float4* __restrict__ rec,
                                                float* __restrict__ p_tape, float* __restrict__ rho_tape) {
    const unsigned id = blockIdx.x * AB + threadIdx.x;
    const int i = (int)(id / LANES), sub = (int)(id % LANES);
    if (i >= n) return;
    float4 xi = xs[i];
    const uint32_t* row = nb + (size_t)i * ld;
    RowHead head = row_head<LANES>(row, ld, cnt + i, sub);
    together(xi, head);
    float rho = 0.0f, pi = 0.0f;
    if (is_fluid_w(xi.w)) {
        rho = C.m * C.kn.W(0.0f);
        for_pairs<LANES>(
            row, head, sub, [&](uint32_t j) { return xs[j]; },
            [&](const float4& xj, bool have) {
                return have ? C.m * C.kn.W(len3(xi.x - xj.x, xi.y - xj.y, xi.z - xj.z)) : -0.0f;
            },
            [&](float t) { rho = add_terms<LANES>(rho, t); });
        pi = p[i] + C.delta * softplus(rho - C.rho0);
    }
    if (sub != 0) return;
    const float4 xc = x[i];
    rec[i] = make_float4(xc.x, xc.y, xc.z, pi);
    p[i] = pi;
    if (p_tape) { p_tape[i] = pi; rho_tape[i] = rho; }
}

// pressure force of an iteration, then the next iteration's prediction (LAST:
// the integration, and the new positions' keys for the next step's sort)
template <int LANES, bool LAST>
__global__ __launch_bounds__(AB) void k_pforce(int n, const float4* __restrict__ x, const float4* __restrict__ v,
                                               const uint32_t* __restrict__ nb, const int* __restrict__ cnt, int ld,
                                               Consts C, const float4* __restrict__ rec, const float4* __restrict__ F,
                                               float4* __restrict__ xs, float4* __restrict__ x_new,
                                               float4* __restrict__ v_new, float* __restrict__ y_tape, upf_params P,
                                               uint32_t* __restrict__ keys, Ctl* ctl) {
    const unsigned id = blockIdx.x * AB + threadIdx.x;
    const int i = (int)(id / LANES), sub = (int)(id % LANES);
    if (i >= n) return;
    float4 xi = x[i];
    float pi = rec[i].w;
    const uint32_t* row = nb + (size_t)i * ld;
    RowHead head = row_head<LANES>(row, ld, cnt + i, sub);
    together(xi, pi, head);
    float4 xn = xi, vn;
    float yw = xi.w;
    if (!is_fluid(xi)) {
        if (sub != 0) return;
        if constexpr (!LAST) {
            xs[i] = xi;
            return;
        }
        vn = v[i];
    } else {
        float fx = 0.0f, fy = 0.0f, fz = 0.0f;
        for_pairs<LANES>(
            row, head, sub, [&](uint32_t j) { return rec[j]; },
            [&](const float4& xj, bool have) {
                const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
                const float s = C.kn.G(len3(dx, dy, dz)) * (pi + xj.w) * C.cp;
                return have ? Term3{dx * s, dy * s, dz * s} : Term3{0.0f, 0.0f, 0.0f};
            },
            [&](const Term3& t) { sub_terms<LANES>(fx, fy, fz, t); });
        if (sub != 0) return;
        const float4 vi = v[i], f = F[i];
        if constexpr (!LAST) {
            xs[i] = predict(xi, vi, fx, fy, fz, f, C, ctl);
            return;
        }
        const float v3[3] = {vi.x + (f.x + fx) * C.q, vi.y + (f.y + fy) * C.q, vi.z + (f.z + fz) * C.q};
        const float xo[3] = {xi.x, xi.y, xi.z};
        float y[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) y[a] = xo[a] + v3[a] * C.dt;
        yw = type_and_out(xi.w, y[0], y[1], y[2], C);
#pragma unroll
        for (int a = 0; a < 3; ++a) y[a] = clampc(y[a], C.cmin[a], C.cmax[a]);
        xn = make_float4(y[0], y[1], y[2], xi.w);
        vn = make_float4(v3[0], v3[1], v3[2], 0.0f);
    }
    x_new[i] = xn;
    v_new[i] = vn;
    if (y_tape) y_tape[i] = yw;
    if (keys) put_key(P, xn.x, xn.y, xn.z, keys + i, ctl);
}

// -------------------------------------------------------------- backward
// reverse of the integration: (gx, gv) = dL/d(x', v') -> nx, nv, gF, and gFp
// with the last iteration's pressure in w.  Both gFp buffers are zero for
// walls, which the pressure force's reverse reads as a neighbour's.
__global__ void kr_integrate(int n, const float* __restrict__ y, const float4* __restrict__ gx,
                             const float4* __restrict__ gv, Consts C, const float* __restrict__ p,
                             float4* __restrict__ nx, float4* __restrict__ nv, float4* __restrict__ gF,
                             float4* __restrict__ gFp, float4* __restrict__ gFp2, float* __restrict__ gp) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float yi = y[i];
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    gp[i] = 0.0f;
    if (!is_fluid_w(yi)) { nx[i] = z4; nv[i] = z4; gF[i] = z4; gFp[i] = z4; gFp2[i] = z4; return; }
    const float4 a = gx[i], b = gv[i];
    float gy[3], gvn[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        gy[k] = moved(yi, k) ? 0.0f : ax(a, k);
        gvn[k] = ax(b, k);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) gvn[k] = gvn[k] + gy[k] * C.dt;
    nx[i] = make_float4(gy[0], gy[1], gy[2], 0.0f);
    nv[i] = make_float4(gvn[0], gvn[1], gvn[2], 0.0f);
    const float4 f = make_float4(gvn[0] * C.q, gvn[1] * C.q, gvn[2] * C.q, 0.0f);
    gF[i] = f;
    gFp[i] = make_float4(f.x, f.y, f.z, p[i]);
}

// reverse of the pressure force of one iteration: dL/dp (running) and dL/dx,
// then dL/drho, which goes with the predicted position into rec, the density
// reverse's one gather per neighbour
template <int LANES>
__global__ __launch_bounds__(AB) void kr_pforce(int n, const float4* __restrict__ x, const uint32_t* __restrict__ nb,
                                                const int* __restrict__ cnt, int ld, Consts C,
                                                const float4* __restrict__ gFp, const float4* __restrict__ xs,
                                                const float* __restrict__ rho, float* __restrict__ gp,
                                                float4* __restrict__ nx, float4* __restrict__ rec) {
    const unsigned id = blockIdx.x * AB + threadIdx.x;
    const int i = (int)(id / LANES), sub = (int)(id % LANES);
    if (i >= n) return;
    float4 xi = x[i], xsi = xs[i], gi = gFp[i];
    const uint32_t* row = nb + (size_t)i * ld;
    RowHead head = row_head<LANES>(row, ld, cnt + i, sub);
    together(xi, xsi, gi, head);
    if (!is_fluid(xi)) {
        if (sub == 0) rec[i] = make_float4(xsi.x, xsi.y, xsi.z, 0.0f);
        return;
    }
    float acc = 0.0f, gxx = 0.0f, gxy = 0.0f, gxz = 0.0f;
    struct Terms {
        float a;
        Term3 g;
    };
    for_pairs<LANES>(
        row, head, sub, [&](uint32_t j) { return Pair4{x[j], gFp[j]}; },
        [&](const Pair4& q, bool have) {
            const float4 &xj = q.a, &gj = q.b;
            if (!have) return Terms{0.0f, {0.0f, 0.0f, 0.0f}};
            const float4 d = make_float4(xi.x - xj.x, xi.y - xj.y, xi.z - xj.z, 0.0f);
            const float r = len3(d.x, d.y, d.z);
            const float4 w = make_float4(gi.x - gj.x, gi.y - gj.y, gi.z - gj.z, 0.0f);
            const float G = C.kn.G(r);
            const float dw = dot3(d, w);
            const float pp = gi.w + gj.w;
            const float s = r > 0.0f ? C.kn.dG(r) / r * dw : 0.0f;
            const float t = C.cp * pp;
            return Terms{C.cp * G * dw, {(w.x * G + d.x * s) * t, (w.y * G + d.y * s) * t, (w.z * G + d.z * s) * t}};
        },
        [&](const Terms& t) {
            acc = sub_terms<LANES>(acc, t.a);
            sub_terms<LANES>(gxx, gxy, gxz, t.g);
        });
    if (sub != 0) return;
    const float g = gp[i] + acc;
    gp[i] = g;
    float4 o = nx[i];
    o.x = o.x + gxx; o.y = o.y + gxy; o.z = o.z + gxz;
    nx[i] = o;
    rec[i] = make_float4(xsi.x, xsi.y, xsi.z, C.delta * g * softplus_grad(rho[i] - C.rho0));
}

// reverse of density, pressure update and prediction of one iteration; p_prev:
// the pressures of the iteration before (null before the first)
template <int LANES>
__global__ __launch_bounds__(AB) void kr_density(int n, const float4* __restrict__ xs, const float4* __restrict__ rec,
                                                 const uint32_t* __restrict__ nb, const int* __restrict__ cnt, int ld,
                                                 Consts C, const float* __restrict__ p_prev, float4* __restrict__ nx,
                                                 float4* __restrict__ nv, float4* __restrict__ gF,
                                                 float4* __restrict__ gFp_prev) {
    const unsigned id = blockIdx.x * AB + threadIdx.x;
    const int i = (int)(id / LANES), sub = (int)(id % LANES);
    if (i >= n) return;
    float w = xs[i].w;
    float4 xi = rec[i];
    const uint32_t* row = nb + (size_t)i * ld;
    RowHead head = row_head<LANES>(row, ld, cnt + i, sub);
    together(w, xi, head);
    if (!is_fluid_w(w)) return;
    float gx = 0.0f, gy = 0.0f, gz = 0.0f;
    for_pairs<LANES>(
        row, head, sub, [&](uint32_t j) { return rec[j]; },
        [&](const float4& xj, bool have) {
            const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
            const float r = len3(dx, dy, dz);
            if (!have || !(r < C.kn.h) || r == 0.0f) return Term3{-0.0f, -0.0f, -0.0f};
            const float gr = xi.w + xj.w;
            const float s = C.m * C.kn.dW(r) / r * gr;
            return Term3{dx * s, dy * s, dz * s};
        },
        [&](const Term3& t) { add_terms<LANES>(gx, gy, gz, t); });
    if (sub != 0) return;
    const float g3[3] = {gx, gy, gz};
    float zb[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) zb[a] = moved(w, a) ? 0.0f : g3[a];
    float4 o = nx[i];
    o.x = o.x + zb[0]; o.y = o.y + zb[1]; o.z = o.z + zb[2];
    nx[i] = o;
    const float vs[3] = {zb[0] * C.dt, zb[1] * C.dt, zb[2] * C.dt};
    float4 ov = nv[i];
    ov.x = ov.x + vs[0]; ov.y = ov.y + vs[1]; ov.z = ov.z + vs[2];
    nv[i] = ov;
    float4 of = gF[i];
    of.x = of.x + vs[0] * C.q; of.y = of.y + vs[1] * C.q; of.z = of.z + vs[2] * C.q;
    gF[i] = of;
    gFp_prev[i] = make_float4(vs[0] * C.q, vs[1] * C.q, vs[2] * C.q, p_prev ? p_prev[i] : 0.0f);
}

// reverse of the viscosity force
template <int LANES>
__global__ __launch_bounds__(AB) void kr_ext(int n, const float4* __restrict__ x, const float4* __restrict__ v,
                                             const uint32_t* __restrict__ nb, const int* __restrict__ cnt, int ld,
                                             Consts C, const float4* __restrict__ gF, float4* __restrict__ nx,
                                             float4* __restrict__ nv) {
    const unsigned id = blockIdx.x * AB + threadIdx.x;
    const int i = (int)(id / LANES), sub = (int)(id % LANES);
    if (i >= n) return;
    float4 xi = x[i], vi = v[i], gi = gF[i];
    const uint32_t* row = nb + (size_t)i * ld;
    RowHead head = row_head<LANES>(row, ld, cnt + i, sub);
    together(xi, vi, gi, head);
    if (!is_fluid(xi)) return;
    float gvx = 0.0f, gvy = 0.0f, gvz = 0.0f, gxx = 0.0f, gxy = 0.0f, gxz = 0.0f;
    struct Rec {
        float4 x, g, v;
    };
    struct Terms {
        Term3 v, x;
    };
    for_pairs<LANES>(
        row, head, sub, [&](uint32_t j) { return Rec{x[j], gF[j], v[j]}; },
        [&](const Rec& q, bool have) {
            const float4 &xj = q.x, &gj = q.g, &vj = q.v;
            Terms t = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
            if (!have || !is_fluid(xj)) return t;
            const float4 d = make_float4(xi.x - xj.x, xi.y - xj.y, xi.z - xj.z, 0.0f);
            const float r = len3(d.x, d.y, d.z);
            const float4 w = make_float4(gi.x - gj.x, gi.y - gj.y, gi.z - gj.z, 0.0f);
            const float sl = C.cvis * C.kn.L(r);
            t.v = {w.x * sl, w.y * sl, w.z * sl};
            if (r > 0.0f) {
                const float4 dv = make_float4(vi.x - vj.x, vi.y - vj.y, vi.z - vj.z, 0.0f);
                const float s = C.cvis * C.kn.dL(r) / r * dot3(dv, w);
                t.x = {d.x * s, d.y * s, d.z * s};
            }
            return t;
        },
        [&](const Terms& t) {
            sub_terms<LANES>(gvx, gvy, gvz, t.v);
            sub_terms<LANES>(gxx, gxy, gxz, t.x);
        });
    if (sub != 0) return;
    float wf[3], wg[3];
    wall_force(C, xi.x, xi.y, xi.z, wf, wg);
    gxx = gxx + gi.x * wg[0];
    gxy = gxy + gi.y * wg[1];
    gxz = gxz + gi.z * wg[2];
    float4 ov = nv[i];
    ov.x = ov.x + gvx; ov.y = ov.y + gvy; ov.z = ov.z + gvz;
    nv[i] = ov;
    float4 o = nx[i];
    o.x = o.x + gxx; o.y = o.y + gxy; o.z = o.z + gxz;
    nx[i] = o;
}

}  // namespace ad
}  // namespace upf

using namespace upf;
using namespace upf::ad;

#define ADCHK(x)                                   \
    do {                                           \
        hipError_t e_ = (x);                       \
        if (e_ != hipSuccess) return UPF_ERR_HIP;  \
    } while (0)

struct upf_adjoint {
    upf_params P;
    int n = 0, steps = 0, K = 0, ckpt = 0, nseg = 0;
    bool have_forward = false;
    hipStream_t st = nullptr;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    float fwd_ms = 0.0f, bwd_ms = 0.0f;
    std::vector<void*> allocs;
    // state between steps (two buffers) and neighbour search
    float4 *x[2] = {nullptr, nullptr}, *v[2] = {nullptr, nullptr};
    uint32_t *keys = nullptr, *skeys = nullptr, *perm = nullptr;
    uint2* cells = nullptr;
    float4* cand = nullptr;
    uint32_t ncells = 0;
    Bins bins = {};            // count null: sorted by key instead (bins_apply)
    void* sort_tmp = nullptr;  // the key sort's arrays: skeys, perm, sort_tmp
    Ctl* ctl = nullptr;
    // forward work; rec: the pair passes' gathered records
    float4 *F = nullptr, *xs = nullptr, *rec = nullptr;
    float* p = nullptr;
    // checkpoints (x, v) at the start of every segment
    float4 *ck_x = nullptr, *ck_v = nullptr;
    // segment tape: per step (after the segment's first) x, v, per step y's
    // type and clamped axes, lists; per iteration x*, p, rho
    float4 *t_x = nullptr, *t_v = nullptr, *t_xs = nullptr;
    uint32_t* t_nb = nullptr;
    int* t_cnt = nullptr;
    float *t_y = nullptr, *t_p = nullptr, *t_rho = nullptr;
    // adjoint state
    float4 *gx = nullptr, *gv = nullptr, *nx = nullptr, *nv = nullptr, *gF = nullptr, *gFp = nullptr, *gFp2 = nullptr;
    float* gp = nullptr;

    template <class T> hipError_t alloc(T** ptr, size_t count) {
        hipError_t e = hipMalloc((void**)ptr, std::max<size_t>(count, 1) * sizeof(T));
        if (e == hipSuccess) allocs.push_back((void*)*ptr);
        return e;
    }
    Consts consts() const {
        Consts C(P.support_radius);
        C.m = P.initial_mass;
        C.rho0 = P.rest_density;
        C.dt = P.dt;
        C.q = P.dt / P.initial_mass;
        C.cvis = (P.initial_mass / P.rest_density) * (P.initial_mass / P.rest_density) * P.visc_const;
        C.cp = (P.initial_mass * P.initial_mass) / (P.rest_density * P.rest_density);
        C.delta = P.density_error_factor;
        C.g = P.gravity;
        C.fd = P.force_distance;
        C.kb = 2.0f * P.max_boundary_force / P.force_distance;
        for (int a = 0; a < 3; ++a) {
            C.cmin[a] = P.collision_min[a];
            C.cmax[a] = P.collision_max[a];
        }
        return C;
    }
    dim3 grid(int per = 1) const { return dim3((unsigned)(((size_t)n * per + AB - 1) / AB)); }
    // Lanes per particle of the pair passes: a row of 16 where quads would
    // leave the SIMDs with less than two waves each (16 lanes of a partial last
    // round idle, and each particle's own work is repeated on all of them).
    int lanes() const { return n < 32768 ? 16 : 4; }
    size_t nb_stride() const { return (size_t)P.max_neighbors * n; }
};

// first keys and an empty cell table for the positions x; each step leaves
// both ready for the next
static void enqueue_begin(upf_adjoint* a, const float4* x) {
    hipLaunchKernelGGL(k_keys, a->grid(), dim3(AB), 0, a->st, a->n, x, a->P, a->keys, a->ctl);
    if (!a->bins.count)
        hipLaunchKernelGGL(k_clear_cells, dim3((a->ncells + AB - 1) / AB), dim3(AB), 0, a->st, a->cells, a->ncells);
}

// one forward step (x, v) -> (xn, vn); with `tape` >= 0 the step's lists and
// iteration states go to tape slot `tape`.  more: another step follows.
template <int LANES>
static void enqueue_step(upf_adjoint* a, const float4* x, const float4* v, float4* xn, float4* vn, int tape, bool more) {
    const int n = a->n, K = a->K, ld = a->P.max_neighbors;
    const Consts C = a->consts();
    const dim3 g = a->grid(LANES), b(AB);
    const bool rec = tape >= 0;
    uint32_t* nb = rec ? a->t_nb + (size_t)tape * a->nb_stride() : a->t_nb;
    int* cnt = rec ? a->t_cnt + (size_t)tape * n : a->t_cnt;
    auto xs = [&](int k) { return rec ? a->t_xs + ((size_t)tape * K + k) * n : a->xs; };
    const CellMap map{3u * a->P.block_shift, nullptr, nullptr};
    if (a->bins.count) {
        (void)cell_bins(a->keys, n, map, a->bins, a->st);
        hipLaunchKernelGGL(k_rank_cand, a->grid(), b, 0, a->st, n, map, a->bins.place, a->cells, x, a->cand, a->ctl);
    } else {
        (void)radix_sort(a->keys, nullptr, a->skeys, a->perm, n, 30, a->sort_tmp, a->st);
        hipLaunchKernelGGL(k_cell_bounds, a->grid(), b, 0, a->st, n, a->skeys, a->perm, x, map.shift3, a->cells, a->cand);
    }
    hipLaunchKernelGGL(k_lists, a->grid(LIST_LANES), b, 0, a->st, n, x, a->cand, a->cells, a->P, nb, cnt, a->ctl);
    hipLaunchKernelGGL(k_ext<LANES>, g, b, 0, a->st, n, x, v, nb, cnt, ld, C, a->F, a->p, xs(0), a->cells,
                       a->bins.count ? 0u : a->ncells, a->ctl);
    for (int k = 0; k < K; ++k) {
        const size_t o = ((size_t)tape * K + k) * n;
        hipLaunchKernelGGL(k_density<LANES>, g, b, 0, a->st, n, x, xs(k), nb, cnt, ld, C, a->p, a->rec,
                           rec ? a->t_p + o : nullptr, rec ? a->t_rho + o : nullptr);
        if (k + 1 < K)
            hipLaunchKernelGGL((k_pforce<LANES, false>), g, b, 0, a->st, n, x, v, nb, cnt, ld, C, a->rec, a->F, xs(k + 1),
                               nullptr, nullptr, nullptr, a->P, nullptr, a->ctl);
        else
            hipLaunchKernelGGL((k_pforce<LANES, true>), g, b, 0, a->st, n, x, v, nb, cnt, ld, C, a->rec, a->F, nullptr, xn,
                               vn, rec ? a->t_y + (size_t)tape * n : nullptr, a->P, more ? a->keys : nullptr, a->ctl);
    }
}

// reverse of the step (x, v) in tape slot `tape`: (gx, gv) -> (gx, gv)
template <int LANES>
static void enqueue_step_back(upf_adjoint* a, const float4* x, const float4* v, int tape) {
    const int n = a->n, K = a->K, ld = a->P.max_neighbors;
    const Consts C = a->consts();
    const dim3 g = a->grid(LANES), b(AB);
    const uint32_t* nb = a->t_nb + (size_t)tape * a->nb_stride();
    const int* cnt = a->t_cnt + (size_t)tape * n;
    const size_t o0 = (size_t)tape * K * n;
    hipLaunchKernelGGL(kr_integrate, a->grid(), b, 0, a->st, n, a->t_y + (size_t)tape * n, a->gx, a->gv, C,
                       a->t_p + o0 + (size_t)(K - 1) * n, a->nx, a->nv, a->gF, a->gFp, a->gFp2, a->gp);
    for (int k = K - 1; k >= 0; --k) {
        const size_t o = o0 + (size_t)k * n;
        hipLaunchKernelGGL(kr_pforce<LANES>, g, b, 0, a->st, n, x, nb, cnt, ld, C, a->gFp, a->t_xs + o, a->t_rho + o,
                           a->gp, a->nx, a->rec);
        hipLaunchKernelGGL(kr_density<LANES>, g, b, 0, a->st, n, a->t_xs + o, a->rec, nb, cnt, ld, C,
                           k > 0 ? a->t_p + o - n : nullptr, a->nx, a->nv, a->gF, a->gFp2);
        std::swap(a->gFp, a->gFp2);
    }
    hipLaunchKernelGGL(kr_ext<LANES>, g, b, 0, a->st, n, x, v, nb, cnt, ld, C, a->gF, a->nx, a->nv);
    std::swap(a->gx, a->nx);
    std::swap(a->gv, a->nv);
}

static int adj_error(upf_adjoint* a) {
    Ctl h;
    ADCHK(hipMemcpyAsync(&h, a->ctl, sizeof(Ctl), hipMemcpyDeviceToHost, a->st));
    ADCHK(hipStreamSynchronize(a->st));
    const int order[] = {UPF_ERR_NAN, UPF_ERR_RANGE, UPF_ERR_NBR_OVERFLOW};
    for (int c : order)
        if (h.err & (1u << c)) return c;
    return UPF_OK;
}

extern "C" {

int upf_adjoint_destroy(upf_adjoint* a) {
    if (!a) return UPF_ERR_ARG;
    if (a->st) (void)hipStreamSynchronize(a->st);
    for (void* p : a->allocs) (void)hipFree(p);
    for (auto& e : a->ev)
        if (e) (void)hipEventDestroy(e);
    if (a->st) (void)hipStreamDestroy(a->st);
    delete a;
    return UPF_OK;
}

int upf_adjoint_create(const upf_params* p, int n, int steps, int iterations, int checkpoint_every, upf_adjoint** out) {
    if (!p || !out || n <= 0 || steps <= 0 || iterations <= 0 || checkpoint_every <= 0) return UPF_ERR_ARG;
    if (upf::check_params(p) != UPF_OK) return UPF_ERR_ARG;
    if (p->add_wall_weight) return UPF_ERR_ARG;  // the differentiable step has no wall weight
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return UPF_ERR_NO_DEVICE;
    upf_adjoint* a = new upf_adjoint();
    a->P = *p;
    a->n = n;
    a->steps = steps;
    a->K = iterations;
    a->ckpt = std::min(checkpoint_every, steps);
    a->nseg = (steps + a->ckpt - 1) / a->ckpt;
    a->ncells = p->grid_dim * p->grid_dim * p->grid_dim;
    const size_t T = (size_t)a->ckpt;
    bool ok = hipStreamCreateWithFlags(&a->st, hipStreamNonBlocking) == hipSuccess;
    for (auto& e : a->ev) ok = ok && hipEventCreate(&e) == hipSuccess;
    ok = ok && a->alloc(&a->x[0], n) == hipSuccess && a->alloc(&a->v[0], n) == hipSuccess &&
         a->alloc(&a->x[1], n) == hipSuccess && a->alloc(&a->v[1], n) == hipSuccess &&
         a->alloc(&a->cand, n) == hipSuccess &&
         a->alloc(&a->keys, n) == hipSuccess && a->alloc(&a->cells, a->ncells) == hipSuccess &&
         a->alloc(&a->ctl, 1) == hipSuccess && a->alloc(&a->F, n) == hipSuccess && a->alloc(&a->rec, n) == hipSuccess &&
         a->alloc(&a->xs, n) == hipSuccess && a->alloc(&a->p, n) == hipSuccess &&
         a->alloc(&a->ck_x, (size_t)a->nseg * n) == hipSuccess && a->alloc(&a->ck_v, (size_t)a->nseg * n) == hipSuccess &&
         a->alloc(&a->t_x, T * n) == hipSuccess && a->alloc(&a->t_v, T * n) == hipSuccess &&
         a->alloc(&a->t_y, T * n) == hipSuccess && a->alloc(&a->t_xs, T * a->K * n) == hipSuccess &&
         a->alloc(&a->t_nb, T * a->nb_stride()) == hipSuccess && a->alloc(&a->t_cnt, T * n) == hipSuccess &&
         a->alloc(&a->t_p, T * a->K * n) == hipSuccess && a->alloc(&a->t_rho, T * a->K * n) == hipSuccess &&
         a->alloc(&a->gx, n) == hipSuccess && a->alloc(&a->gv, n) == hipSuccess && a->alloc(&a->nx, n) == hipSuccess &&
         a->alloc(&a->nv, n) == hipSuccess && a->alloc(&a->gF, n) == hipSuccess && a->alloc(&a->gFp, n) == hipSuccess &&
         a->alloc(&a->gFp2, n) == hipSuccess && a->alloc(&a->gp, n) == hipSuccess;
    if (ok && bins_apply(n, a->ncells)) {
        a->bins.cells = a->cells;
        a->bins.ncells = a->ncells;
        ok = a->alloc(&a->bins.at, n) == hipSuccess && a->alloc(&a->bins.place, n) == hipSuccess &&
             a->alloc(&a->bins.sums, BIN_BLOCKS) == hipSuccess && a->alloc(&a->bins.count, a->ncells) == hipSuccess &&
             hipMemsetAsync(a->bins.count, 0, (size_t)a->ncells * sizeof(uint32_t), a->st) == hipSuccess;
    } else if (ok) {
        void* tmp = nullptr;
        ok = a->alloc(&a->skeys, n) == hipSuccess && a->alloc(&a->perm, n) == hipSuccess &&
             hipMalloc(&tmp, radix_sort_temp_bytes(n)) == hipSuccess;
        if (ok) { a->sort_tmp = tmp; a->allocs.push_back(tmp); }
    }
    if (!ok) {
        upf_adjoint_destroy(a);
        return UPF_ERR_HIP;
    }
    *out = a;
    return UPF_OK;
}

int upf_adjoint_forward(upf_adjoint* a, const float* pos4, const float* vel4, const int* type, float* pos_out4,
                        float* vel_out4) {
    if (!a || !pos4 || !type) return UPF_ERR_ARG;
    const int n = a->n;
    std::vector<float> x((size_t)4 * n), v((size_t)4 * n, 0.0f);
    for (int i = 0; i < n; ++i) {
        if (type[i] != UPF_LIQUID && type[i] != UPF_FROZEN) return UPF_ERR_ARG;
        for (int c = 0; c < 3; ++c) {
            x[4 * i + c] = pos4[4 * i + c];
            if (vel4) v[4 * i + c] = vel4[4 * i + c];
            if (!(a->P.scales[c] * (pos4[4 * i + c] + a->P.support_radius) < 1024.0f) || !(pos4[4 * i + c] >= 0.0f))
                return UPF_ERR_RANGE;
        }
        std::memcpy(&x[4 * i + 3], &type[i], 4);
    }
    // the state at the start of segment k lives in checkpoint k
    ADCHK(hipMemcpyAsync(a->ck_x, x.data(), (size_t)n * 16, hipMemcpyHostToDevice, a->st));
    ADCHK(hipMemcpyAsync(a->ck_v, v.data(), (size_t)n * 16, hipMemcpyHostToDevice, a->st));
    ADCHK(hipMemsetAsync(a->ctl, 0, sizeof(Ctl), a->st));
    ADCHK(hipEventRecord(a->ev[0], a->st));
    float4 *cx = a->ck_x, *cv = a->ck_v;
    enqueue_begin(a, cx);
    for (int s = 0; s < a->steps; ++s) {
        const bool more = s + 1 < a->steps;
        float4 *xn = a->x[s & 1], *vn = a->v[s & 1];
        if (more && (s + 1) % a->ckpt == 0) {
            xn = a->ck_x + (size_t)((s + 1) / a->ckpt) * n;
            vn = a->ck_v + (size_t)((s + 1) / a->ckpt) * n;
        }
        if (a->lanes() == 16) enqueue_step<16>(a, cx, cv, xn, vn, -1, more);
        else enqueue_step<4>(a, cx, cv, xn, vn, -1, more);
        cx = xn;
        cv = vn;
    }
    ADCHK(hipEventRecord(a->ev[1], a->st));
    ADCHK(hipGetLastError());
    int rc = adj_error(a);
    if (rc) return rc;
    ADCHK(hipEventElapsedTime(&a->fwd_ms, a->ev[0], a->ev[1]));
    if (pos_out4 || vel_out4) {
        ADCHK(hipMemcpy(x.data(), cx, (size_t)n * 16, hipMemcpyDeviceToHost));
        ADCHK(hipMemcpy(v.data(), cv, (size_t)n * 16, hipMemcpyDeviceToHost));
        for (int i = 0; i < n; ++i)
            for (int c = 0; c < 4; ++c) {
                if (pos_out4) pos_out4[4 * i + c] = c < 3 ? x[4 * i + c] : 0.0f;
                if (vel_out4) vel_out4[4 * i + c] = c < 3 ? v[4 * i + c] : 0.0f;
            }
    }
    a->have_forward = true;
    return UPF_OK;
}

int upf_adjoint_backward(upf_adjoint* a, const float* dl_dpos4, const float* dl_dvel4, float* dl_dpos0_4,
                         float* dl_dvel0_4) {
    if (!a || !dl_dpos4) return UPF_ERR_ARG;
    if (!a->have_forward) return UPF_ERR_STATE;
    const int n = a->n;
    std::vector<float> g((size_t)4 * n), h((size_t)4 * n, 0.0f);
    for (size_t k = 0; k < g.size(); ++k) {
        g[k] = (k & 3) == 3 ? 0.0f : dl_dpos4[k];
        if (dl_dvel4) h[k] = (k & 3) == 3 ? 0.0f : dl_dvel4[k];
    }
    ADCHK(hipMemcpyAsync(a->gx, g.data(), (size_t)n * 16, hipMemcpyHostToDevice, a->st));
    ADCHK(hipMemcpyAsync(a->gv, h.data(), (size_t)n * 16, hipMemcpyHostToDevice, a->st));
    ADCHK(hipEventRecord(a->ev[2], a->st));
    for (int seg = a->nseg - 1; seg >= 0; --seg) {
        const int s0 = seg * a->ckpt, s1 = std::min(s0 + a->ckpt, a->steps);
        // the states of the segment: its checkpoint, then tape slots 1, 2, ...;
        // the state after its last step is not read (slot 0)
        auto x = [&](int t) { return t == 0 ? a->ck_x + (size_t)seg * n : a->t_x + (size_t)t * n; };
        auto v = [&](int t) { return t == 0 ? a->ck_v + (size_t)seg * n : a->t_v + (size_t)t * n; };
        enqueue_begin(a, x(0));
        for (int t = 0; t < s1 - s0; ++t) {  // recompute, taping
            const bool more = t + 1 < s1 - s0;
            float4 *xn = more ? x(t + 1) : a->t_x, *vn = more ? v(t + 1) : a->t_v;
            if (a->lanes() == 16) enqueue_step<16>(a, x(t), v(t), xn, vn, t, more);
            else enqueue_step<4>(a, x(t), v(t), xn, vn, t, more);
        }
        for (int t = s1 - s0 - 1; t >= 0; --t) {
            if (a->lanes() == 16) enqueue_step_back<16>(a, x(t), v(t), t);
            else enqueue_step_back<4>(a, x(t), v(t), t);
        }
    }
    ADCHK(hipEventRecord(a->ev[3], a->st));
    ADCHK(hipGetLastError());
    int rc = adj_error(a);
    if (rc) return rc;
    ADCHK(hipEventElapsedTime(&a->bwd_ms, a->ev[2], a->ev[3]));
    ADCHK(hipMemcpy(g.data(), a->gx, (size_t)n * 16, hipMemcpyDeviceToHost));
    ADCHK(hipMemcpy(h.data(), a->gv, (size_t)n * 16, hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i)
        for (int c = 0; c < 4; ++c) {
            if (dl_dpos0_4) dl_dpos0_4[4 * i + c] = c < 3 ? g[4 * i + c] : 0.0f;
            if (dl_dvel0_4) dl_dvel0_4[4 * i + c] = c < 3 ? h[4 * i + c] : 0.0f;
        }
    return UPF_OK;
}

int upf_adjoint_timing(upf_adjoint* a, float* forward_ms, float* backward_ms, size_t* device_bytes) {
    if (!a) return UPF_ERR_ARG;
    if (forward_ms) *forward_ms = a->fwd_ms;
    if (backward_ms) *backward_ms = a->bwd_ms;
    if (device_bytes) {
        const size_t n = (size_t)a->n, T = (size_t)a->ckpt, K = (size_t)a->K;
        *device_bytes = n * 16 * (4 + 1 + 3 + 2 * a->nseg + 2 * T + T * K + 7) + n * 4 * (3 + 2 * T + 2 * T * K) +
                        T * a->nb_stride() * 4 + (size_t)a->ncells * 8;
        *device_bytes += a->bins.count ? n * 12 + (size_t)a->ncells * 4 + BIN_BLOCKS * 4
                                       : n * 8 + radix_sort_temp_bytes(a->n);
    }
    return UPF_OK;
}

}  // extern "C"
