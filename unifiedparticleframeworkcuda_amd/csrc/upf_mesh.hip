// upf_mesh.hip -- OBJ model -> particles, the scene-input path of the
// reference's rigid objects: ObjLoader::Load / LoadFaces (src/cpu/ObjLoader.cpp:18-258)
// read the triangles, ObjectLoader::LoadParticles (src/cpu/ObjectLoader.cpp:8-97)
// keeps the lattice points inside the mesh or on a face (Polygon,
// src/cpu/Polygon.cpp).  The reader runs on the host; the point-in-mesh test of
// every lattice point against every face -- the O(points x faces) part -- runs
// on the GPU, one thread per lattice point over the faces that interval bounds
// leave for its tile of 64 points, and the kept points are compacted in the
// reference's loop order.
//
// Floating point: -ffp-contract=off and correctly rounded division, every
// expression in the reference's evaluation order, so the particle set and its
// positions equal the reference's bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "upf.h"

namespace upf {
namespace {

#define MCHK(x)                                     \
    do {                                            \
        if ((x) != hipSuccess) return UPF_ERR_HIP; \
    } while (0)

struct F3 {
    float x, y, z;
};

// ---------------------------------------------------------------- the reader
// Two passes with a 256-byte fgets buffer under while (!feof(fp)): the fgets
// that meets the end of the file returns nothing and leaves the buffer as it
// was, so the reference processes its last line twice (a file ending in a
// face line gets that face twice).  No faces or no vertices: the reference's
// FileError, i.e. an empty model.
int read_obj(const char* path, std::vector<F3>& tri) {
    tri.clear();
    FILE* fp = std::fopen(path, "r");
    if (!fp) return UPF_ERR_IO;
    char line[256];
    std::memset(line, 0, sizeof(line));
    long n_vertex = 0, n_face = 0;
    while (!std::feof(fp)) {
        if (std::fgets(line, sizeof(line), fp) == nullptr) {
            // end of file: `line` keeps the previous line
        }
        if (std::strncmp("vt ", line, 3) == 0 || std::strncmp("vn ", line, 3) == 0) continue;
        if (std::strncmp("v ", line, 2) == 0) ++n_vertex;
        else if (std::strncmp("f ", line, 2) == 0) ++n_face;
    }
    std::fclose(fp);
    if (n_face == 0 || n_vertex == 0) return UPF_OK;
    fp = std::fopen(path, "r");
    if (!fp) return UPF_ERR_IO;
    std::memset(line, 0, sizeof(line));
    std::vector<F3> vertex;
    std::vector<int> corner;
    bool bad = false;
    while (!std::feof(fp)) {
        if (std::fgets(line, sizeof(line), fp) == nullptr) {
        }
        if (std::strncmp("vt ", line, 3) == 0 || std::strncmp("vn ", line, 3) == 0) continue;
        if (std::strncmp("v ", line, 2) == 0) {
            F3 v{0.0f, 0.0f, 0.0f};
            bad |= std::sscanf(line + 2, "%f%f%f", &v.x, &v.y, &v.z) != 3;
            vertex.push_back(v);
        } else if (std::strncmp("f ", line, 2) == 0) {
            // v/vt/vn triples; the vertex index of the third corner is field 7
            int f[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
            const int got = std::sscanf(line + 2, "%d/%d/%d %d/%d/%d %d/%d/%d", &f[0], &f[1], &f[2], &f[3], &f[4],
                                        &f[5], &f[6], &f[7], &f[8]);
            bad |= got < 7;
            corner.push_back(f[0] - 1);
            corner.push_back(f[3] - 1);
            corner.push_back(f[6] - 1);
        }
    }
    std::fclose(fp);
    if (bad) return UPF_ERR_ARG;  // a line the reference reads into undefined values
    tri.reserve(corner.size());
    for (int c : corner) {
        if (c < 0 || c >= (int)vertex.size()) return UPF_ERR_ARG;
        tri.push_back(vertex[(size_t)c]);
    }
    return UPF_OK;
}

// ----------------------------------------------------------- face constants
// Per face, what the crossing and touching tests read: the unit normal n
// (Polygon::AddVertex: (v0 - v1) x (v2 - v1), vmml's normalize with 1/l in
// double), d = -(v0 . n), the numerator -(d + o . n) of the segment parameter
// for the common segment start o, and for the in-plane test the corners and
// its far point (box minimum - 1, the box starting at the origin like the
// reference's) projected on the two coordinates that it reads, with the side
// of each edge that the far point lies on.  64 bytes: one scalar load.
struct alignas(64) Face {
    float nx, ny, nz, d;
    float va[3], oa;  // first projected coordinate: corners, far point
    float vb[3], ob;  // second
    float num;
    int code;  // 1: the first coordinate is y (else x), 2: the second is z (else y), 4 << k: side of edge k
    int pad[2];
};
constexpr int FACE_Y = 1, FACE_Z = 2, FACE_SIDE = 4;

inline float dot(const F3& a, const F3& b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

void face_box(const F3* v, F3& mn, F3& mx) {
    mn = {0.0f, 0.0f, 0.0f};
    mx = {0.0f, 0.0f, 0.0f};
    for (int k = 0; k < 3; ++k) {
        const float c[3] = {v[k].x, v[k].y, v[k].z};
        float* pmn = &mn.x;
        float* pmx = &mx.x;
        for (int i = 0; i < 3; ++i) {
            pmn[i] = std::min(c[i], pmn[i]);
            pmx[i] = std::max(c[i], pmx[i]);
        }
    }
}

F3 face_normal(const F3* v) {
    const F3 a{v[0].x - v[1].x, v[0].y - v[1].y, v[0].z - v[1].z};
    const F3 b{v[2].x - v[1].x, v[2].y - v[1].y, v[2].z - v[1].z};
    F3 n{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
    const float l = std::sqrt(n.x * n.x + n.y * n.y + n.z * n.z);
    if (l != 0.0f) {
        const float ll = (float)(1.0 / (double)l);
        n.x *= ll;
        n.y *= ll;
        n.z *= ll;
    }
    return n;
}

// ------------------------------------------------------------------ device
// Polygon::IsPointInPlaneInside (Polygon.cpp:118-137): the edges that the
// segment from the far point to (pa, pb) crosses, by
// Polygon::ArePointsOnBothSidesOfTheLine (Polygon.cpp:73-103) of the corners
// against the segment's line (g) and of its ends against the edge's line.
__device__ __forceinline__ bool in_plane_inside(const Face& f, float px, float py, float pz) {
    const float pa = f.code & FACE_Y ? py : px, pb = f.code & FACE_Z ? pz : py;
    const float dx = pa - f.oa, dy = f.ob - pb;
    bool g[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) g[k] = (dy * (f.va[k] - pa)) > ((pb - f.vb[k]) * dx);
    bool inside = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int e = k == 2 ? 0 : k + 1;
        const bool h = ((f.vb[k] - f.vb[e]) * (pa - f.va[e])) > ((f.vb[e] - pb) * (f.va[e] - f.va[k]));
        inside ^= (g[k] != g[e]) && h != ((f.code & (FACE_SIDE << k)) != 0);
    }
    return inside;
}

constexpr int MF_BLOCK = 256;  // points per block of the count and emit kernels
constexpr int MT_BLOCK = 512;  // points (threads) per block of the test
constexpr int MT_LIST = 2048;  // faces a block holds between its two rulings

// ------------------------------------------------- faces that cannot matter
// Interval bounds of the test's own float expressions over a tile of lattice
// points.  A rounded sum, difference, product or quotient is monotone in each
// operand, so an expression evaluated at the right ends of its operands'
// ranges bounds every value it takes inside them, rounding included: a face
// that these bounds rule out neither toggles nor keeps any point of the tile.
struct Iv {
    float lo, hi;
};
__device__ __forceinline__ Iv iv_mul(const Iv& a, const Iv& b) {
    const float p = a.lo * b.lo, q = a.lo * b.hi, r = a.hi * b.lo, s = a.hi * b.hi;
    return {fminf(fminf(p, q), fminf(r, s)), fmaxf(fmaxf(p, q), fmaxf(r, s))};
}
__device__ __forceinline__ Iv iv_mul(const Iv& a, float c) {
    const float p = a.lo * c, q = a.hi * c;
    return {fminf(p, q), fmaxf(p, q)};
}
// l > r over the ranges: 1 always, 0 never, -1 undecided
__device__ __forceinline__ int iv_greater(const Iv& l, const Iv& r) {
    return l.lo > r.hi ? 1 : (l.hi <= r.lo ? 0 : -1);
}
__device__ __forceinline__ Iv iv_dot(const Iv& x, const Iv& y, const Iv& z, const float3& n) {
    const Iv a = iv_mul(x, n.x), b = iv_mul(y, n.y), c = iv_mul(z, n.z);
    return {a.lo + b.lo + c.lo, a.hi + b.hi + c.hi};
}

// in_plane_inside() is false for every point whose projected coordinates lie
// in a x b: each edge toggles for all of them or for none, an even number do.
__device__ __forceinline__ bool outside_in_plane(const Face& f, const Iv& a, const Iv& b) {
    const Iv dy = {f.ob - b.hi, f.ob - b.lo}, dx = {a.lo - f.oa, a.hi - f.oa};
    int g[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
        g[k] = iv_greater(iv_mul(dy, Iv{f.va[k] - a.hi, f.va[k] - a.lo}), iv_mul(Iv{b.lo - f.vb[k], b.hi - f.vb[k]}, dx));
    bool sure = true, odd = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int e = k == 2 ? 0 : k + 1;
        const int h = iv_greater(iv_mul(Iv{a.lo - f.va[e], a.hi - f.va[e]}, f.vb[k] - f.vb[e]),
                                 iv_mul(Iv{f.vb[e] - b.hi, f.vb[e] - b.lo}, f.va[e] - f.va[k]));
        const int ho = f.code & (FACE_SIDE << k) ? 1 : 0;
        const bool gsure = g[k] >= 0 && g[e] >= 0;
        const bool never = (gsure && g[k] == g[e]) || h == ho;
        odd ^= !never;  // always toggles, if sure
        sure = sure && (never || (gsure && h >= 0));
    }
    return sure && !odd;
}

// a box of lattice points and their offsets from o
struct Box {
    Iv x, y, z, dx, dy, dz;
};

__device__ __forceinline__ bool face_matters(const Face& f, const Box& B, const float3& o) {
    const float3 n = make_float3(f.nx, f.ny, f.nz);
    const Iv eq = iv_dot(B.x, B.y, B.z, n);
    const bool touch = eq.lo + f.d <= 0.000001f && eq.hi + f.d >= -0.000001f;
    const Iv den = iv_dot(B.dx, B.dy, B.dz, n);
    // segment parameters in [0, 1] that the box's points can have
    bool cross = den.hi >= 0.000001f || den.lo <= -0.000001f;
    Iv t = {0.0f, 1.0f};
    if (den.lo >= 0.000001f || den.hi <= -0.000001f) {  // one sign: the quotient is monotone
        const float p = f.num / den.lo, q = f.num / den.hi;
        const float lo = fminf(p, q), hi = fmaxf(p, q);
        cross = !(hi < 0.0f || lo > 1.0f);
        t = {fmaxf(lo, 0.0f), fminf(hi, 1.0f)};
    }
    if (!cross && !touch) return false;
    const bool fy = f.code & FACE_Y, fz = f.code & FACE_Z;
    const Iv pa = fy ? B.y : B.x, pb = fz ? B.z : B.y;
    Iv a = pa, b = pb;
    if (cross) {  // crossing points o + d t, joined with the points themselves if those can touch
        const Iv ma = iv_mul(fy ? B.dy : B.dx, t), mb = iv_mul(fz ? B.dz : B.dy, t);
        const float ba = fy ? o.y : o.x, bb = fz ? o.z : o.y;
        const Iv ca = {ba + ma.lo, ba + ma.hi}, cb = {bb + mb.lo, bb + mb.hi};
        a = touch ? Iv{fminf(pa.lo, ca.lo), fmaxf(pa.hi, ca.hi)} : ca;
        b = touch ? Iv{fminf(pb.lo, cb.lo), fmaxf(pb.hi, cb.hi)} : cb;
    }
    return !outside_in_plane(f, a, b);
}

// the lattice of a launch: extents, and log2 of a block's and of a wave's box
struct Lattice {
    int n[3], bb[3], wb[3];
};

// the box of the points p0 .. p1 (inclusive); odd x: y and z start half a
// spacing later, and coordinates never decrease along a row
__device__ __forceinline__ Box lattice_box(const float* __restrict__ X, const float* __restrict__ Y,
                                           const float* __restrict__ Z, const Lattice& L, const int* p0, const int* p1,
                                           const float3& o) {
    Box B;
    B.x = {X[p0[0]], X[p1[0]]};
    B.y = {fminf(Y[p0[1]], Y[L.n[1] + p0[1]]), fmaxf(Y[p1[1]], Y[L.n[1] + p1[1]])};
    B.z = {fminf(Z[p0[2]], Z[L.n[2] + p0[2]]), fmaxf(Z[p1[2]], Z[L.n[2] + p1[2]])};
    B.dx = {B.x.lo - o.x, B.x.hi - o.x};
    B.dy = {B.y.lo - o.y, B.y.hi - o.y};
    B.dz = {B.z.lo - o.z, B.z.hi - o.z};
    return B;
}

// One block per box of 512 lattice points (8 x 8 x 8 unless the lattice is
// thin), one wave per 64 of them (4 x 4 x 4).  The block rules faces out for
// its box, one face per thread; each wave rules out what is left for its own
// box, one face per lane; the faces left after that run in file order, one
// lattice point per lane: Polygon::DoesLineIntersect of the segment from o to
// the point toggles the point; otherwise Polygon::DoesPointTouch keeps it and
// ends its scan.  keep[] gets the decision.
// Bound by VALU.  652,228 points and 6,400 faces: 26.9 ms with every pair
// tested, 1.03 ms now (4.0 ms with one ruling per wave over all faces staged
// in LDS); of a wave's 6,400 faces about 360 are left, since few faces are met
// along the segments to a small box.  A face left is one scalar load.  `cull` 0: coordinates so large that a
// product may overflow; every face runs.
__global__ __launch_bounds__(MT_BLOCK) void k_mesh_test(const Face* __restrict__ faces, int nf,
                                                        const float* __restrict__ X, const float* __restrict__ Y,
                                                        const float* __restrict__ Z, Lattice L, float3 o, int cull,
                                                        uint8_t* __restrict__ keep) {
    constexpr int WAVES = MT_BLOCK / 64;
    __shared__ int list[MT_LIST];  // faces the block's box leaves, in file order
    __shared__ int wcnt[WAVES];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // the block's box, the wave's box in it, the lane's point
    const int nby = ((L.n[1] - 1) >> L.bb[1]) + 1, nbz = ((L.n[2] - 1) >> L.bb[2]) + 1;
    const int b0[3] = {(int)(blockIdx.x / (nby * nbz)) << L.bb[0], (int)(blockIdx.x / nbz % nby) << L.bb[1],
                       (int)(blockIdx.x % nbz) << L.bb[2]};
    const int sy = L.bb[1] - L.wb[1], sz = L.bb[2] - L.wb[2];
    const int w0[3] = {b0[0] + ((w >> (sy + sz)) << L.wb[0]), b0[1] + (((w >> sz) & ((1 << sy) - 1)) << L.wb[1]),
                       b0[2] + ((w & ((1 << sz) - 1)) << L.wb[2])};
    const int x = w0[0] + (lane >> (L.wb[1] + L.wb[2])), y = w0[1] + ((lane >> L.wb[2]) & ((1 << L.wb[1]) - 1)),
              z = w0[2] + (lane & ((1 << L.wb[2]) - 1));
    const bool wave = w0[0] < L.n[0] && w0[1] < L.n[1] && w0[2] < L.n[2];
    const bool live = wave && x < L.n[0] && y < L.n[1] && z < L.n[2];
    int b1[3], w1[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        b1[a] = min(b0[a] + (1 << L.bb[a]), L.n[a]) - 1;
        w1[a] = min(w0[a] + (1 << L.wb[a]), L.n[a]) - 1;
    }
    const Box bbox = lattice_box(X, Y, Z, L, b0, b1, o);
    Box wbox = bbox;
    if (wave) wbox = lattice_box(X, Y, Z, L, w0, w1, o);
    float3 p = make_float3(0.f, 0.f, 0.f);
    if (live) p = make_float3(X[x], Y[(x & 1) * L.n[1] + y], Z[(x & 1) * L.n[2] + z]);
    // segment o -> p
    const float3 dv = make_float3(p.x - o.x, p.y - o.y, p.z - o.z);
    bool add = false, done = !live;
    int len = 0;  // list entries so far (the same in every thread)
    for (int f0 = 0; f0 < nf; f0 += MT_BLOCK) {
        const int fi = f0 + (int)threadIdx.x;
        bool in = fi < nf;
        if (in && cull) in = face_matters(faces[fi], bbox, o);
        const uint64_t m = __ballot(in);
        if (lane == 0) wcnt[w] = __popcll(m);
        __syncthreads();
        int at = len;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) {
            const int c = wcnt[k];
            if (k < w) at += c;
            len += c;
        }
        if (in) list[at + __popcll(m & ((1ull << lane) - 1ull))] = fi;
        __syncthreads();
        if (len <= MT_LIST - MT_BLOCK && f0 + MT_BLOCK < nf) continue;  // room for another round
        for (int g = 0; wave && g < len; g += 64) {
            bool mine = g + lane < len;
            const int my = mine ? list[g + lane] : 0;
            if (mine && cull) mine = face_matters(faces[my], wbox, o);
            for (uint64_t left = __ballot(mine); left; left &= left - 1) {
                const Face& f = faces[__builtin_amdgcn_readlane(my, __builtin_ctzll(left))];
                if (done) continue;
                bool crosses = false;
                const float den = dv.x * f.nx + dv.y * f.ny + dv.z * f.nz;
                if (!(fabsf(den) < 0.000001f)) {
                    const float dof = f.num / den;
                    if (!(dof < 0.0f || dof > 1.0f))
                        crosses = in_plane_inside(f, o.x + dv.x * dof, o.y + dv.y * dof, o.z + dv.z * dof);
                }
                if (crosses) {
                    add = !add;
                } else {
                    const float eq = (p.x * f.nx + p.y * f.ny + p.z * f.nz) + f.d;
                    if (!(fabsf(eq) > 0.000001f) && in_plane_inside(f, p.x, p.y, p.z)) {
                        add = true;
                        done = true;
                    }
                }
            }
        }
        len = 0;
        if (__syncthreads_count(!done) == 0) break;  // also: every wave is past the list
    }
    if (live) keep[((long long)x * L.n[1] + y) * L.n[2] + z] = (uint8_t)add;
}

// kept points of each block of MF_BLOCK lattice points (x-major, then y, then
// z: the reference's loop order)
__global__ __launch_bounds__(MF_BLOCK) void k_mesh_count(const uint8_t* __restrict__ keep, long long npts,
                                                         int* __restrict__ counts) {
    const long long idx = (long long)blockIdx.x * MF_BLOCK + threadIdx.x;
    const int c = __syncthreads_count(idx < npts && keep[idx]);
    if (threadIdx.x == 0) counts[blockIdx.x] = c;
}

// exclusive prefix of the block counts (one block)
__global__ __launch_bounds__(1024) void k_mesh_scan(int* __restrict__ counts, int nb, int* __restrict__ total) {
    __shared__ int part[1024];
    const int per = (nb + 1023) / 1024;
    const int beg = threadIdx.x * per, end = min(beg + per, nb);
    int s = 0;
    for (int i = beg; i < end; ++i) s += counts[i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    int run = threadIdx.x ? part[threadIdx.x - 1] : 0;
    for (int i = beg; i < end; ++i) {
        const int c = counts[i];
        counts[i] = run;
        run += c;
    }
    if (threadIdx.x == 1023) *total = part[1023];
}

// kept points in lattice order: (p - box minimum) * scale
__global__ __launch_bounds__(MF_BLOCK) void k_mesh_emit(const uint8_t* __restrict__ keep,
                                                        const int* __restrict__ offsets, const float* __restrict__ X,
                                                        const float* __restrict__ Y, const float* __restrict__ Z,
                                                        int nx, int ny, int nz, float3 mn, float3 sc,
                                                        float4* __restrict__ out, int cap) {
    __shared__ int wave_base[MF_BLOCK / 64];
    const long long npts = (long long)nx * ny * nz;
    const long long idx = (long long)blockIdx.x * MF_BLOCK + threadIdx.x;
    const bool k = idx < npts && keep[idx];
    const uint64_t m = __ballot(k);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) wave_base[w] = __popcll(m);
    __syncthreads();
    int base = offsets[blockIdx.x];
    for (int i = 0; i < w; ++i) base += wave_base[i];
    const uint64_t below = lane ? (m & (~0ull >> (64 - lane))) : 0ull;
    const int slot = base + __popcll(below);
    if (k && slot < cap) {
        const int z = (int)(idx % nz);
        const int y = (int)((idx / nz) % ny);
        const int x = (int)(idx / ((long long)ny * nz));
        const int par = x & 1;
        out[slot] = make_float4((X[x] - mn.x) * sc.x, (Y[par * ny + y] - mn.y) * sc.y, (Z[par * nz + z] - mn.z) * sc.z,
                                0.0f);
    }
}

// number of lattice steps: the reference's `for (int i = 0; i <= steps; ++i)`
long long loop_count(float steps) {
    if (!(steps >= 0.0f)) return 0;
    if (steps >= 16777216.0f) return -1;  // past exact float integers: refused
    long long c = 0;
    while ((float)c <= steps) ++c;
    return c;
}

}  // namespace
}  // namespace upf

using namespace upf;

extern "C" {

int upf_obj_read(const char* path, float* faces9, int cap, int* n_faces) {
    if (!path || !n_faces || (faces9 && cap < 0)) return UPF_ERR_ARG;
    std::vector<F3> tri;
    const int rc = read_obj(path, tri);
    if (rc) return rc;
    const int n = (int)(tri.size() / 3);
    *n_faces = n;
    if (faces9) {
        if (cap < n) return UPF_ERR_RANGE;
        std::memcpy(faces9, tri.data(), tri.size() * sizeof(F3));
    }
    return UPF_OK;
}

int upf_mesh_fill(const float* faces9, int n_faces, const float scale[3], float spacing, float* pos4, int cap,
                  int* n_out) {
    if (!n_out || n_faces < 0 || (n_faces > 0 && !faces9) || !scale || (pos4 && cap < 0)) return UPF_ERR_ARG;
    if (!(spacing > 0.0f) || !(scale[0] > 0.0f) || !(scale[1] > 0.0f) || !(scale[2] > 0.0f)) return UPF_ERR_ARG;
    *n_out = 0;
    if (n_faces == 0) return UPF_OK;
    // faces: the box of each (from the origin) and of the model, constants
    std::vector<Face> faces((size_t)n_faces);
    const F3* tri = reinterpret_cast<const F3*>(faces9);
    F3 mn{}, mx{};
    std::vector<F3> fmn((size_t)n_faces), fmx((size_t)n_faces), fn((size_t)n_faces);
    for (int f = 0; f < n_faces; ++f) {
        face_box(tri + 3 * (size_t)f, fmn[f], fmx[f]);
        fn[f] = face_normal(tri + 3 * (size_t)f);
    }
    mn = fmn[0];
    mx = fmx[0];
    for (int f = 0; f < n_faces; ++f) {
        float* a = &mn.x;
        float* b = &mx.x;
        const float* c = &fmn[f].x;
        const float* d = &fmx[f].x;
        for (int i = 0; i < 3; ++i) {
            a[i] = std::min(a[i], c[i]);
            b[i] = std::max(b[i], d[i]);
        }
    }
    const F3 o{mn.x - spacing, mn.y - spacing, mn.z - spacing};  // the segments' common start
    for (int f = 0; f < n_faces; ++f) {
        const F3* v = tri + 3 * (size_t)f;
        const F3& n = fn[f];
        const float d = -dot(v[0], n);
        const float num = -(d + dot(o, n));
        Face& F = faces[(size_t)f];
        const bool fy = n.x != 0, fz = fy || n.y != 0;
        F.nx = n.x;
        F.ny = n.y;
        F.nz = n.z;
        F.d = d;
        F.num = num;
        F.code = (fy ? FACE_Y : 0) | (fz ? FACE_Z : 0);
        F.oa = (fy ? fmn[f].y : fmn[f].x) - 1.0f;
        F.ob = (fz ? fmn[f].z : fmn[f].y) - 1.0f;
        for (int k = 0; k < 3; ++k) {
            F.va[k] = fy ? v[k].y : v[k].x;
            F.vb[k] = fz ? v[k].z : v[k].y;
        }
        for (int k = 0; k < 3; ++k) {
            const int e = k == 2 ? 0 : k + 1;
            if (((F.vb[k] - F.vb[e]) * (F.oa - F.va[e])) > ((F.vb[e] - F.ob) * (F.va[e] - F.va[k])))
                F.code |= FACE_SIDE << k;
        }
    }
    // the lattice: coordinates accumulated step by step as the reference's
    // loops do (odd x: y and z start half a spacing later)
    const float xs = (mx.x - mn.x) * scale[0] / spacing;
    const float ys = (mx.y - mn.y) * scale[1] / spacing;
    const float zs = (mx.z - mn.z) * scale[2] / spacing;
    const long long nx = loop_count(xs), ny = loop_count(ys), nz = loop_count(zs);
    if (nx < 0 || ny < 0 || nz < 0) return UPF_ERR_ARG;
    if (nx == 0 || ny == 0 || nz == 0) return UPF_OK;
    const long long npts = nx * ny * nz;
    if (npts > (1ll << 31) - 1) return UPF_ERR_ARG;
    std::vector<float> X((size_t)nx), Y(2 * (size_t)ny), Z(2 * (size_t)nz);
    {
        float cx = mn.x;
        for (long long x = 0; x < nx; ++x) {
            X[(size_t)x] = cx;
            cx += spacing / scale[0];
        }
        for (int par = 0; par < 2; ++par) {
            float cy = mn.y + par * spacing / (2 * scale[1]);
            for (long long y = 0; y < ny; ++y) {
                Y[(size_t)(par * ny + y)] = cy;
                cy += spacing / scale[1];
            }
            float cz = mn.z + par * spacing / (2 * scale[2]);
            for (long long z = 0; z < nz; ++z) {
                Z[(size_t)(par * nz + z)] = cz;
                cz += spacing / scale[2];
            }
        }
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return UPF_ERR_NO_DEVICE;
    const int nb = (int)((npts + MF_BLOCK - 1) / MF_BLOCK);
    // log2 extents of the boxes of 64 and 512 points: a cube bounds its faces
    // best; an axis with fewer points hands its share to the others
    Lattice lat = {{(int)nx, (int)ny, (int)nz}, {0, 0, 0}, {0, 0, 0}};
    for (int k = 0; k < 9; ++k) {
        int best = -1;
        for (int a = 2; a >= 0; --a)
            if (((lat.n[a] - 1) >> lat.bb[a]) && (best < 0 || lat.bb[a] < lat.bb[best])) best = a;
        ++lat.bb[best < 0 ? 2 : best];
        if (k == 5) std::copy(lat.bb, lat.bb + 3, lat.wb);
    }
    long long boxes = 1;
    for (int a = 0; a < 3; ++a) boxes *= ((lat.n[a] - 1) >> lat.bb[a]) + 1;
    // within these bounds no product of the interval tests overflows
    int cull = spacing <= 1e8f && X.back() <= 1e8f && Y[(size_t)ny - 1] <= 1e8f && Y.back() <= 1e8f &&
               Z[(size_t)nz - 1] <= 1e8f && Z.back() <= 1e8f;
    for (size_t k = 0; k < 9 * (size_t)n_faces; ++k) cull &= std::fabs(faces9[k]) <= 1e8f;
    Face* d_faces = nullptr;
    float *d_x = nullptr, *d_y = nullptr, *d_z = nullptr;
    uint8_t* d_keep = nullptr;
    int *d_counts = nullptr, *d_total = nullptr;
    float4* d_out = nullptr;
    hipStream_t st = nullptr;
    int rc = UPF_OK;
    auto ok = [&](hipError_t e) {
        if (e != hipSuccess && rc == UPF_OK) rc = UPF_ERR_HIP;
        return rc == UPF_OK;
    };
    int total = 0;
    if (ok(hipStreamCreateWithFlags(&st, hipStreamNonBlocking)) && ok(hipMalloc(&d_faces, faces.size() * sizeof(Face))) &&
        ok(hipMalloc(&d_x, X.size() * sizeof(float))) && ok(hipMalloc(&d_y, Y.size() * sizeof(float))) &&
        ok(hipMalloc(&d_z, Z.size() * sizeof(float))) && ok(hipMalloc(&d_keep, (size_t)npts)) &&
        ok(hipMalloc(&d_counts, (size_t)nb * sizeof(int))) && ok(hipMalloc(&d_total, sizeof(int))) &&
        ok(hipMemcpyAsync(d_faces, faces.data(), faces.size() * sizeof(Face), hipMemcpyHostToDevice, st)) &&
        ok(hipMemcpyAsync(d_x, X.data(), X.size() * sizeof(float), hipMemcpyHostToDevice, st)) &&
        ok(hipMemcpyAsync(d_y, Y.data(), Y.size() * sizeof(float), hipMemcpyHostToDevice, st)) &&
        ok(hipMemcpyAsync(d_z, Z.data(), Z.size() * sizeof(float), hipMemcpyHostToDevice, st))) {
        hipLaunchKernelGGL(k_mesh_test, dim3((unsigned)boxes), dim3(MT_BLOCK), 0, st, d_faces, n_faces, d_x, d_y, d_z,
                           lat, make_float3(o.x, o.y, o.z), cull, d_keep);
        hipLaunchKernelGGL(k_mesh_count, dim3(nb), dim3(MF_BLOCK), 0, st, d_keep, npts, d_counts);
        hipLaunchKernelGGL(k_mesh_scan, dim3(1), dim3(1024), 0, st, d_counts, nb, d_total);
        if (ok(hipGetLastError()) && ok(hipMemcpyAsync(&total, d_total, sizeof(int), hipMemcpyDeviceToHost, st)) &&
            ok(hipStreamSynchronize(st))) {
            *n_out = total;
            if (pos4 && cap < total) rc = UPF_ERR_RANGE;
            if (rc == UPF_OK && pos4 && total > 0 && ok(hipMalloc(&d_out, (size_t)total * sizeof(float4)))) {
                hipLaunchKernelGGL(k_mesh_emit, dim3(nb), dim3(MF_BLOCK), 0, st, d_keep, d_counts, d_x, d_y, d_z,
                                   (int)nx, (int)ny, (int)nz, make_float3(mn.x, mn.y, mn.z),
                                   make_float3(scale[0], scale[1], scale[2]), d_out, total);
                if (ok(hipGetLastError()))
                    ok(hipMemcpyAsync(pos4, d_out, (size_t)total * sizeof(float4), hipMemcpyDeviceToHost, st)) &&
                        ok(hipStreamSynchronize(st));
            }
        }
    }
    if (st) (void)hipStreamSynchronize(st);
    for (void* p : {(void*)d_faces, (void*)d_x, (void*)d_y, (void*)d_z, (void*)d_keep, (void*)d_counts,
                    (void*)d_total, (void*)d_out})
        if (p) (void)hipFree(p);
    if (st) (void)hipStreamDestroy(st);
    return rc;
}

}  // extern "C"
