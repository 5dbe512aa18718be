// Device build of a substrate (dsim_substrate_create_device, include/dsim.h):
// triangle records, the uniform grid as CSR with its cell-major copies and the
// per-cell clearance, computed on the GPU with the arithmetic of the host build
// (host.cpp) in the same order, so both builds give identical arrays.
//
//   k_tri_records   one thread per triangle: reference helpers
//                   (spinSystem.cpp:612-648), the 64-byte reference and
//                   Moller-Trumbore records, the bounding box
//   k_pairs<false>  per triangle, the number of cells it is listed in
//                   (reference grid: populateCubes' box test,
//                   spinSystem.cpp:1094-1352; AABB grid: box overlap)
//   exclusive scan  -> each triangle's first pair
//   k_pairs<true>   the (cell, triangle) pairs in triangle order, and the
//                   per-cell counts
//   radix sort      stable by cell: lists in ascending triangle order
//   exclusive scan  of the counts -> cell_start
//   k_ring_*        Chebyshev ring distance to the nearest occupied cell
//   k_clearance     the clearance of each cell
//   build_walk_tables  the walk's search lists and fine clearance (both builds)
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_reduce.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "../../include/dsim.h"
#include "host_common.h"
#include "tribox.h"

using dsim_host::DevBuf;
using dsim_host::fail;

namespace {

constexpr uint32_t kFar = 0xFFFFFFFFu;
constexpr uint32_t kBlock = 256;

__device__ __forceinline__ int64_t imin(int64_t a, int64_t b) { return a < b ? a : b; }
__device__ __forceinline__ int64_t imax(int64_t a, int64_t b) { return a > b ? a : b; }

struct Geom {
    uint32_t kind;
    uint32_t dims[3];
    float lo[3], cell[3];
    float eps;
    float L;  // reference grid: cube edge 2/n
    int64_t exact_rings;  // cells at ring distance <= this refine the clearance
};

struct F3 {
    float x, y, z;
};
__device__ __forceinline__ F3 f3(float x, float y, float z) { return F3{x, y, z}; }
__device__ __forceinline__ F3 operator-(F3 a, F3 b) { return f3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ F3 operator+(F3 a, F3 b) { return f3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ F3 operator*(F3 a, float s) { return f3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ float dotv(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// m_triangleHelpers, spinSystem.cpp:612-648.
__device__ void helpers_of(const float *V, const uint32_t *T, float *h) {
    const uint32_t p1 = T[0], p2 = T[1], p3 = T[2];
    const float x1 = V[p1 * 3 + 0], y1 = V[p1 * 3 + 1], z1 = V[p1 * 3 + 2];
    const float x2 = V[p2 * 3 + 0], y2 = V[p2 * 3 + 1], z2 = V[p2 * 3 + 2];
    const float x3 = V[p3 * 3 + 0], y3 = V[p3 * 3 + 1], z3 = V[p3 * 3 + 2];
    const float nx = (y2 - y1) * (z3 - z1) - (z2 - z1) * (y3 - y1);
    const float ny = (z2 - z1) * (x3 - x1) - (x2 - x1) * (z3 - z1);
    const float nz = (x2 - x1) * (y3 - y1) - (y2 - y1) * (x3 - x1);
    const float len = sqrtf(nx * nx + ny * ny + nz * nz);
    h[0] = nx / len; h[1] = ny / len; h[2] = nz / len;
    h[3] = x3 - x1; h[4] = y3 - y1; h[5] = z3 - z1;
    h[6] = x2 - x1; h[7] = y2 - y1; h[8] = z2 - z1;
    h[9] = (x3 - x1) * (x2 - x1) + (y3 - y1) * (y2 - y1) + (z3 - z1) * (z2 - z1);
    h[10] = (x3 - x1) * (x3 - x1) + (y3 - y1) * (y3 - y1) + (z3 - z1) * (z3 - z1);
    h[11] = (x2 - x1) * (x2 - x1) + (y2 - y1) * (y2 - y1) + (z2 - z1) * (z2 - z1);
}

__global__ __launch_bounds__(kBlock) void k_tri_records(uint32_t n_tri, const float *V,
                                                        const uint32_t *T, const uint32_t *info3,
                                                        float *helpers, float4 *ref, float4 *mt,
                                                        float4 *box) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n_tri) return;
    float h[12];
    helpers_of(V, T + (size_t)t * 3, h);
    for (int k = 0; k < 12; ++k) helpers[(size_t)t * 12 + k] = h[k];
    const uint32_t info = (info3[t * 3] & 0xFFFFu) | (info3[t * 3 + 1] << 16);
    const uint32_t P1 = info3[t * 3 + 2];
    ref[t * 4 + 0] = make_float4(h[0], h[1], h[2], h[3]);
    ref[t * 4 + 1] = make_float4(h[4], h[5], h[6], h[7]);
    ref[t * 4 + 2] = make_float4(h[8], h[9], h[10], h[11]);
    ref[t * 4 + 3] = make_float4(V[P1 * 3], V[P1 * 3 + 1], V[P1 * 3 + 2], __uint_as_float(info));
    const uint32_t a = T[t * 3], b = T[t * 3 + 1], c = T[t * 3 + 2];
    const float v0x = V[a * 3], v0y = V[a * 3 + 1], v0z = V[a * 3 + 2];
    const float nd = fmaf(h[0], v0x, fmaf(h[1], v0y, h[2] * v0z));
    mt[t * 4 + 0] = make_float4(h[0], h[1], h[2], nd);
    mt[t * 4 + 1] = make_float4(v0x, v0y, v0z, __uint_as_float(info));
    const float e1x = V[b * 3] - v0x, e1y = V[b * 3 + 1] - v0y, e1z = V[b * 3 + 2] - v0z;
    const float e2x = V[c * 3] - v0x, e2y = V[c * 3 + 1] - v0y, e2z = V[c * 3 + 2] - v0z;
    const float cx = fmaf(e1y, e2z, -(e1z * e2y));
    const float cy = fmaf(e1z, e2x, -(e1x * e2z));
    const float cz = fmaf(e1x, e2y, -(e1y * e2x));
    const float graze = 1e-6f * fmaf(cx, cx, fmaf(cy, cy, cz * cz));
    mt[t * 4 + 2] = make_float4(e1x, e1y, e1z, graze);
    mt[t * 4 + 3] = make_float4(e2x, e2y, e2z, 0.f);
    float mn[3], mx[3];
    for (int k = 0; k < 3; ++k) {
        const float p = V[a * 3 + k], q = V[b * 3 + k], r = V[c * 3 + k];
        mn[k] = p; if (q < mn[k]) mn[k] = q; if (r < mn[k]) mn[k] = r;
        mx[k] = p; if (q > mx[k]) mx[k] = q; if (r > mx[k]) mx[k] = r;
    }
    box[t * 2 + 0] = make_float4(mn[0], mn[1], mn[2], __uint_as_float(info));
    box[t * 2 + 1] = make_float4(mx[0], mx[1], mx[2], 0.f);
}

// ---- reference grid membership (populateCubes, spinSystem.cpp:1094-1379) ----

__device__ __forceinline__ bool point_in_box(F3 p, F3 mn, F3 mx) {
    return ((p.x <= mx.x) && (p.x >= mn.x)) && ((p.y <= mx.y) && (p.y >= mn.y)) &&
           ((p.z <= mx.z) && (p.z >= mn.z));
}

// rayTriangleIntersect, spinSystem.cpp:1360-1379.
__device__ bool segment_hits_triangle(F3 r1, F3 r2, F3 t1, F3 t2, F3 t3) {
    const F3 u = t2 - t1, v = t3 - t1;
    F3 n = f3(u.y * v.z - u.z * v.y, u.z * v.x - u.x * v.z, u.x * v.y - u.y * v.x);
    const float nl = sqrtf(n.x * n.x + n.y * n.y + n.z * n.z);
    float s = 2.0f, t = 2.0f;
    n.x = n.x / nl; n.y = n.y / nl; n.z = n.z / nl;
    const float r = dotv(n, t1 - r1) / dotv(n, r2 - r1);
    if ((0 < r) & (r < 1)) {
        const F3 w = (r1 + (r2 - r1) * r) - t1;
        const float uv = dotv(u, v), wv = dotv(w, v), vv = dotv(v, v), wu = dotv(w, u),
                    uu = dotv(u, u);
        s = (uv * wv - vv * wu) / (uv * uv - uu * vv);
        t = (uv * wu - uu * wv) / (uv * uv - uu * vv);
    }
    return (s >= 0) && (t >= 0) && (s + t <= 1);
}

// Corner c of a box: bit 0 picks max x, bit 1 max y, bit 2 max z; edges and
// faces in the argument order of spinSystem.cpp:1189-1244.
__device__ __forceinline__ F3 corner(F3 mn, F3 mx, int c) {
    return f3((c & 1) ? mx.x : mn.x, (c & 2) ? mx.y : mn.y, (c & 4) ? mx.z : mn.z);
}
__constant__ int kBoxEdges[12][2] = {{0, 1}, {0, 2}, {0, 4}, {6, 2}, {6, 4}, {6, 7},
                                     {3, 2}, {3, 1}, {3, 7}, {5, 7}, {5, 1}, {5, 4}};
__constant__ int kBoxFaces[12][3] = {{0, 1, 2}, {0, 4, 2}, {0, 4, 1}, {6, 2, 4},
                                     {6, 2, 7}, {6, 4, 7}, {3, 2, 1}, {3, 7, 1},
                                     {3, 7, 2}, {5, 4, 7}, {5, 1, 7}, {5, 4, 1}};

__device__ bool triangle_in_box(F3 p1, F3 p2, F3 p3, F3 mn, F3 mx) {
    if (point_in_box(p1, mn, mx) || point_in_box(p2, mn, mx) || point_in_box(p3, mn, mx))
        return true;
    for (int e = 0; e < 12; ++e)
        if (segment_hits_triangle(corner(mn, mx, kBoxEdges[e][0]), corner(mn, mx, kBoxEdges[e][1]),
                                  p1, p2, p3))
            return true;
    const F3 a[3] = {p1, p1, p2}, b[3] = {p2, p3, p3};
    for (int s = 0; s < 3; ++s)
        for (int f = 0; f < 12; ++f)
            if (segment_hits_triangle(a[s], b[s], corner(mn, mx, kBoxFaces[f][0]),
                                      corner(mn, mx, kBoxFaces[f][1]),
                                      corner(mn, mx, kBoxFaces[f][2])))
                return true;
    return false;
}

// calcCubePos with the reference's division and min/max clamp.
__device__ __forceinline__ uint32_t ref_cell(float p, float lo, float cell, uint32_t n) {
    const float q = floorf((p - lo) / cell);
    const float hi = (float)(n - 1);
    const float mn = (hi < q) ? hi : q;
    const float mx = (0.0f < mn) ? mn : 0.0f;
    return (uint32_t)mx;
}

// Lanes that take a triangle's cells together.
constexpr uint32_t kPairLanes = 16;

// The cells that list triangle t, shared out over kPairLanes lanes: calls
// fn(cell, listed) on every lane the same number of times.
template <class Fn>
__device__ void cells_of(const Geom &g, const float *V, const uint32_t *T, uint32_t t, uint32_t lane,
                         Fn fn) {
    if (g.kind == DSIM_GRID_REFERENCE) {
        const uint32_t n = g.dims[0];
        const float L = g.L;
        F3 p[3];
        for (int j = 0; j < 3; ++j) {
            const uint32_t vi = T[t * 3 + j];
            p[j] = f3(V[vi * 3], V[vi * 3 + 1], V[vi * 3 + 2]);
        }
        F3 mn = p[0], mx = p[0];
        if (p[1].x < mn.x) mn.x = p[1].x; if (p[2].x < mn.x) mn.x = p[2].x;
        if (p[1].y < mn.y) mn.y = p[1].y; if (p[2].y < mn.y) mn.y = p[2].y;
        if (p[1].z < mn.z) mn.z = p[1].z; if (p[2].z < mn.z) mn.z = p[2].z;
        if (p[1].x > mx.x) mx.x = p[1].x; if (p[2].x > mx.x) mx.x = p[2].x;
        if (p[1].y > mx.y) mx.y = p[1].y; if (p[2].y > mx.y) mx.y = p[2].y;
        if (p[1].z > mx.z) mx.z = p[1].z; if (p[2].z > mx.z) mx.z = p[2].z;
        const uint32_t c0[3] = {ref_cell(mn.x, -1.0f, L, n), ref_cell(mn.y, -1.0f, L, n),
                                ref_cell(mn.z, -1.0f, L, n)};
        const uint32_t c1[3] = {ref_cell(mx.x, -1.0f, L, n), ref_cell(mx.y, -1.0f, L, n),
                                ref_cell(mx.z, -1.0f, L, n)};
        if (c1[0] < c0[0] || c1[1] < c0[1] || c1[2] < c0[2]) return;
        // at most 1024^3 cells
        const uint32_t ny = c1[1] - c0[1] + 1, nz = c1[2] - c0[2] + 1;
        const uint32_t all = (c1[0] - c0[0] + 1) * ny * nz;
        for (uint32_t i0 = 0; i0 < all; i0 += kPairLanes) {
            const uint32_t i = i0 + lane;
            const uint32_t zc = c0[2] + i % nz, yc = c0[1] + i / nz % ny, xc = c0[0] + i / nz / ny;
            const F3 bmin = f3(-1 + (float)xc * L, -1 + (float)yc * L, -1 + (float)zc * L);
            const F3 bmax = f3(-1 + (float)(xc + 1) * L, -1 + (float)(yc + 1) * L,
                               -1 + (float)(zc + 1) * L);
            fn((zc * n + yc) * n + xc,
               i < all && triangle_in_box(p[0], p[1], p[2], bmin, bmax));
        }
        return;
    }
    float mn[3], mx[3];
    int64_t i0[3], i1[3];
    double v[3][3];
    for (int k = 0; k < 3; ++k) {
        const float a = V[T[t * 3] * 3 + k], b = V[T[t * 3 + 1] * 3 + k],
                    c = V[T[t * 3 + 2] * 3 + k];
        v[0][k] = a; v[1][k] = b; v[2][k] = c;
        mn[k] = a; if (b < mn[k]) mn[k] = b; if (c < mn[k]) mn[k] = c;
        mx[k] = a; if (b > mx[k]) mx[k] = b; if (c > mx[k]) mx[k] = c;
        mn[k] = mn[k] - g.eps; mx[k] = mx[k] + g.eps;
        i0[k] = (int64_t)floorf((mn[k] - g.lo[k]) / g.cell[k]) - 1;
        i1[k] = (int64_t)floorf((mx[k] - g.lo[k]) / g.cell[k]) + 1;
        if (i0[k] < 0) i0[k] = 0;
        if (i1[k] > (int64_t)g.dims[k] - 1) i1[k] = (int64_t)g.dims[k] - 1;
        if (i0[k] > i1[k]) return;
    }
    const uint32_t nx = (uint32_t)(i1[0] - i0[0] + 1), ny = (uint32_t)(i1[1] - i0[1] + 1);
    const uint32_t all = nx * ny * (uint32_t)(i1[2] - i0[2] + 1);  // at most the grid's 2^28
    for (uint32_t q0 = 0; q0 < all; q0 += kPairLanes) {
        const uint32_t q = q0 + lane;
        const int64_t idx[3] = {i0[0] + q % nx, i0[1] + q / nx % ny, i0[2] + q / nx / ny};
        bool in = q < all;
        for (int k = 0; k < 3; ++k) {
            const float b0 = g.lo[k] + (float)idx[k] * g.cell[k],
                        b1 = g.lo[k] + (float)(idx[k] + 1) * g.cell[k];
            if (b0 > mx[k] || mn[k] > b1) in = false;
        }
        if (in && g.kind == DSIM_GRID_TRIBOX) {
            // exact membership: host.cpp tri_cell_separated
            double b0[3], b1[3];
            for (int k = 0; k < 3; ++k) {
                b0[k] = (double)g.lo[k] + (double)idx[k] * (double)g.cell[k];
                b1[k] = (double)g.lo[k] + (double)(idx[k] + 1) * (double)g.cell[k];
            }
            dsim_host::TriBoxAxes X;
            dsim_host::tribox_setup(v[0], v[1], v[2], b0, b1, X);
            in = !dsim_host::tribox_separated(X, (double)g.eps);
        }
        fn((uint32_t)((idx[2] * g.dims[1] + idx[1]) * g.dims[0] + idx[0]), in);
    }
}

// EMIT false: count[t] = pairs of triangle t.  EMIT true: the pairs of t at
// offset[t] (cell keys, triangle values; a stable sort by cell follows, so
// their order here does not matter) and the per-cell counts.  kPairLanes lanes
// take a triangle's cells together: a wall that spans a voxel overlaps
// thousands of cells, and one lane a triangle left most of the device idle
// (24,768 triangles, 100 x 240 x 100 cells: 5.8 and 5.1 ms, 22 and 31 before; a
// reference grid of 50^3 cells 0.35 ms each, 8 and 9).
template <bool EMIT>
__global__ __launch_bounds__(kBlock) void k_pairs(Geom g, uint32_t n_tri, const float *V,
                                                  const uint32_t *T, uint32_t *count_or_offset,
                                                  uint32_t *keys, uint32_t *vals,
                                                  uint32_t *cell_count) {
    const uint32_t t = (uint32_t)(((uint64_t)blockIdx.x * kBlock + threadIdx.x) / kPairLanes);
    if (t >= n_tri) return;
    const uint32_t lane = threadIdx.x % kPairLanes;
    const uint32_t shift = threadIdx.x % 64u / kPairLanes * kPairLanes;
    constexpr uint32_t mask = (1u << kPairLanes) - 1u;
    uint32_t o = EMIT ? count_or_offset[t] : 0u;
    cells_of(g, V, T, t, lane, [&](uint32_t c, bool listed) {
        const uint32_t m = (uint32_t)(__ballot(listed) >> shift) & mask;  // of this triangle
        if (EMIT && listed) {
            const uint32_t at = o + (uint32_t)__popc(m & ((1u << lane) - 1u));
            keys[at] = c;
            vals[at] = t;
            atomicAdd(&cell_count[c], 1u);
        }
        o += (uint32_t)__popc(m);
    });
    if (!EMIT && lane == 0) count_or_offset[t] = o;
}

__global__ __launch_bounds__(kBlock) void k_ring_init(uint32_t n_cells, const uint32_t *start,
                                                      uint32_t *ring) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= n_cells) return;
    ring[c] = start[c + 1] > start[c] ? 0u : kFar;
}

// Cells still unreached that touch (26-neighbourhood) a cell of ring r-1 get
// ring r: after step r every ring value up to r is final.
__global__ __launch_bounds__(kBlock) void k_ring_step(uint32_t dx, uint32_t dy, uint32_t dz,
                                                      uint32_t *ring, uint32_t r,
                                                      uint32_t *changed) {
    const uint64_t c = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c >= (uint64_t)dx * dy * dz) return;
    if (ring[c] != kFar) return;
    const int64_t ix = c % dx, iy = (c / dx) % dy, iz = c / ((uint64_t)dx * dy);
    for (int64_t z = imax(0, iz - 1); z <= imin((int64_t)dz - 1, iz + 1); ++z)
        for (int64_t y = imax(0, iy - 1); y <= imin((int64_t)dy - 1, iy + 1); ++y)
            for (int64_t x = imax(0, ix - 1); x <= imin((int64_t)dx - 1, ix + 1); ++x)
                if (ring[((uint64_t)z * dy + y) * dx + x] == r - 1) {
                    ring[c] = r;
                    *changed = 1u;
                    return;
                }
}

// The largest float whose square is at most x >= 0.
__device__ float float_sqrt_floor(double x) {
    if (!(x >= 0.0)) return 0.0f;
    float f = (float)sqrt(x);
    while (f > 0.0f && (double)f * (double)f > x) f = nextafterf(f, 0.0f);
    for (;;) {
        const float g = nextafterf(f, 3.0e38f);
        if ((double)g * (double)g > x) break;
        f = g;
    }
    return f;
}

// Clearance of each cell, as compute_clearance in host.cpp: from the ring
// distance alone beyond g.exact_rings, else the smallest box-to-box distance to
// the triangles of the rings around the cell.
__global__ __launch_bounds__(kBlock) void k_clearance(Geom g, const uint32_t *ring,
                                                      const uint32_t *start, const uint32_t *tri,
                                                      const float4 *box, const float *V,
                                                      const uint32_t *T, float *out) {
    const int64_t D[3] = {g.dims[0], g.dims[1], g.dims[2]};
    const uint64_t c = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c >= (uint64_t)D[0] * D[1] * D[2]) return;
    const uint32_t rc = ring[c];
    if (rc == kFar) { out[c] = 1e30f; return; }
    double hmin = (double)g.cell[0];
    if ((double)g.cell[1] < hmin) hmin = (double)g.cell[1];
    if ((double)g.cell[2] < hmin) hmin = (double)g.cell[2];
    if ((int64_t)rc > g.exact_rings) {
        // an occupied cell (ring 0) has no clearance
        const double best = rc > 0 ? (double)(rc - 1) * hmin : 0.0;
        float f = (float)best;
        if ((double)f > best) f = nextafterf(f, 0.0f);
        out[c] = f;
        return;
    }
    const int64_t ix = c % D[0], iy = (c / D[0]) % D[1], iz = c / ((uint64_t)D[0] * D[1]);
    const int64_t idx[3] = {ix, iy, iz};
    double b0[3], b1[3];
    for (int k = 0; k < 3; ++k) {
        b0[k] = (double)g.lo[k] + (double)idx[k] * g.cell[k];
        b1[k] = b0[k] + g.cell[k];
    }
    double best2 = 1e60;
    for (int64_t r = rc;; ++r) {
        if (r > 0) {
            const double q = (double)(r - 1) * hmin;
            if (q * q >= best2) break;
        }
        if (r > D[0] && r > D[1] && r > D[2]) break;
        for (int64_t z = imax(0, iz - r); z <= imin(D[2] - 1, iz + r); ++z)
            for (int64_t y = imax(0, iy - r); y <= imin(D[1] - 1, iy + r); ++y)
                for (int64_t x = imax(0, ix - r); x <= imin(D[0] - 1, ix + r); ++x) {
                    const int64_t ax = x > ix ? x - ix : ix - x, ay = y > iy ? y - iy : iy - y,
                                  az = z > iz ? z - iz : iz - z;
                    if (imax(imax(ax, ay), az) != r) continue;  // the ring at radius r only
                    const uint64_t cc = ((uint64_t)z * D[1] + y) * D[0] + x;
                    for (uint32_t k = start[cc]; k < start[cc + 1] && best2 > 0.0; ++k) {
                        double d2 = 0;
                        if (g.kind == DSIM_GRID_TRIBOX) {
                            // host.cpp: the largest separating-axis gap
                            const uint32_t t = tri[k];
                            double a[3], b[3], c[3];
                            for (int q = 0; q < 3; ++q) {
                                a[q] = V[T[t * 3] * 3 + q];
                                b[q] = V[T[t * 3 + 1] * 3 + q];
                                c[q] = V[T[t * 3 + 2] * 3 + q];
                            }
                            dsim_host::TriBoxAxes X;
                            dsim_host::tribox_setup(a, b, c, b0, b1, X);
                            d2 = dsim_host::tribox_gap2(X, best2);
                        } else {
                            const float4 a = box[(size_t)tri[k] * 2], b = box[(size_t)tri[k] * 2 + 1];
                            const double lo3[3] = {a.x, a.y, a.z}, hi3[3] = {b.x, b.y, b.z};
                            for (int q = 0; q < 3; ++q) {
                                double gap = 0.0;
                                if (lo3[q] - b1[q] > gap) gap = lo3[q] - b1[q];
                                if (b0[q] - hi3[q] > gap) gap = b0[q] - hi3[q];
                                d2 += gap * gap;
                            }
                        }
                        if (d2 < best2) best2 = d2;
                    }
                }
    }
    out[c] = float_sqrt_floor(best2);
}

// Fine clearance: the walk completes a step from o to p without a search when
// the clearances of the fine cells of o and p add up to more than the step's
// length (the two balls cover the segment).  Each byte is the distance from
// its fine cell to the nearest triangle of the grid, rounded down to a
// multiple of q after taking off the margin for the walk's float arithmetic.
//
// The distance comes from the exact point-triangle distance of the cell's
// centre, less the cell's half diagonal, over the triangles listed in the 3^k
// grid cells around it (a triangle listed in none of them is no nearer than
// the edge of that block), or from the grid's own clearance where that is
// larger.  On an axis of one cell every distance is taken in the projection
// along it: the bound then holds whatever the coordinate on that axis, and a
// step's length leaves the axis out.
struct FineGeom {
    uint32_t sub[3];    // fine cells per grid cell and axis (1 on collapsed axes)
    uint32_t dims[3];   // fine cells per axis
    float cell[3];      // fine cell edge
    float w[3];         // 0 on collapsed axes
    float half_diag, q;
    float margin;       // kFineMargin for the substrate's coordinates
};
// Covers FP32 rounding of positions, distances and lookups at coordinates up to
// 2 (times the substrate's margin_scale beyond).
constexpr float kFineMargin = 1e-5f;
constexpr float kFineRange = 32.0f;   // q = grid cell / kFineRange: bytes reach 8 grid cells

struct D3 {
    double x, y, z;
};
__device__ __forceinline__ D3 operator-(D3 a, D3 b) { return D3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ double dotv(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ D3 cross3(D3 a, D3 b) {
    return D3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
// Squared distance of r (point - a) from the segment a + t e.
__device__ __forceinline__ double seg_dist2(D3 r, D3 e) {
    const double ee = dotv(e, e);
    const double t = ee > 0.0 ? fmin(fmax(dotv(r, e) / ee, 0.0), 1.0) : 0.0;
    const D3 d = D3{r.x - t * e.x, r.y - t * e.y, r.z - t * e.z};
    return dotv(d, d);
}

// Squared distance of point c from the triangle with record m, in the
// projection w: the nearest of the three edges, or the plane's where the
// point projects into the triangle or within the margin of it.  In double and
// from the edges the walk tests (the normal of a long thin triangle is off by
// more than the margin in FP32); a degenerate triangle is its edges.
// A triangle whose plane is farther than sqrt(enough) gives `enough`.
__device__ double tri_dist2(const float4 *__restrict__ m, D3 c, D3 w, double enough, float margin) {
    const float4 v4 = m[1], a4 = m[2], b4 = m[3];
    const D3 e1 = D3{a4.x * w.x, a4.y * w.y, a4.z * w.z};
    const D3 e2 = D3{b4.x * w.x, b4.y * w.y, b4.z * w.z};
    const D3 r = D3{(c.x - v4.x) * w.x, (c.y - v4.y) * w.y, (c.z - v4.z) * w.z};
    const D3 n = cross3(e1, e2);
    const double nn = dotv(n, n), h = dotv(n, r);
    // (not a sliver's, whose plane is uncertain)
    if (h * h > 1.0001 * enough * nn && nn > 1e-12 * dotv(e1, e1) * dotv(e2, e2)) return enough;
    const D3 e3 = e2 - e1, r1 = r - e1;
    double d2 = fmin(fmin(seg_dist2(r, e1), seg_dist2(r, e2)), seg_dist2(r1, e3));
    if (nn > 0.0) {
        const double k = -(double)margin * sqrt(nn);
        if (dotv(n, cross3(e1, r)) >= k * sqrt(dotv(e1, e1)) &&
            dotv(n, cross3(r, e2)) >= k * sqrt(dotv(e2, e2)) &&
            dotv(n, cross3(e3, r1)) >= k * sqrt(dotv(e3, e3))) {
            d2 = fmin(d2, h * h / nn);
        }
    }
    return d2;
}

__global__ __launch_bounds__(kBlock) void k_fine_clearance(Geom g, FineGeom f,
                                                           const uint32_t *__restrict__ start,
                                                           const uint32_t *__restrict__ tri,
                                                           const float4 *__restrict__ mt,
                                                           const float *__restrict__ coarse,
                                                           uint8_t *__restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= (uint64_t)f.dims[0] * f.dims[1] * f.dims[2]) return;
    const uint32_t fx = (uint32_t)(i % f.dims[0]), fy = (uint32_t)(i / f.dims[0] % f.dims[1]),
                   fz = (uint32_t)(i / ((uint64_t)f.dims[0] * f.dims[1]));
    const uint32_t fi[3] = {fx, fy, fz};
    int32_t c[3], a0[3], a1[3];
    float edge = 3.0e38f, ctr[3];
    bool inner = true;
    for (int k = 0; k < 3; ++k) {
        c[k] = (int32_t)(fi[k] / f.sub[k]);
        ctr[k] = g.lo[k] + ((float)fi[k] + 0.5f) * f.cell[k];
        a0[k] = a1[k] = c[k];
        if (f.w[k] == 0.0f) continue;
        // the block of neighbours lies in the grid; its faces are one grid
        // cell and the fine cell's offset away
        inner &= c[k] > 0 && c[k] + 1 < (int32_t)g.dims[k];
        a0[k] = c[k] - 1; a1[k] = c[k] + 1;
        const uint32_t o = fi[k] % f.sub[k];
        edge = fminf(edge, g.cell[k] + (float)min(o, f.sub[k] - 1 - o) * f.cell[k]);
    }
    double d = coarse[((uint64_t)c[2] * g.dims[1] + c[1]) * g.dims[0] + c[0]];
    if (inner && d < edge) {
        const double reach = (double)edge + f.half_diag;
        double d2 = reach * reach;
        const D3 p = D3{ctr[0], ctr[1], ctr[2]}, w = D3{f.w[0], f.w[1], f.w[2]};
        for (int32_t z = a0[2]; z <= a1[2]; ++z)
            for (int32_t y = a0[1]; y <= a1[1]; ++y) {
                // the cells of a row are consecutive, and so are their entries
                const uint64_t row = ((uint64_t)z * g.dims[1] + y) * g.dims[0];
                const uint32_t k1 = start[row + a1[0] + 1];
                for (uint32_t k = start[row + a0[0]]; k < k1; ++k)
                    d2 = fmin(d2, tri_dist2(mt + (size_t)tri[k] * 4, p, w, d2, f.margin));
            }
        d = fmax(d, sqrt(d2) - f.half_diag);
    }
    out[i] = (uint8_t)fmin(fmax(floor((d - f.margin) / f.q), 0.0), 255.0);
}

// ---- search lists of the walk ---------------------------------------------- //
// A wall facet is two triangles of one plane (equal records), so a search that lists them as one entry tests half the planes.  And
// most planes a segment crosses it crosses beyond the facet (a wall's
// neighbouring facets are nearly one plane): the lateral record bounds the
// facet across its narrow direction, and rejects those before the triangle
// test.

constexpr uint32_t kNoTri = 0xFFFFFFFFu;

// Sort key of triangle t: a hash of its plane and first vertex, whose equality
// k_pair_triangles checks on the full records.
__device__ __forceinline__ uint64_t mix64(uint64_t h, uint32_t v) {
    h = (h ^ v) * 0x9E3779B97F4A7C15ull;
    return h ^ (h >> 29);
}
__global__ __launch_bounds__(kBlock) void k_plane_keys(uint32_t n_tri, const float4 *mt,
                                                       uint64_t *keys, uint32_t *vals) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n_tri) return;
    const float4 a = mt[(size_t)t * 4], v = mt[(size_t)t * 4 + 1];
    const float f[7] = {a.x, a.y, a.z, a.w, v.x, v.y, v.z};
    uint64_t h = 1;
    for (int k = 0; k < 7; ++k) h = mix64(h, __float_as_uint(f[k] + 0.0f));  // -0 as +0
    keys[t] = h;
    vals[t] = t;
}

// Pairs the triangles of each run of equal keys two by two, in ascending
// order (the sort is stable), where their planes are equal: every side test
// then gives one result for both.
__global__ __launch_bounds__(kBlock) void k_pair_triangles(uint32_t n_tri, const uint64_t *keys,
                                                           const uint32_t *vals, const float4 *mt,
                                                           uint32_t *partner) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n_tri || (i > 0 && keys[i] == keys[i - 1])) return;  // the run's first thread
    uint32_t k = i;
    while (k < n_tri && keys[k] == keys[i]) {
        const uint32_t t = vals[k];
        partner[t] = kNoTri;
        if (k + 1 < n_tri && keys[k + 1] == keys[i]) {
            const uint32_t u = vals[k + 1];
            const float4 p = mt[(size_t)t * 4], q = mt[(size_t)u * 4];
            if (p.x == q.x && p.y == q.y && p.z == q.z && p.w == q.w) {
                partner[t] = u;
                partner[u] = t;
                k += 2;
                continue;
            }
        }
        ++k;
    }
}

// Records of triangle t and its partner: the plane, and the lateral record
// (d / W, m / W) with d the unit vector in the plane across the triangle's
// longest edge and [m - W, m + W] the extent of both along d, widened by
// kFineMargin (margins times); (0, 0, 0, 0), which bounds nothing, for a
// degenerate triangle.
// eps: the largest distance of a vertex from its own record's plane.
__global__ __launch_bounds__(kBlock) void k_walk_records(uint32_t n_tri, const float4 *mt,
                                                         const uint32_t *partner, float margins,
                                                         float4 *rec, uint32_t *eps) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n_tri) return;
    const float4 pl = mt[(size_t)t * 4];
    double lo = 0, hi = 0, dev = 0;
    D3 d = D3{0, 0, 0};
    uint32_t u = t;
    for (int q = 0; q < 2; ++q) {
        const float4 v4 = mt[(size_t)u * 4 + 1], a4 = mt[(size_t)u * 4 + 2],
                     b4 = mt[(size_t)u * 4 + 3];
        const D3 v0 = D3{v4.x, v4.y, v4.z}, e1 = D3{a4.x, a4.y, a4.z}, e2 = D3{b4.x, b4.y, b4.z};
        const D3 e3 = e2 - e1;
        if (q == 0) {
            const double l1 = dotv(e1, e1), l2 = dotv(e2, e2), l3 = dotv(e3, e3);
            const D3 l = l1 >= l2 && l1 >= l3 ? e1 : l2 >= l3 ? e2 : e3;
            d = cross3(cross3(e1, e2), l);
            const double n = sqrt(dotv(d, d));
            d = n > 0.0 ? D3{d.x / n, d.y / n, d.z / n} : D3{0, 0, 0};
            lo = hi = dotv(d, v0);
        }
        const double c0 = dotv(d, v0), c1 = c0 + dotv(d, e1), c2 = c0 + dotv(d, e2);
        lo = fmin(lo, fmin(c0, fmin(c1, c2)));
        hi = fmax(hi, fmax(c0, fmax(c1, c2)));
        const D3 n = D3{pl.x, pl.y, pl.z};
        const double s0 = dotv(n, v0) - (double)pl.w;
        dev = fmax(dev, fmax(fabs(s0), fmax(fabs(s0 + dotv(n, e1)), fabs(s0 + dotv(n, e2)))));
        u = partner[t];
        if (u == kNoTri) break;
    }
    const double W = 0.5 * (hi - lo) + (double)kFineMargin * margins, m = 0.5 * (hi + lo);
    // false for a degenerate or NaN triangle, or one off its own plane
    const bool ok = dotv(d, d) > 0.5 && W < 1e30 && dev < margins;
    rec[(size_t)t * 2] = pl;
    rec[(size_t)t * 2 + 1] = ok ? make_float4((float)(d.x / W), (float)(d.y / W), (float)(d.z / W),
                                              (float)(m / W))
                                : make_float4(0.f, 0.f, 0.f, 0.f);
    if (ok) atomicMax(eps, __float_as_uint((float)dev));
}

// Reference mode: per list entry the triangle's normal and its first vertex
// with the triangle's index.
__global__ __launch_bounds__(kBlock) void k_ref_records(uint32_t n, const uint32_t *tri,
                                                        const float4 *ref, float4 *rec) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= n) return;
    const uint32_t t = tri[k];
    const float4 a = ref[(size_t)t * 4], d = ref[(size_t)t * 4 + 3];
    rec[(size_t)k * 2] = make_float4(a.x, a.y, a.z, 0.f);
    rec[(size_t)k * 2 + 1] = make_float4(d.x, d.y, d.z, __uint_as_float(t));
}

// StepParams::ref_mask of each cell; boxes reach no further than the grid.
__global__ __launch_bounds__(kBlock) void k_ref_masks(uint32_t dx, uint32_t dy, uint32_t dz,
                                                      const uint32_t *start, uint32_t *mask) {
    const uint64_t c = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (c >= (uint64_t)dx * dy * dz) return;
    const int x = (int)(c % dx), y = (int)(c / dx % dy), z = (int)(c / ((uint64_t)dx * dy));
    uint32_t listed = 0, m = 0;  // same bit order
    for (int k = 0; k < 27; ++k) {
        const int qx = x + k % 3 - 1, qy = y + k / 3 % 3 - 1, qz = z + k / 9 - 1;
        if (qx < 0 || qy < 0 || qz < 0 || qx >= (int)dx || qy >= (int)dy || qz >= (int)dz) continue;
        const uint64_t q = ((uint64_t)qz * dy + qy) * dx + qx;
        if (start[q + 1] > start[q]) listed |= 1u << k;
    }
    for (int k = 0; k < 27; ++k) {
        const int ex = k % 3 - 1, ey = k / 3 % 3 - 1, ez = k / 9 - 1;
        bool any = false;
        for (int b = 0; b < 8; ++b) {
            const int bx = b & 1 ? ex : 0, by = b & 2 ? ey : 0, bz = b & 4 ? ez : 0;
            any |= (listed >> ((bx + 1) + 3 * (by + 1) + 9 * (bz + 1))) & 1u;
        }
        if (any) m |= 1u << k;
    }
    mask[c] = m;
}

// Place of triangle t in the ascending list [a, b), or b.
__device__ __forceinline__ uint32_t find_tri(const uint32_t *tri, uint32_t a, uint32_t b, uint32_t t) {
    const uint32_t end = b;
    while (a < b) {
        const uint32_t m = (a + b) >> 1;
        if (tri[m] < t) a = m + 1; else b = m;
    }
    return a < end && tri[a] == t ? a : end;
}

// Cells of a block's list builds go to its threads one each, those of more than
// kFewEntries to all of them together afterwards.  A grid of one cell, 60,000
// triangles: 78 ms a build with a thread over its list, 4.2 so (3584 triangles in
// pairs: 4.2 ms and 0.6); cells of a few entries are built as fast as before.
constexpr uint32_t kFewEntries = 64;
struct BigCells {
    uint32_t n, cell[kBlock], wave[kBlock / 64];
};
// Number of the block's threads before this one with `on`; `all` gets the block's.
__device__ __forceinline__ uint32_t block_rank(BigCells &B, bool on, uint32_t &all) {
    const unsigned long long m = __ballot(on);
    const uint32_t w = threadIdx.x / 64u, lane = threadIdx.x % 64u;
    __syncthreads();
    if (lane == 0) B.wave[w] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t r = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
    all = 0;
    for (uint32_t k = 0; k < kBlock / 64; ++k) {
        r += k < w ? B.wave[k] : 0u;
        all += B.wave[k];
    }
    return r;
}
// The entries [k0, k1) of `cell` by the whole block: keep(k) says whether one
// counts, put(place, k) writes it; done(end) closes the cell, on one thread.
template <class Keep, class Put, class Done>
__device__ __forceinline__ void by_block(BigCells &B, uint32_t k0, uint32_t k1, uint32_t first,
                                         Keep keep, Put put, Done done) {
    uint32_t n = first;
    for (uint32_t base = k0; base < k1; base += kBlock) {
        const uint32_t k = base + threadIdx.x;
        const bool on = k < k1 && k >= base && keep(k);
        uint32_t all;
        const uint32_t r = block_rank(B, on, all);
        if (on) put(n + r, k);
        n += all;
        if (base > 0xFFFFFFFFu - kBlock) break;
    }
    if (threadIdx.x == 0) done(n);
}

// Entries of cell c: EMIT false counts them, true writes them at start[c]
// (and their records, cell-major).  A triangle whose partner precedes it in
// the cell's list is that one's entry.
template <bool EMIT>
__global__ __launch_bounds__(kBlock) void k_walk_lists(uint32_t n_cells, const uint32_t *cell_start,
                                                       const uint32_t *cell_tri,
                                                       const uint32_t *partner, uint32_t *start,
                                                       uint2 *ent, const float4 *rec,
                                                       float4 *cell_rec) {
    __shared__ BigCells B;
    if (threadIdx.x == 0) B.n = 0;
    __syncthreads();
    // the partner of entry k where it is in the list too
    auto with = [&](uint32_t k0, uint32_t k1, uint32_t k) {
        const uint32_t u = partner[cell_tri[k]];
        return u != kNoTri && find_tri(cell_tri, k0, k1, u) != k1 ? u : kNoTri;
    };
    auto put = [&](uint32_t n, uint32_t t, uint32_t u) {
        ent[n] = make_uint2(t, u);
        if (cell_rec) {
            cell_rec[(size_t)n * 2] = rec[(size_t)t * 2];
            cell_rec[(size_t)n * 2 + 1] = rec[(size_t)t * 2 + 1];
        }
    };
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c < n_cells) {
        const uint32_t k0 = cell_start[c], k1 = cell_start[c + 1];
        if (k1 - k0 > kFewEntries) {
            B.cell[atomicAdd(&B.n, 1u)] = c;
        } else {
            uint32_t n = EMIT ? start[c] : 0u;
            for (uint32_t k = k0; k < k1; ++k) {
                const uint32_t t = cell_tri[k], u = with(k0, k1, k);
                if (u < t) continue;  // (kNoTri is the largest)
                if (EMIT) put(n, t, u);
                ++n;
            }
            if (!EMIT) start[c] = n;
        }
    }
    __syncthreads();
    for (uint32_t b = 0; b < B.n; ++b) {
        const uint32_t q = B.cell[b], k0 = cell_start[q], k1 = cell_start[q + 1];
        uint32_t t = 0, u = 0;
        by_block(
            B, k0, k1, EMIT ? start[q] : 0u,
            [&](uint32_t k) {
                t = cell_tri[k];
                u = with(k0, k1, k);
                return u >= t;
            },
            [&](uint32_t n, uint32_t) { if (EMIT) put(n, t, u); },
            [&](uint32_t n) { if (!EMIT) start[q] = n; });
    }
}

// The labeller's rows: the grid's cells along axis A, rows by the two other
// axes (B, then C), and what decides whether a triangle is listed in them.
struct RowGeom {
    uint32_t dims[3];
    float lo[3], cell[3];
    int A, B, C;
    float face;  // the grid's far face on A
    bool exact;
};

// Does the triangle stand at the ends of rows rather than where their cells
// list it?  AABB grids: its box starts past the grid's face on the ray's side
// (no row lists it in a cell the ray can reach).  Exact-membership grids: its
// box reaches past that face (the ray may cross it beyond the grid, where no
// row cell lists it).
__device__ __forceinline__ bool past_grid(const RowGeom &g, const float4 *box, uint32_t t) {
    const float4 v = box[2 * (size_t)t + (g.exact ? 1 : 0)];
    return (g.A == 0 ? v.x : g.A == 1 ? v.y : v.z) > g.face;
}

// A row entry's extents on the axes across (LabelParams::row_box).
__device__ __forceinline__ float4 row_extent(const RowGeom &g, const float4 *box, uint32_t t) {
    const float4 lo = box[2 * (size_t)t], hi = box[2 * (size_t)t + 1];
    return make_float4(g.B == 0 ? lo.x : lo.y, g.B == 0 ? hi.x : hi.y, g.C == 1 ? lo.y : lo.z,
                       g.C == 1 ? hi.y : hi.z);
}

// Ranges of the rows that a box of extents e may meet, from one cell to either
// side.
struct RowRange {
    uint32_t b, c, wide, high;
};
__device__ __forceinline__ RowRange row_range(const RowGeom &g, const float4 e) {
    const uint32_t nb = g.dims[g.B], nc = g.dims[g.C];
    const float b0 = (e.x - g.lo[g.B]) / g.cell[g.B], b1 = (e.y - g.lo[g.B]) / g.cell[g.B];
    const float c0 = (e.z - g.lo[g.C]) / g.cell[g.C], c1 = (e.w - g.lo[g.C]) / g.cell[g.C];
    auto slack = [](float v) { return 1.0f + 1e-6f * fabsf(v); };
    const int bl = (int)fminf(fmaxf(b0 - slack(b0), 0.0f), (float)(nb - 1));
    const int bh = (int)fminf(fmaxf(b1 + slack(b1), 0.0f), (float)(nb - 1));
    const int cl = (int)fminf(fmaxf(c0 - slack(c0), 0.0f), (float)(nc - 1));
    const int ch = (int)fminf(fmaxf(c1 + slack(c1), 0.0f), (float)(nc - 1));
    return RowRange{(uint32_t)bl, (uint32_t)cl, (uint32_t)max(bh - bl + 1, 0),
                    (uint32_t)max(ch - cl + 1, 0)};
}

// The triangles past the grid, after their count; *ends (of all zero before):
// the sum of their rows, in 64 bits.
__global__ __launch_bounds__(kBlock) void k_row_outside(RowGeom g, uint32_t n_tri,
                                                        const float4 *box, uint32_t *outside,
                                                        unsigned long long *ends) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= n_tri || !past_grid(g, box, t)) return;
    outside[1 + atomicAdd(&outside[0], 1u)] = t;
    const RowRange r = row_range(g, row_extent(g, box, t));
    atomicAdd(ends, (unsigned long long)r.wide * r.high);
}

// The list that every row shares, at its place.
__global__ __launch_bounds__(kBlock) void k_row_shared(RowGeom g, const uint32_t *outside,
                                                       const float4 *box, uint32_t *tri,
                                                       float4 *rec) {
    const uint32_t j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= outside[0]) return;
    const uint32_t t = outside[1 + j];
    tri[j] = t;
    rec[j] = row_extent(g, box, t);
}

// Their entries: in every row whose cells' boxes, computed as label_cell does,
// meet the triangle's on the axes across.  One block per triangle in turn.
// EMIT false counts a row's; true fills the places before the row's end, and
// counts them back to zero.
template <bool EMIT>
__global__ __launch_bounds__(kBlock) void k_row_ends(RowGeom g, const uint32_t *outside,
                                                     const float4 *box, uint32_t *count,
                                                     const uint32_t *start, uint32_t *tri,
                                                     float4 *rec) {
    const uint32_t n = outside[0], nb = g.dims[g.B];
    for (uint32_t j = blockIdx.x; j < n; j += gridDim.x) {
        const uint32_t t = outside[1 + j];
        const float4 e = row_extent(g, box, t);
        const RowRange w = row_range(g, e);
        const uint64_t all = (uint64_t)w.wide * w.high;
        for (uint64_t k = threadIdx.x; k < all; k += kBlock) {
            const uint32_t b = w.b + (uint32_t)(k % w.wide), c = w.c + (uint32_t)(k / w.wide);
            if (e.y < g.lo[g.B] + (float)b * g.cell[g.B] ||
                e.x > g.lo[g.B] + (float)(b + 1) * g.cell[g.B] ||
                e.w < g.lo[g.C] + (float)c * g.cell[g.C] ||
                e.z > g.lo[g.C] + (float)(c + 1) * g.cell[g.C])
                continue;
            const uint32_t r = c * nb + b;
            if (EMIT) {
                const uint32_t at = start[(r + 1) * g.dims[g.A]] - atomicSub(&count[r], 1u);
                tri[at] = t;
                rec[at] = e;
            } else {
                atomicAdd(&count[r], 1u);
            }
        }
    }
}

// Row entries of the cell at place r of the row order: the listed triangles
// that the next cell of the row does not list, and for the row's last cell the
// places of the entries of k_row_ends after them (ends counts a row's).  EMIT
// false counts them, true writes those listed at start[r].
template <bool EMIT>
__global__ __launch_bounds__(kBlock) void k_row_lists(RowGeom g, uint32_t n_cells,
                                                      const uint32_t *cell_start,
                                                      const uint32_t *cell_tri, const float4 *box,
                                                      const uint32_t *ends, uint32_t *start,
                                                      uint32_t *tri, float4 *rec) {
    __shared__ BigCells B;
    if (threadIdx.x == 0) B.n = 0;
    __syncthreads();
    // cell at place r, its list and that of the row's next cell
    struct Lists {
        uint32_t k0, k1, a, b;
        bool last;
    };
    auto lists = [&](uint32_t r) {
        const uint32_t x = r % g.dims[g.A], y = r / g.dims[g.A] % g.dims[g.B],
                       z = r / g.dims[g.A] / g.dims[g.B];  // along A, B and C
        const uint32_t s1 = g.dims[0], s2 = g.dims[0] * g.dims[1];
        const uint32_t sa = g.A == 0 ? 1u : g.A == 1 ? s1 : s2, sb = g.B == 0 ? 1u : s1,
                       sc = g.C == 1 ? s1 : s2;
        const uint32_t c = x * sa + y * sb + z * sc;
        const bool last = x + 1 == g.dims[g.A];
        return Lists{cell_start[c], cell_start[c + 1], last ? 0u : cell_start[c + sa],
                     last ? 0u : cell_start[c + sa + 1], last};
    };
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r < n_cells) {
        const Lists L = lists(r);
        if (L.k1 - L.k0 > kFewEntries) {
            B.cell[atomicAdd(&B.n, 1u)] = r;
        } else {
            uint32_t n = EMIT ? start[r] : 0u, a = L.a;
            for (uint32_t k = L.k0; k < L.k1; ++k) {
                const uint32_t t = cell_tri[k];
                while (a < L.b && cell_tri[a] < t) ++a;  // both lists ascend
                if ((a < L.b && cell_tri[a] == t) || past_grid(g, box, t)) continue;
                if (EMIT) {
                    tri[n] = t;
                    rec[n] = row_extent(g, box, t);
                }
                ++n;
            }
            if (!EMIT) start[r] = n + (L.last ? ends[r / g.dims[g.A]] : 0u);
        }
    }
    __syncthreads();
    for (uint32_t b = 0; b < B.n; ++b) {
        const uint32_t q = B.cell[b];
        const Lists L = lists(q);
        by_block(
            B, L.k0, L.k1, EMIT ? start[q] : 0u,
            [&](uint32_t k) {
                const uint32_t t = cell_tri[k];
                return !past_grid(g, box, t) && find_tri(cell_tri, L.a, L.b, t) == L.b;
            },
            [&](uint32_t n, uint32_t k) {
                if (!EMIT) return;
                tri[n] = cell_tri[k];
                rec[n] = row_extent(g, box, cell_tri[k]);
            },
            [&](uint32_t n) {
                if (!EMIT) start[q] = n + (L.last ? ends[q / g.dims[g.A]] : 0u);
            });
    }
}

uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

}  // namespace

// Fine cells per grid cell and axis.  Planar grids take 4 (16 bytes a grid
// cell), less where the table would pass kFineMaxBytes; three-dimensional ones
// take 1: with 2 (8 bytes) 50,000 spins among crossing bundles walk no faster
// (22.8 ms and 22.9), the device full of larger substrates by 5% (1.34e10
// spin-steps/s against 1.27e10), for 7 bytes a cell and twice the build time.
constexpr uint32_t kFineSub2D = 4, kFineSub3D = 1;
constexpr uint64_t kFineMaxBytes = 1ull << 29;

static int build_fine_clearance(dsim_substrate *S, hipStream_t st) {
    int axes = 0;
    for (int k = 0; k < 3; ++k) axes += S->dims[k] > 1;
    if (axes == 0 || !S->d_clearance.p) return DSIM_OK;  // no table: every step searches
    uint32_t sub = axes == 3 ? kFineSub3D : kFineSub2D;
    uint64_t n = 0;
    FineGeom f{};
    for (;; sub /= 2) {
        n = 1;
        for (int k = 0; k < 3; ++k) {
            f.sub[k] = S->dims[k] > 1 ? sub : 1;
            f.dims[k] = S->dims[k] * f.sub[k];
            n *= f.dims[k];
        }
        if (sub == 1 || n <= kFineMaxBytes) break;
    }
    Geom g{};
    g.kind = S->kind;
    float smallest = 3.0e38f, h2 = 0.0f;
    for (int k = 0; k < 3; ++k) {
        g.dims[k] = S->dims[k]; g.lo[k] = S->lo[k]; g.cell[k] = S->cell[k];
        f.cell[k] = S->cell[k] / (float)f.sub[k];
        f.w[k] = S->dims[k] > 1 ? 1.0f : 0.0f;
        if (f.w[k] != 0.0f) {
            smallest = std::min(smallest, S->cell[k]);
            h2 += 0.25f * f.cell[k] * f.cell[k];
        }
        S->fine_dims[k] = f.dims[k];
        S->fine_inv[k] = S->inv_cell[k] * (float)f.sub[k];
        S->fine_w[k] = f.w[k];
    }
    f.half_diag = std::sqrt(h2) * 1.00001f;
    f.margin = kFineMargin * S->margins;
    f.q = S->fine_q = smallest / kFineRange;
    if (int rc = S->d_fine.alloc(n))  // no table: every step searches
        return rc == DSIM_ERR_NOMEM ? DSIM_OK : rc;
    hipLaunchKernelGGL(k_fine_clearance, dim3(blocks_for(n)), dim3(kBlock), 0, st, g, f,
                       S->d_cell_start.p, S->d_cell_tri.p, S->tri_mt.p, S->d_clearance.p,
                       S->d_fine.p);
    HIP_TRY(hipGetLastError());
    return DSIM_OK;
}

namespace {
template <class T>
struct TempBuf : DevBuf<T> {
    ~TempBuf() { this->release(); }
};
}  // namespace

static int build_search_lists(dsim_substrate *S, hipStream_t st) {
    const uint32_t nT = S->n_tri, nC = S->n_cells;
    const size_t nt1 = std::max<uint32_t>(nT, 1);
    const bool cell_major = S->kind != DSIM_GRID_TRIBOX;
    TempBuf<uint64_t> keys, keys2;
    TempBuf<uint32_t> vals, vals2, partner, eps;
    TempBuf<float4> rec;
    TempBuf<uint8_t> temp;
    int rc;
    if ((rc = keys.alloc(nt1)) || (rc = keys2.alloc(nt1)) || (rc = vals.alloc(nt1)) ||
        (rc = vals2.alloc(nt1)) || (rc = partner.alloc(nt1)) || (rc = eps.alloc(1)) ||
        (rc = rec.alloc(nt1 * 2)) || (rc = S->walk_start.alloc((size_t)nC + 1)))
        return rc;
    HIP_TRY(hipMemsetAsync(eps.p, 0, 4, st));
    size_t tb_sort = 0, tb_scan = 0;
    if (nT)
        HIP_TRY(rocprim::radix_sort_pairs(nullptr, tb_sort, keys.p, keys2.p, vals.p, vals2.p, nT, 0,
                                          64, st));
    HIP_TRY(rocprim::exclusive_scan(nullptr, tb_scan, S->walk_start.p, S->walk_start.p, 0u,
                                    (size_t)nC + 1, rocprim::plus<uint32_t>(), st));
    if ((rc = temp.alloc(std::max({tb_sort, tb_scan, (size_t)1})))) return rc;
    if (nT) {
        hipLaunchKernelGGL(k_plane_keys, dim3(blocks_for(nT)), dim3(kBlock), 0, st, nT, S->tri_mt.p,
                           keys.p, vals.p);
        HIP_TRY(rocprim::radix_sort_pairs(temp.p, tb_sort, keys.p, keys2.p, vals.p, vals2.p, nT, 0,
                                          64, st));
        hipLaunchKernelGGL(k_pair_triangles, dim3(blocks_for(nT)), dim3(kBlock), 0, st, nT, keys2.p,
                           vals2.p, S->tri_mt.p, partner.p);
        hipLaunchKernelGGL(k_walk_records, dim3(blocks_for(nT)), dim3(kBlock), 0, st, nT, S->tri_mt.p,
                           partner.p, S->margins, rec.p, eps.p);
    }
    hipLaunchKernelGGL(k_walk_lists<false>, dim3(blocks_for(nC)), dim3(kBlock), 0, st, nC,
                       S->d_cell_start.p, S->d_cell_tri.p, partner.p, S->walk_start.p,
                       (uint2 *)nullptr, (const float4 *)nullptr, (float4 *)nullptr);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemsetAsync(S->walk_start.p + nC, 0, 4, st));
    HIP_TRY(rocprim::exclusive_scan(temp.p, tb_scan, S->walk_start.p, S->walk_start.p, 0u,
                                    (size_t)nC + 1, rocprim::plus<uint32_t>(), st));
    uint32_t n = 0;
    float dev = 0.0f;
    HIP_TRY(hipMemcpyAsync(&n, S->walk_start.p + nC, 4, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipMemcpyAsync(&dev, eps.p, 4, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    const size_t n1 = std::max<uint32_t>(n, 1);
    if ((rc = S->walk_ent.alloc(n1)) || (cell_major && (rc = S->walk_rec.alloc(n1 * 2)))) return rc;
    hipLaunchKernelGGL(k_walk_lists<true>, dim3(blocks_for(nC)), dim3(kBlock), 0, st, nC,
                       S->d_cell_start.p, S->d_cell_tri.p, partner.p, S->walk_start.p, S->walk_ent.p,
                       rec.p, S->walk_rec.p);
    HIP_TRY(hipGetLastError());
    // side distances are off by the record's own error and by FP32 rounding at
    // coordinates up to 2 (three fused operations of half an ulp, 4e-7)
    S->walk_eps = 2.0f * dev + 1e-6f * S->margins;
    if (!cell_major) std::swap(S->walk_rec, static_cast<DevBuf<float4> &>(rec));
    HIP_TRY(hipStreamSynchronize(st));  // the temporary arrays are freed on return
    return DSIM_OK;
}

// Masks of grids up to this many cells (256 MB); larger ones list every box.
constexpr uint32_t kRefMaskCells = 1u << 26;

static int build_ref_tables(dsim_substrate *S, hipStream_t st) {
    const uint32_t n = (uint32_t)S->d_cell_tri.n;  // one unused entry where the grid lists none
    if (int rc = S->ref_rec.alloc((size_t)n * 2)) return rc;
    if (S->n_tri) {
        hipLaunchKernelGGL(k_ref_records, dim3(blocks_for(n)), dim3(kBlock), 0, st, n,
                           S->d_cell_tri.p, S->tri_ref.p, S->ref_rec.p);
        HIP_TRY(hipGetLastError());
    }
    if (S->n_cells > kRefMaskCells) return DSIM_OK;
    if (int rc = S->ref_mask.alloc(S->n_cells)) return rc;
    hipLaunchKernelGGL(k_ref_masks, dim3(blocks_for(S->n_cells)), dim3(kBlock), 0, st, S->dims[0],
                       S->dims[1], S->dims[2], S->d_cell_start.p, S->ref_mask.p);
    HIP_TRY(hipGetLastError());
    return DSIM_OK;
}

int dsim_host::build_row_lists(const dsim_substrate *S, RowLists &R, uint64_t most,
                               uint64_t room, hipStream_t st) {
    const uint32_t nT = S->n_tri, nC = S->n_cells;
    RowGeom g{};
    g.A = (int)S->label_axis;
    g.B = g.A == 0 ? 1 : 0;
    g.C = g.A == 2 ? 1 : 2;
    g.exact = S->kind == DSIM_GRID_TRIBOX;
    g.face = S->lo[g.A] + (float)S->dims[g.A] * S->cell[g.A];
    for (int k = 0; k < 3; ++k) { g.dims[k] = S->dims[k]; g.lo[k] = S->lo[k]; g.cell[k] = S->cell[k]; }
    const uint32_t n_rows = g.dims[g.B] * g.dims[g.C], n_blocks = std::min(nT, 1024u);
    // Scratch of the pool, not of the runtime, whose hipFree waits for the whole
    // device: a server makes lists while its requests step.  The pool does not
    // wait, so an early return waits for the stream here.
    struct Scratch {
        hipStream_t st;
        dsim_host::PoolBuf<uint8_t> temp;
        // the sum of the rows to fill (two words), the triangles past the grid after
        // their count, and the rows' counts of their entries
        dsim_host::PoolBuf<uint32_t> outside;
        bool waited = false;
        ~Scratch() {
            if (!waited) (void)hipStreamSynchronize(st);
            temp.release(); outside.release();
        }
    } scratch{st, {}, {}};
    auto &temp = scratch.temp;
    int rc;
    size_t tb = 0;
    HIP_TRY(rocprim::exclusive_scan(nullptr, tb, R.start.p, R.start.p, 0u,
                                    (size_t)nC + 1, rocprim::plus<uint32_t>(), st));
    const uint64_t making = tb + ((uint64_t)nT + 1 + n_rows) * 4 + 64 + ((uint64_t)nC + 1) * 4;
    if (!pool_room(making, room)) return DSIM_OK;
    if ((rc = temp.alloc(std::max(tb, (size_t)1))) || (rc = R.start.alloc((size_t)nC + 1)) ||
        (rc = scratch.outside.alloc((size_t)nT + 3 + n_rows)))
        return rc;
    unsigned long long *sum = reinterpret_cast<unsigned long long *>(scratch.outside.p);
    uint32_t *outside = scratch.outside.p + 2, *ends = outside + nT + 1;
    HIP_TRY(hipMemsetAsync(scratch.outside.p, 0, scratch.outside.n * 4, st));
    if (nT)
        hipLaunchKernelGGL(k_row_outside, dim3(blocks_for(nT)), dim3(kBlock), 0, st, g, nT,
                           S->tri_aabb.p, outside, sum);
    HIP_TRY(hipGetLastError());
    uint32_t seen[3] = {0, 0, 0};
    HIP_TRY(hipMemcpyAsync(seen, scratch.outside.p, 12, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    const uint32_t n_out = seen[2];
    const uint64_t n_ends = seen[0] | (uint64_t)seen[1] << 32;
    const RowPlan plan = row_plan(nC, S->d_cell_tri.n, n_out, n_ends);
    if (plan == kRowsNone) {
        R.start.release();
        return DSIM_OK;
    }
    if (plan == kRowsEnds && n_out)
        hipLaunchKernelGGL(k_row_ends<false>, dim3(n_blocks), dim3(kBlock), 0, st, g, outside,
                           S->tri_aabb.p, ends, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                           (float4 *)nullptr);
    hipLaunchKernelGGL(k_row_lists<false>, dim3(blocks_for(nC)), dim3(kBlock), 0, st, g, nC,
                       S->d_cell_start.p, S->d_cell_tri.p, S->tri_aabb.p, ends, R.start.p,
                       (uint32_t *)nullptr, (float4 *)nullptr);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemsetAsync(R.start.p + nC, 0, 4, st));
    HIP_TRY(rocprim::exclusive_scan(temp.p, tb, R.start.p, R.start.p, 0u,
                                    (size_t)nC + 1, rocprim::plus<uint32_t>(), st));
    uint32_t n = 0;
    HIP_TRY(hipMemcpyAsync(&n, R.start.p + nC, 4, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    R.shared = n;
    R.n_shared = plan == kRowsShared ? n_out : 0u;
    // a lane past its row's end reads entry 0
    const size_t n1 = std::max<size_t>((size_t)n + R.n_shared, 1);
    if (((uint64_t)nC + 1) * 4 + (uint64_t)n1 * 20 > most ||
        !pool_room(making + (uint64_t)n1 * 20, room)) {
        R.start.release();
        return DSIM_OK;
    }
    if ((rc = R.tri.alloc(n1)) || (rc = R.box.alloc(n1))) return rc;
    hipLaunchKernelGGL(k_row_lists<true>, dim3(blocks_for(nC)), dim3(kBlock), 0, st, g, nC,
                       S->d_cell_start.p, S->d_cell_tri.p, S->tri_aabb.p, ends, R.start.p,
                       R.tri.p, R.box.p);
    if (plan == kRowsEnds && n_out)
        hipLaunchKernelGGL(k_row_ends<true>, dim3(n_blocks), dim3(kBlock), 0, st, g, outside,
                           S->tri_aabb.p, ends, R.start.p, R.tri.p, R.box.p);
    if (R.n_shared)
        hipLaunchKernelGGL(k_row_shared, dim3(blocks_for(R.n_shared)), dim3(kBlock), 0, st, g,
                           outside, S->tri_aabb.p, R.tri.p + n, R.box.p + n);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(st));
    scratch.waited = true;
    return DSIM_OK;
}

int dsim_host::build_walk_tables(dsim_substrate *S, hipStream_t st) {
    const uint64_t most = S->kind == DSIM_GRID_AABB ? ~0ull : kRowKeepBytes;
    if (S->kind != DSIM_GRID_REFERENCE)
        if (int rc = build_row_lists(S, S->rows, most, ~0ull, st)) {
            if (rc != DSIM_ERR_NOMEM) return rc;
            S->rows.release();  // labelled without, or with those that a call can make
        }
    if (S->kind == DSIM_GRID_REFERENCE)
        if (int rc = build_ref_tables(S, st)) return rc;
    if (int rc = build_search_lists(S, st)) return rc;
    return build_fine_clearance(S, st);
}

extern "C" int dsim_substrate_create_device(const dsim_mesh *mesh, const dsim_grid_params *grid,
                                            dsim_substrate **out) {
    if (!mesh || !grid || !out) return fail(DSIM_ERR_ARG, "NULL argument");
    *out = nullptr;
    if (int rc = dsim_host::check_mesh(mesh)) return rc;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(DSIM_ERR_STATE, "dsim_substrate_create_device needs a HIP device");
    const uint32_t nT = mesh->n_triangles, nV = mesh->n_vertices;
    Geom g{};
    g.kind = grid->kind;
    auto *S = new dsim_substrate();
    S->n_tri = nT;
    S->n_vert = nV;
    S->kind = grid->kind;
    if (grid->kind == DSIM_GRID_REFERENCE) {
        const uint32_t n = grid->dims[0];
        if (n == 0 || n > 1024) { delete S; return fail(DSIM_ERR_ARG, "reference grid n=%u", n); }
        const float L = 2.0f / (float)n;  // m_cubeLength, spinSystem.cpp:1115
        g.L = L;
        for (int k = 0; k < 3; ++k) {
            S->dims[k] = n; S->lo[k] = -1.0f; S->cell[k] = L; S->inv_cell[k] = 1.0f / L;
        }
    } else if (grid->kind == DSIM_GRID_AABB || grid->kind == DSIM_GRID_TRIBOX) {
        for (int k = 0; k < 3; ++k) {
            if (grid->dims[k] == 0 || !(grid->cell[k] > 0.0f)) {
                delete S;
                return fail(DSIM_ERR_ARG, "AABB grid dims/cell invalid on axis %d", k);
            }
            S->dims[k] = grid->dims[k]; S->lo[k] = grid->lo[k]; S->cell[k] = grid->cell[k];
            S->inv_cell[k] = 1.0f / grid->cell[k];
        }
        if ((uint64_t)S->dims[0] * S->dims[1] * S->dims[2] > (1ull << 28)) {
            delete S;
            return fail(DSIM_ERR_ARG, "grid too large");
        }
        g.eps = grid->eps;
        g.exact_rings = dsim_host::clearance_rings(grid);
    } else {
        delete S;
        return fail(DSIM_ERR_ARG, "unknown grid kind %u", grid->kind);
    }
    for (int k = 0; k < 3; ++k) { g.dims[k] = S->dims[k]; g.lo[k] = S->lo[k]; g.cell[k] = S->cell[k]; }
    S->n_cells = S->dims[0] * S->dims[1] * S->dims[2];
    uint32_t nf = 0;
    for (uint32_t t = 0; t < nT; ++t) nf = std::max(nf, mesh->tri_info[t * 3] + 1);
    S->n_fibers = nf;
    std::vector<uint8_t> myel(std::max(1u, nf), 0);
    for (uint32_t t = 0; t < nT; ++t)
        if (mesh->tri_info[t * 3 + 1] == 1) myel[mesh->tri_info[t * 3]] = 1;
    S->on_device = true;
    S->device_built = true;
    S->label_axis = dsim_host::label_axis_of(mesh);
    S->margins = dsim_host::margin_scale(mesh, S);

    int rc = DSIM_OK;
    const hipStream_t st = nullptr;
    DevBuf<float> dV;
    DevBuf<uint32_t> dT, dI, cnt, offs, keys, vals, keys2, vals2, ccount, ring, flag, maxc;
    DevBuf<uint8_t> temp;
    auto cleanup = [&] {
        dV.release(); dT.release(); dI.release(); cnt.release(); offs.release(); keys.release();
        vals.release();
        keys2.release(); vals2.release(); ccount.release(); ring.release(); flag.release();
        maxc.release(); temp.release();
    };
    auto bail = [&](int code) {
        cleanup();
        delete S;
        return code;
    };
#define GRID_TRY(expr)                                                                      \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess)                                                               \
            return bail(fail(DSIM_ERR_HIP, "device grid build: %s: %s", #expr,              \
                             hipGetErrorString(e_)));                                       \
    } while (0)

    // mesh upload and triangle records
    const size_t nt1 = std::max<uint32_t>(nT, 1);
    if ((rc = dV.alloc(std::max<size_t>((size_t)nV * 3, 1))) || (rc = dT.alloc(nt1 * 3)) ||
        (rc = dI.alloc(nt1 * 3)) || (rc = S->d_helpers.alloc(nt1 * 12)) ||
        (rc = S->tri_ref.alloc(nt1 * 4)) || (rc = S->tri_mt.alloc(nt1 * 4)) ||
        (rc = S->tri_aabb.alloc(nt1 * 2)) || (rc = cnt.alloc(nt1 + 1)) || (rc = offs.alloc(nt1 + 1)) ||
        (rc = S->d_cell_start.alloc((size_t)S->n_cells + 1)) ||
        (rc = ccount.alloc((size_t)S->n_cells + 1)) || (rc = maxc.alloc(4)) ||
        (rc = flag.alloc(1)))
        return bail(rc);
    if (nV) GRID_TRY(hipMemcpy(dV.p, mesh->vertices, (size_t)nV * 12, hipMemcpyHostToDevice));
    if (nT) {
        GRID_TRY(hipMemcpy(dT.p, mesh->triangles, (size_t)nT * 12, hipMemcpyHostToDevice));
        GRID_TRY(hipMemcpy(dI.p, mesh->tri_info, (size_t)nT * 12, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(k_tri_records, dim3(blocks_for(nT)), dim3(kBlock), 0, st, nT, dV.p,
                           dT.p, dI.p, S->d_helpers.p, S->tri_ref.p, S->tri_mt.p, S->tri_aabb.p);
        GRID_TRY(hipGetLastError());
    }
    if ((rc = dsim_host::upload(S->fiber_myelin, myel))) return bail(rc);

    // pairs per triangle, their offsets, the pairs, the per-cell counts
    GRID_TRY(hipMemsetAsync(cnt.p, 0, (nt1 + 1) * 4, st));
    GRID_TRY(hipMemsetAsync(ccount.p, 0, ((size_t)S->n_cells + 1) * 4, st));
    if (nT) {
        hipLaunchKernelGGL(k_pairs<false>, dim3(blocks_for((uint64_t)nT * kPairLanes)), dim3(kBlock), 0, st, g, nT, dV.p,
                           dT.p, cnt.p, (uint32_t *)nullptr, (uint32_t *)nullptr,
                           (uint32_t *)nullptr);
        GRID_TRY(hipGetLastError());
    }
    // exclusive scan over nT + 1 counts: offsets, and the total in the last
    size_t tb_scan1 = 0, tb_scan2 = 0, tb_sort = 0, tb_red = 0;
    GRID_TRY(rocprim::exclusive_scan(nullptr, tb_scan1, cnt.p, offs.p, 0u, nT + 1,
                                     rocprim::plus<uint32_t>(), st));
    GRID_TRY(rocprim::exclusive_scan(nullptr, tb_scan2, ccount.p, S->d_cell_start.p, 0u,
                                     (size_t)S->n_cells + 1, rocprim::plus<uint32_t>(), st));
    GRID_TRY(rocprim::reduce(nullptr, tb_red, ccount.p, maxc.p, 0u, (size_t)S->n_cells,
                             rocprim::maximum<uint32_t>(), st));
    // the pairs in 64 bits: their places and numbers are 32-bit
    const auto wide = rocprim::make_transform_iterator(
        cnt.p, [] __device__(uint32_t v) { return (unsigned long long)v; });
    unsigned long long *total = reinterpret_cast<unsigned long long *>(maxc.p + 2);
    size_t tb_sum = 0;
    GRID_TRY(rocprim::reduce(nullptr, tb_sum, wide, total, 0ull, (size_t)nT,
                             rocprim::plus<unsigned long long>(), st));
    const size_t tb0 = std::max({tb_scan1, tb_scan2, tb_red, tb_sum, (size_t)1});
    if ((rc = temp.alloc(tb0))) return bail(rc);
    if (nT)
        GRID_TRY(rocprim::reduce(temp.p, tb_sum, wide, total, 0ull, (size_t)nT,
                                 rocprim::plus<unsigned long long>(), st));
    {
        size_t b = tb_scan1;
        GRID_TRY(rocprim::exclusive_scan(temp.p, b, cnt.p, offs.p, 0u, nT + 1,
                                         rocprim::plus<uint32_t>(), st));
    }
    unsigned long long n_listed = 0;
    if (nT) GRID_TRY(hipMemcpyAsync(&n_listed, total, 8, hipMemcpyDeviceToHost, st));
    GRID_TRY(hipStreamSynchronize(st));
    if (n_listed > 0xFFFFFFFFull)
        return bail(fail(DSIM_ERR_ARG, "grid too fine: %llu entries in its cells, more than 2^32 - 1",
                         n_listed));
    const uint32_t n_pairs = (uint32_t)n_listed;
    const size_t np1 = std::max<uint32_t>(n_pairs, 1);
    if ((rc = keys.alloc(np1)) || (rc = vals.alloc(np1)) || (rc = keys2.alloc(np1)) ||
        (rc = S->d_cell_tri.alloc(np1)))
        return bail(rc);
    if (nT) {
        hipLaunchKernelGGL(k_pairs<true>, dim3(blocks_for((uint64_t)nT * kPairLanes)), dim3(kBlock), 0, st, g, nT, dV.p,
                           dT.p, offs.p, keys.p, vals.p, ccount.p);
        GRID_TRY(hipGetLastError());
    }
    // stable sort by cell: each cell's list in ascending triangle order
    unsigned end_bit = 1;
    while (end_bit < 32 && (1ull << end_bit) < S->n_cells) ++end_bit;
    if (n_pairs) {
        GRID_TRY(rocprim::radix_sort_pairs(nullptr, tb_sort, keys.p, keys2.p, vals.p,
                                           S->d_cell_tri.p, n_pairs, 0, end_bit, st));
        if (tb_sort > temp.n) {
            temp.release();
            if ((rc = temp.alloc(tb_sort))) return bail(rc);
        }
        size_t b = tb_sort;
        GRID_TRY(rocprim::radix_sort_pairs(temp.p, b, keys.p, keys2.p, vals.p, S->d_cell_tri.p,
                                           n_pairs, 0, end_bit, st));
    } else {
        GRID_TRY(hipMemsetAsync(S->d_cell_tri.p, 0, 4, st));
    }
    {
        size_t b = tb_scan2;
        GRID_TRY(rocprim::exclusive_scan(temp.p, b, ccount.p, S->d_cell_start.p, 0u,
                                         (size_t)S->n_cells + 1, rocprim::plus<uint32_t>(), st));
        b = tb_red;
        GRID_TRY(rocprim::reduce(temp.p, b, ccount.p, maxc.p, 0u, (size_t)S->n_cells,
                                 rocprim::maximum<uint32_t>(), st));
    }
    GRID_TRY(hipMemcpyAsync(&S->max_per_cell, maxc.p, 4, hipMemcpyDeviceToHost, st));
    S->n_entries = n_pairs;

    // clearance (AABB and exact-membership grids)
    if (grid->kind != DSIM_GRID_REFERENCE) {
        if ((rc = ring.alloc(S->n_cells)) || (rc = S->d_clearance.alloc(S->n_cells)))
            return bail(rc);
        const uint32_t nb = blocks_for(S->n_cells);
        hipLaunchKernelGGL(k_ring_init, dim3(nb), dim3(kBlock), 0, st, S->n_cells,
                           S->d_cell_start.p, ring.p);
        GRID_TRY(hipGetLastError());
        // rings grow by one per step; the flag is read every 8 steps (steps
        // past the last ring change nothing)
        const uint32_t max_r = std::max({S->dims[0], S->dims[1], S->dims[2]});
        for (uint32_t r = 1; n_pairs && r <= max_r; r += 8) {
            GRID_TRY(hipMemsetAsync(flag.p, 0, 4, st));
            for (uint32_t q = r; q < r + 8; ++q)
                hipLaunchKernelGGL(k_ring_step, dim3(nb), dim3(kBlock), 0, st, S->dims[0],
                                   S->dims[1], S->dims[2], ring.p, q, flag.p);
            GRID_TRY(hipGetLastError());
            uint32_t changed = 0;
            GRID_TRY(hipMemcpyAsync(&changed, flag.p, 4, hipMemcpyDeviceToHost, st));
            GRID_TRY(hipStreamSynchronize(st));
            if (!changed) break;
        }
        hipLaunchKernelGGL(k_clearance, dim3(nb), dim3(kBlock), 0, st, g, ring.p,
                           S->d_cell_start.p, S->d_cell_tri.p, S->tri_aabb.p, dV.p, dT.p,
                           S->d_clearance.p);
        GRID_TRY(hipGetLastError());
    }
    if ((rc = dsim_host::build_walk_tables(S, st))) return bail(rc);
    GRID_TRY(hipStreamSynchronize(st));
#undef GRID_TRY
    cleanup();
    *out = S;
    return DSIM_OK;
}
