// Shared pieces of the host runtime: error reporting, device buffers and the
// substrate object (used by host.cpp and sim.cpp).
#pragma once

#include <cstdint>
#include <cstring>
#include <vector>

#include <hip/hip_runtime_api.h>
#include <hip/hip_vector_types.h>

#include "../../include/dsim.h"

struct dsim_substrate;
namespace dsim_host {

// Records a message for dsim_last_error() and returns code.
int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

// Checks the mesh arrays of dsim_substrate_create (indices, membranes, fibres).
int check_mesh(const dsim_mesh *mesh);
// Axis (0 x, 1 y, 2 z) of the physical mode's labelling rays for a mesh.
uint32_t label_axis_of(const dsim_mesh *mesh);
// The margins of the walk's tables are set for coordinates up to 2,
// the normalised ones; this is the factor for a mesh and grid beyond those, half
// their largest finite coordinate (1 at least): the rounding that the margins
// cover grows with it.
float margin_scale(const dsim_mesh *mesh, const dsim_substrate *S);
// Exact clearance refinement of exact-membership grids by default: rings 0-1.
// Their exact distances cost a separating-axis gap per listed triangle of the
// surrounding cells; measured on crossing substrates, refining rings 0-1 keeps
// the walk within 1% of refining 0-3 at a third of the build time, and the
// ring distance alone costs 6-17% of the walk.
constexpr int64_t kTriboxRings = 1;
// Rings of exact clearance refinement of a grid (cells at ring distance at
// most this; -1 none).
int64_t clearance_rings(const dsim_grid_params *g);

// The largest float whose square is at most x >= 0 (the float floor of the
// square root, whatever the rounding of the double square root: the square of
// a float is exact in double).
inline float float_sqrt_floor(double x) {
    if (!(x >= 0.0)) return 0.0f;
    float f = (float)__builtin_sqrt(x);
    while (f > 0.0f && (double)f * (double)f > x) f = __builtin_nextafterf(f, 0.0f);
    for (;;) {
        const float g = __builtin_nextafterf(f, 3.0e38f);
        if ((double)g * (double)g > x) break;
        f = g;
    }
    return f;
}

// Device memory.  dev_alloc fails with nullptr and the runtime's error in *e;
// before it does, it gives the pool's idle blocks back and tries again.
void *dev_alloc(size_t bytes, hipError_t *e);

// Idle blocks of simulation and waveform handles, kept for the next handle
// while any simulation or server is alive (pool_ref, pool_unref), up to
// 1/kPoolShare of each device's memory, the oldest given back first, and all
// given back when an allocation here would fail.  A block stays with the device
// that was current when it was allocated, whichever is when it is given back.  Handles come and go with
// every request or run of waveforms, and gigabytes freed and allocated each
// time cost the runtime far more than the work at times: freeing the 9.5 GB of
// 1024 waveforms of 500,000 spins took 1.5 ms or, once a run had allocated
// about the device's memory, 180 ms of a 270 ms pass.  A block goes to a
// request of at least three quarters of its size.  The caller of pool_give
// has waited for the device, as hipFree does.
constexpr size_t kPoolShare = 16, kPoolBlocks = 256;
void *pool_take(size_t bytes, size_t *got, int *device, hipError_t *e);
void pool_give(void *p, size_t bytes, int device);
// Idle blocks of the device given back, oldest first, until `most` bytes of them
// are left.
void pool_trim_to(int device, uint64_t most);
// May `need` more bytes be taken out of `room` (~0 no limit), which idle blocks
// of the current device share?  Gives back those that do not fit beside them.
bool pool_room(uint64_t need, uint64_t room);
void pool_ref();
void pool_unref();

template <class T, bool POOL = false>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    size_t block = 0;  // bytes of the pool's block
    int device = -1;   // that it lies on
    int alloc(size_t count) {
        n = count;
        if (count == 0) return DSIM_OK;
        hipError_t e = hipSuccess;
        p = static_cast<T *>(POOL ? pool_take(count * sizeof(T), &block, &device, &e)
                                  : dev_alloc(count * sizeof(T), &e));
        if (!p) {
            n = 0;
            return fail(DSIM_ERR_NOMEM, "hipMalloc(%zu bytes): %s", count * sizeof(T),
                        hipGetErrorString(e));
        }
        return DSIM_OK;
    }
    // Bytes of the block past the buffer's own.
    uint64_t slack() const { return p && POOL ? block - n * sizeof(T) : 0; }
    void release() {
        if (p && POOL) pool_give(p, block, device);
        else if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
};
template <class T>
using PoolBuf = DevBuf<T, true>;

template <class T>
int upload(DevBuf<T> &d, const std::vector<T> &h) {
    int rc = d.alloc(h.size());
    if (rc) return rc;
    if (!h.empty()) {
        hipError_t e = hipMemcpy(d.p, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice);
        if (e != hipSuccess) return fail(DSIM_ERR_HIP, "upload: %s", hipGetErrorString(e));
    }
    return DSIM_OK;
}

}  // namespace dsim_host

struct dsim_substrate;
namespace dsim_host {
// Builds the walk's search lists and fine clearance from the device grid,
// records and clearance (grid.hip).
int build_walk_tables(dsim_substrate *S, hipStream_t st);

// Row lists of the labeller (LabelParams::row_start).  A substrate keeps its own,
// on an exact-membership grid up to kRowKeepBytes; above that every labelling
// makes them and gives them back, or goes without where there is no memory for
// them.  On an AABB grid they are a third of the substrate or less (4 bytes a
// cell of its 13, 20 an entry of its 44), and its rows were cheap to walk without
// lists: 1000 spins on 400^3 cells take 35 us with them kept (1.4 GB in all), 1.47
// ms with them made by the call.  On crossing bundles, exact-membership grids, the
// lists are about half of a substrate, for a call made once a spin set, and
// making them adds about 0.3 ms to it for every 50 MiB of them.  Labelling 1e5
// spins with lists kept / made by the call: 200 axons (61 MiB of lists) 0.22 /
// 0.56 ms, 400 (108) 0.41 / 0.93, 800 (210) 0.80 / 1.72, 1600 (417) 2.07 / 4.02.
// So the line trades memory for a factor of two in a call that walks of 20 ms and
// more follow; it lies where the lists pass 100 MiB, below which a device full of
// such substrates holds a thousand of them.
constexpr uint64_t kRowKeepBytes = 128ull << 20;
struct RowLists {
    PoolBuf<uint32_t> start, tri;
    PoolBuf<float4> box;
    uint32_t shared = 0, n_shared = 0;  // entries of every row (kRowsShared)
    void release() { start.release(); tri.release(); box.release(); }
    uint64_t bytes() const { return (start.n + tri.n) * 4 + box.n * 16; }
};
// Where the triangles past the grid's face stand: an entry in every row that
// their boxes meet (`ends` at most), or, where those would be more than the
// grid's own cells and entries or than kRowEndsMax (320 MB; their counting, an
// atomic addition each, would take tens of ms and more), once in a list that
// every row shares.  Places are 32-bit: a grid whose entries alone pass that
// gets no row lists, and its spins go through the pass over all triangles.
enum RowPlan { kRowsNone, kRowsShared, kRowsEnds };
constexpr uint64_t kRowEndsMax = 1ull << 24;
inline RowPlan row_plan(uint64_t n_cells, uint64_t n_entries, uint64_t n_outside, uint64_t ends) {
    constexpr uint64_t most = 0xFFFFFF00ull;
    if (n_entries + n_outside > most) return kRowsNone;
    if (ends > n_cells + n_entries || ends > kRowEndsMax || n_entries + ends > most)
        return kRowsShared;
    return kRowsEnds;
}
// Lists of more than `most` bytes, or for which `room` is too small with the
// scratch of their making (pool_room), or none by row_plan, are left empty.
// Waits for st.
int build_row_lists(const dsim_substrate *S, RowLists &R, uint64_t most, uint64_t room,
                    hipStream_t st);
}  // namespace dsim_host

#define HIP_TRY(expr)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess)                                                                \
            return dsim_host::fail(DSIM_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

struct dsim_substrate {
    uint32_t n_tri = 0, n_vert = 0, n_fibers = 0;
    std::vector<float> helpers;  // [n_tri*12]
    std::vector<uint32_t> cell_start, cell_tri;
    uint32_t n_cells = 0, max_per_cell = 0;
    uint32_t kind = 0;
    uint32_t label_axis = 0;  // ray axis of the physical-mode labeller (0 x, 1 y, 2 z)
    uint32_t dims[3] = {0, 0, 0};
    float lo[3] = {0, 0, 0}, cell[3] = {0, 0, 0}, inv_cell[3] = {0, 0, 0};
    std::vector<float> clearance;  // per cell: lower bound of the distance to any triangle
    dsim_host::DevBuf<float4> tri_ref, tri_mt, tri_aabb;
    dsim_host::DevBuf<uint32_t> d_cell_start, d_cell_tri;
    dsim_host::DevBuf<float> d_clearance, d_helpers;
    // Reference grids: entry records and neighbour masks of the reference mode
    // (StepParams::ref_rec, ref_mask).
    dsim_host::DevBuf<float4> ref_rec;
    dsim_host::DevBuf<uint32_t> ref_mask;
    // The labeller's rows, where they are kept; not for the reference grid.
    dsim_host::RowLists rows;
    // Search lists of the physical-mode walk (build_walk_tables): per grid cell
    // its triangles, two of one plane in one entry (the second kNone where there
    // is none), and the entries' plane and lateral records, cell-major for
    // reference and AABB grids and by triangle (walk_rec[2 t]) for
    // exact-membership grids, whose long triangles are listed in many cells.
    dsim_host::DevBuf<uint32_t> walk_start;
    dsim_host::DevBuf<uint2> walk_ent;
    dsim_host::DevBuf<float4> walk_rec;
    float walk_eps = 0;  // bound of the error of a side distance (see walk_test, kernels.hip)
    float margins = 1.0f;  // margin_scale of the mesh and grid
    // Fine clearance of the walk: one byte per fine cell, a lower bound of the distance to any registered triangle
    // in units of fine_q; axes with one grid cell are collapsed (fine_w 0).
    dsim_host::DevBuf<uint8_t> d_fine;
    uint32_t fine_dims[3] = {0, 0, 0};
    float fine_inv[3] = {0, 0, 0}, fine_w[3] = {0, 0, 0}, fine_q = 0;
    dsim_host::DevBuf<uint8_t> fiber_myelin;
    int refs = 0;
    bool on_device = false;
    // built by dsim_substrate_create_device: the grid, helpers and clearance
    // live on the device only (the host vectors stay empty)
    bool device_built = false;
    uint32_t n_entries = 0;
    ~dsim_substrate() {
        tri_ref.release(); tri_mt.release(); tri_aabb.release();
        walk_start.release(); walk_ent.release(); walk_rec.release();
        ref_rec.release(); ref_mask.release();
        rows.release();
        d_clearance.release(); d_helpers.release(); d_fine.release();
        d_cell_start.release(); d_cell_tri.release(); fiber_myelin.release();
    }
};
