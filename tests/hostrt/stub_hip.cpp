// A HIP runtime of host memory for tests of the library's host code: two
// devices whose allocations are recorded with the device they were made on and
// can be made to fail, streams and events that are always done, and stand-ins
// for the kernel launches (most do nothing).
#include "stub_hip.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include <hip/hip_runtime_api.h>

#include "../../dsim_amd/csrc/dsim_internal.h"
#include "../../dsim_amd/csrc/host_common.h"

namespace stub {
std::mutex mu;
std::map<void *, Block> blocks;
size_t used[kDevices], peak[kDevices];
size_t total[kDevices] = {1ull << 30, 1ull << 28}, capacity[kDevices] = {1ull << 30, 1ull << 28};
uint64_t n_malloc, n_free;
uint32_t flag_bits, n_label_rows, n_label_all, n_row_builds;
uint64_t row_bytes;
bool keep_rows;
thread_local int device;
thread_local hipError_t last = hipSuccess;
hipError_t err(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
}  // namespace stub
using stub::err;

extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = stub::kDevices; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = stub::device; return hipSuccess; }
hipError_t hipSetDevice(int d) { stub::device = d; return hipSuccess; }
hipError_t hipDeviceTotalMem(size_t *b, int d) { *b = stub::total[d]; return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = stub::last; stub::last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "stub error"; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> l(stub::mu);
    const int d = stub::device;
    if (stub::used[d] + n > stub::capacity[d]) return err(hipErrorOutOfMemory);
    *p = malloc(n ? n : 1);
    memset(*p, 0xCD, n);
    stub::blocks[*p] = {d, n};
    stub::used[d] += n;
    stub::peak[d] = std::max(stub::peak[d], stub::used[d]);
    ++stub::n_malloc;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    std::lock_guard<std::mutex> l(stub::mu);
    auto it = stub::blocks.find(p);
    if (it == stub::blocks.end()) abort();
    stub::used[it->second.device] -= it->second.bytes;
    stub::blocks.erase(it);
    free(p);
    ++stub::n_free;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    if (!d || !s) return err(hipErrorInvalidValue);
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h,
                       hipMemcpyKind) {
    for (size_t r = 0; r < h; ++r) memcpy((char *)d + r * dp, (const char *)s + r * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    if (!d) return err(hipErrorInvalidValue);
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = reinterpret_cast<hipGraphExec_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { free(e); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = reinterpret_cast<hipEvent_t>(malloc(1));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { *t = 0.0f; return hipSuccess; }
}

// Kernel launches.  As the library's own do, they report an error left behind
// by an earlier call.
namespace dsim {
hipError_t launch_gather(uint32_t n, const uint32_t *perm, const Fields &f, hipStream_t) {
    for (uint32_t k = 0; k < f.count; ++k)
        for (uint32_t i = 0; i < n; ++i) f.dst[k][i] = f.src[k][perm[i]];
    return hipGetLastError();
}
hipError_t launch_init_seeds(uint32_t n, uint32_t *seed, uint32_t, uint32_t, hipStream_t) {
    for (uint32_t i = 0; i < 2 * n; ++i) seed[i] = i + 1;
    return hipGetLastError();
}
hipError_t launch_init_uniform(uint32_t n, float *x, float *y, float *z, float *mag, float *phase,
                               uint32_t *label, uint32_t *id, uint32_t *wrap, const float *,
                               const float *, uint32_t, uint32_t, uint64_t, hipStream_t) {
    for (uint32_t i = 0; i < n; ++i) {
        x[i] = y[i] = z[i] = 0.25f;
        mag[i] = 1.0f;
        phase[i] = 0.0f;
        label[i] = 0;
        id[i] = i;
        wrap[i] = 0;
    }
    return hipGetLastError();
}
hipError_t launch_label(const LabelParams &p, hipStream_t) {
    ++stub::n_label_all;
    for (uint32_t i = 0; i < p.n; ++i) p.label[i] = 7u << 8;
    return hipGetLastError();
}
hipError_t launch_label_row(const LabelParams &p, hipStream_t) {
    ++stub::n_label_rows;
    // everything the kernels write
    memset(p.retry, 0xEE, (size_t)p.n * 8);
    if (p.order) memset(p.order, 0xEE, (size_t)p.n * 4);
    memset(p.group, 0xEE, (size_t)kLabelGroups * 4);
    for (uint32_t i = 0; i < p.n; ++i) p.label[i] = 7u << 8;
    return hipGetLastError();
}
hipError_t launch_moment_reset(uint32_t n, const float *x, const float *y, const float *z, float *x0,
                               float *disp, float *mom, float *momc, float *mag, hipStream_t) {
    for (uint32_t i = 0; i < n; ++i) { x0[i] = x[i]; x0[n + i] = y[i]; x0[2 * n + i] = z[i]; mag[i] = 1.0f; }
    for (size_t i = 0; i < 3 * (size_t)n; ++i) disp[i] = mom[i] = momc[i] = 0.0f;
    return hipGetLastError();
}
hipError_t launch_moment_signal(uint32_t, const float *, const float *, const float *, float,
                                const uint32_t *, uint32_t ndir, const float *, float, double *partial,
                                uint32_t n_blocks, double *out, hipStream_t) {
    for (size_t k = 0; k < (size_t)ndir * n_blocks * 15; ++k) partial[k] = 0.0;
    for (size_t k = 0; k < (size_t)ndir * 15; ++k) out[k] = 1.0;
    return hipGetLastError();
}
hipError_t launch_pack_state(uint32_t n, const uint32_t *x, const uint32_t *y, const uint32_t *z,
                             const uint32_t *mag, const uint32_t *phase, const uint32_t *label,
                             const uint32_t *id, const uint32_t *flags, uint32_t *out_flags,
                             uint32_t *pos, uint32_t *spins, hipStream_t) {
    memcpy(out_flags, flags, 16);
    for (uint32_t j = 0; j < n; ++j) {
        const size_t i = 3 * (size_t)(id ? id[j] : j);
        if (pos) { pos[i] = x[j]; pos[i + 1] = y[j]; pos[i + 2] = z[j]; }
        if (spins) {
            spins[i] = mag[j];
            spins[i + 1] = phase[j];
            spins[i + 2] = (label[j] & 0xFFu) | (label[j] >> 8 << 16);
        }
    }
    return hipGetLastError();
}
hipError_t launch_phase_gemm(const float *, uint32_t, uint32_t n_pad, uint32_t, uint32_t,
                             const uint16_t *, const uint16_t *, uint32_t, uint32_t, uint32_t n_wave,
                             float *phase, uint32_t *comp, bool, hipStream_t) {
    for (size_t k = 0; k < (size_t)n_pad * n_wave; ++k) phase[k] = (float)k;
    for (size_t k = 0; k < (size_t)n_pad / 2 * n_wave; ++k) comp[k] = (uint32_t)k * 2654435761u;
    return hipGetLastError();
}
hipError_t launch_phase_operands(const float *, uint32_t, uint32_t, uint32_t, float, uint16_t *,
                                 uint16_t *, double *, hipStream_t) {
    return hipGetLastError();
}
hipError_t launch_phase_rows(uint32_t s0, uint32_t m, const float *phase, const uint32_t *comp,
                             uint32_t n_wave, uint32_t n_wpad, float *p_out, float *c_out,
                             hipStream_t) {
    for (uint32_t r = 0; r < m; ++r)
        for (uint32_t w = 0; w < n_wave; ++w) {
            if (p_out) p_out[(size_t)r * n_wave + w] = phase[(size_t)(s0 + r) * n_wpad + w];
            const uint32_t word = comp[(size_t)((s0 + r) / 2) * n_wpad + w];
            const uint32_t bits = ((s0 + r) & 1u) ? word & 0xffff0000u : word << 16;
            if (c_out) memcpy(&c_out[(size_t)r * n_wave + w], &bits, 4);
        }
    return hipGetLastError();
}
hipError_t launch_phase_signal(uint32_t, const float *, uint32_t n_wave, const double *, const float *,
                               const uint32_t *, const float *, const uint32_t *, double *, uint32_t,
                               double *out, hipStream_t) {
    for (size_t k = 0; k < (size_t)n_wave * 15; ++k) out[k] = 1.0;
    return hipGetLastError();
}
hipError_t launch_signal(uint32_t, const float *, const float *, const uint32_t *, double *partial,
                         uint32_t n_blocks, double *out, hipStream_t) {
    for (size_t k = 0; k < (size_t)n_blocks * 15; ++k) partial[k] = 0.0;
    for (int k = 0; k < 15; ++k) out[k] = 1.0;
    return hipGetLastError();
}
hipError_t sort_temp_bytes(uint32_t n, size_t *bytes) { *bytes = (size_t)n * 4; return hipSuccess; }
// The permutation that turns the order round.
hipError_t launch_sort_perm(const StepParams &p, uint32_t *, uint32_t *, uint32_t *vals_a, uint32_t *,
                            void *, size_t, hipStream_t, const uint32_t **perm) {
    for (uint32_t i = 0; i < p.n; ++i) vals_a[i] = p.n - 1 - i;
    *perm = vals_a;
    return hipGetLastError();
}
// A step moves spin s to (s, s + 1, s + 2) and raises stub::flag_bits.
hipError_t launch_step(const StepParams &p, uint32_t iters, int, int, int, int, bool, hipStream_t) {
    *p.flags |= stub::flag_bits;
    for (uint32_t i = 0; i < p.n; ++i) {
        p.x[i] = (float)p.spin_id[i];
        p.y[i] = p.x[i] + 1.0f;
        p.z[i] = p.x[i] + 2.0f;
    }
    // rows 3 * step + axis of the launch, in the tiles' chunks; each holds its number
    for (uint32_t k = 0; p.traj && k < 3 * iters; ++k)
        for (uint32_t i = 0; i < p.n; ++i) {
            const uint32_t id = p.spin_id[i];
            p.traj[(size_t)(id / kTrajTile) * p.traj_stride +
                   (size_t)(k / kTrajChunk) * (kTrajTile * kTrajChunk) +
                   (id % kTrajTile) * kTrajChunk + k % kTrajChunk] = (float)(3 * p.step0 + k);
        }
    return hipGetLastError();
}
hipError_t launch_walk_batch(const WalkTable *, uint32_t, bool, int, hipStream_t) {
    return hipGetLastError();
}
}  // namespace dsim

namespace dsim_host {
int build_walk_tables(dsim_substrate *S, hipStream_t) {
    if (!stub::keep_rows) return DSIM_OK;
    if (int rc = S->rows.start.alloc(16)) return rc;
    if (int rc = S->rows.tri.alloc(4)) return rc;
    return S->rows.box.alloc(4);
}
int build_row_lists(const dsim_substrate *, RowLists &R, uint64_t, uint64_t room, hipStream_t) {
    if (!pool_room(stub::row_bytes + 96, room)) return DSIM_OK;
    ++stub::n_row_builds;
    if (int rc = R.start.alloc(16)) return rc;
    if (int rc = R.tri.alloc(4)) return rc;
    return R.box.alloc(stub::row_bytes / 16 + 1);
}
}  // namespace dsim_host
