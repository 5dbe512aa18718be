// Waveform phases of the dsim C ABI (include/dsim_phase.h): one walk of a
// simulation handle, its displacement recorded chunk by chunk and multiplied
// by the waveforms' gradients on the matrix cores (k_phase_gemm), FP64
// readout (k_phase_partial).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "../../include/dsim.h"
#include "../../include/dsim_phase.h"
#include "dsim_internal.h"
#include "host_common.h"
#include "sim_internal.h"

using dsim_host::PoolBuf;
using dsim_host::fail;

struct dsim_waveforms {
    dsim_sim *sim = nullptr;
    uint32_t n = 0, n_pad = 0, n_wave = 0, n_steps = 0, chunk = 0, done = 0;
    uint32_t n_wpad = 0;          // waveforms padded with zero ones to a multiple of kPhaseTileN
    uint32_t buffer = 0;          // steps walked per trajectory buffer (a multiple of chunk)
    // One allocation: gsum [n_wpad][3], sum_t pc * G_w(t); the readout's partial
    // sums and out [n_wpad][15]; the bf16 halves g_hi, g_lo [n_wpad][3*n_steps]
    // of the gradients, pc folded in.
    PoolBuf<double> work;
    double *gsum = nullptr, *partial = nullptr, *out = nullptr;
    uint16_t *g_hi = nullptr, *g_lo = nullptr;
    PoolBuf<float> traj;          // n_pad / kTrajTile tiles of [3*len][kTrajTile] (len <= buffer)
    // phase [n_pad][n_wpad] (rows past n: padding), and after it comp
    // [n_pad / 2][n_wpad]: Kahan compensation of spins 2m, 2m + 1 as bf16 in the
    // low and high half.  Written by the first product, which starts from zero.
    PoolBuf<float> phase;
    uint32_t *comp = nullptr;
    bool empty = true;            // no product yet: the pairs are zero and not in memory
    double walk_ms = 0.0, gemm_ms = 0.0;
    ~dsim_waveforms() {
        work.release(); traj.release(); phase.release();
    }
};

namespace {

constexpr uint32_t kPhaseBlocks = 512;  // spin blocks of the readout

// Of get_phase's row blocks, at most (two rows, if those are more).
constexpr uint64_t kStagingBytes = 64ull << 20;

// The pairs before any product, for a readout: zero.
int clear_pairs(dsim_waveforms *W, hipStream_t st) {
    if (!W->empty) return DSIM_OK;
    HIP_TRY(hipMemsetAsync(W->phase.p, 0, W->phase.n * 4, st));
    W->empty = false;
    return DSIM_OK;
}

// The pairs copied at their stride, without device memory.  The stream is idle.
int get_phase_strided(dsim_waveforms *W, float *phase, float *comp) {
    HIP_TRY(hipStreamSynchronize(dsim_host::sim_stream(W->sim)));
    const size_t row = (size_t)W->n_wave * 4, pad = (size_t)W->n_wpad * 4;
    if (phase)
        HIP_TRY(hipMemcpy2D(phase, row, W->phase.p, pad, row, W->n, hipMemcpyDeviceToHost));
    // a row holds two spins, in its halves
    const uint32_t pairs = (W->n + 1) / 2;
    std::vector<uint32_t> v;
    for (uint32_t p0 = 0, m; comp && p0 < pairs; p0 += m) {
        m = std::min<uint32_t>(pairs - p0, (uint32_t)std::max<uint64_t>(kStagingBytes / pad, 1));
        v.resize((size_t)m * W->n_wpad);
        HIP_TRY(hipMemcpy(v.data(), W->comp + (size_t)p0 * W->n_wpad, v.size() * 4,
                          hipMemcpyDeviceToHost));
        for (uint32_t s = 2 * p0; s < std::min(W->n, 2 * (p0 + m)); ++s)
            for (uint32_t w = 0; w < W->n_wave; ++w) {
                const uint32_t word = v[(size_t)(s / 2 - p0) * W->n_wpad + w];
                const uint32_t bits = (s & 1u) ? word & 0xffff0000u : word << 16;
                memcpy(&comp[(size_t)s * W->n_wave + w], &bits, 4);
            }
    }
    return DSIM_OK;
}

}  // namespace

extern "C" int dsim_waveforms_create(dsim_sim *sim, uint32_t n_wave, uint32_t n_steps,
                                     const float *grads, float pc, uint32_t chunk,
                                     dsim_waveforms **out) {
    if (!sim || !grads || !out) return fail(DSIM_ERR_ARG, "NULL argument");
    *out = nullptr;
    if (n_wave == 0) return fail(DSIM_ERR_ARG, "n_wave must be positive");
    if (chunk == 0 || chunk % dsim::kPhaseSliceK || n_steps == 0 || n_steps % dsim::kPhaseSliceK)
        return fail(DSIM_ERR_ARG, "chunk_steps and n_steps must be multiples of %u",
                    dsim::kPhaseSliceK);
    auto *W = new dsim_waveforms();
    W->sim = sim;
    W->n = dsim_host::sim_spins(sim);
    W->n_pad = (W->n + dsim::kPhaseTileM - 1) / dsim::kPhaseTileM * dsim::kPhaseTileM;
    W->n_wave = n_wave;
    // the GEMM's waveform tiles take 128 waveforms (256 where they divide into
    // those); zero waveforms fill the last tile and are never read out
    const uint32_t nwp = (n_wave + dsim::kPhaseTileN - 1) / dsim::kPhaseTileN * dsim::kPhaseTileN;
    W->n_wpad = nwp;
    W->n_steps = n_steps;
    W->chunk = chunk;
    W->buffer = chunk;
    const size_t K = (size_t)3 * n_steps, ng = (size_t)nwp * K;
    const size_t nw = (size_t)std::max<uint32_t>(W->n_pad, 1) * nwp;
    const size_t n_sum = (size_t)nwp * 3, n_part = (size_t)kPhaseBlocks * nwp * 15;
    const size_t n_out = (size_t)nwp * 15;
    const size_t n_given = (size_t)n_steps * n_wave * 3;
    PoolBuf<float> g;  // the gradients as given, where the pairs have no room for them
    int rc;
    if ((rc = W->work.alloc(n_sum + n_part + n_out + (2 * ng * 2 + 7) / 8)) ||
        (rc = W->traj.alloc((size_t)3 * chunk * W->n_pad)) ||
        (rc = W->phase.alloc(nw + (size_t)std::max<uint32_t>(W->n_pad / 2, 1) * nwp)) ||
        (W->phase.n < n_given && (rc = g.alloc(n_given)))) {
        delete W;
        return rc;
    }
    float *given = g.p ? g.p : W->phase.p;  // nothing is in the pairs yet
    W->gsum = W->work.p;
    W->partial = W->gsum + n_sum;
    W->out = W->partial + n_part;
    W->g_hi = reinterpret_cast<uint16_t *>(W->out + n_out);
    W->g_lo = W->g_hi + ng;
    W->comp = reinterpret_cast<uint32_t *>(W->phase.p + nw);
    // The trajectory needs no clearing: padded spins reach only padded rows of
    // the pairs, which nothing reads.
    hipStream_t st = dsim_host::sim_stream(sim);
    hipError_t e = hipMemcpyAsync(given, grads, n_given * 4, hipMemcpyHostToDevice, st);
    if (e == hipSuccess)
        e = dsim::launch_phase_operands(given, n_steps, n_wave, nwp, pc, W->g_hi, W->g_lo, W->gsum, st);
    const hipError_t es = hipStreamSynchronize(st);
    if (e == hipSuccess) e = es;
    g.release();
    if (e != hipSuccess) {
        delete W;
        return fail(DSIM_ERR_HIP, "waveform init: %s", hipGetErrorString(e));
    }
    *out = W;
    return DSIM_OK;
}

extern "C" int dsim_waveforms_set_buffer(dsim_waveforms *W, uint32_t buffer_steps) {
    if (!W) return fail(DSIM_ERR_ARG, "NULL waveforms");
    if (buffer_steps == 0 || buffer_steps % W->chunk)
        return fail(DSIM_ERR_ARG, "buffer_steps must be a positive multiple of chunk_steps (%u)",
                    W->chunk);
    if (buffer_steps == W->buffer && (W->traj.p || !W->n_pad)) return DSIM_OK;
    HIP_TRY(hipStreamSynchronize(dsim_host::sim_stream(W->sim)));
    W->traj.release();
    if (int rc = W->traj.alloc((size_t)3 * buffer_steps * W->n_pad)) {
        // the buffer as it was, or the smallest; a run without any is refused
        if (W->traj.alloc((size_t)3 * W->buffer * W->n_pad)) {
            W->buffer = W->chunk;
            (void)W->traj.alloc((size_t)3 * W->buffer * W->n_pad);
        }
        return rc;
    }
    W->buffer = buffer_steps;
    return DSIM_OK;
}

extern "C" int dsim_waveforms_destroy(dsim_waveforms *W) {
    if (!W) return DSIM_OK;
    (void)hipStreamSynchronize(dsim_host::sim_stream(W->sim));  // the blocks go back to the pool
    delete W;
    return DSIM_OK;
}

extern "C" int dsim_waveforms_run(dsim_waveforms *W, uint32_t steps, float *traj_out) {
    if (!W) return fail(DSIM_ERR_ARG, "NULL waveforms");
    if (steps % dsim::kPhaseSliceK || W->done + steps > W->n_steps)
        return fail(DSIM_ERR_ARG, "steps must be a multiple of %u within the waveforms' %u",
                    dsim::kPhaseSliceK, W->n_steps);
    if (W->n_pad && !W->traj.p) return fail(DSIM_ERR_NOMEM, "no trajectory buffer");
    hipStream_t st = dsim_host::sim_stream(W->sim);
    hipEvent_t ev[3];
    for (auto &e : ev) HIP_TRY(hipEventCreate(&e));
    int rc = DSIM_OK;
    for (uint32_t c = 0; c < steps && rc == DSIM_OK;) {
        const uint32_t len = std::min(W->buffer, steps - c);  // a multiple of 32
        HIP_TRY(hipEventRecord(ev[0], st));
        if ((rc = dsim_host::sim_walk_traj(W->sim, len, W->traj.p))) break;
        HIP_TRY(hipEventRecord(ev[1], st));
        hipError_t e = dsim::launch_phase_gemm(W->traj.p, W->n, W->n_pad, 3 * len, 3 * W->chunk,
                                               W->g_hi, W->g_lo, 3 * W->n_steps, 3 * W->done,
                                               W->n_wpad, W->phase.p, W->comp, W->empty, st);
        if (e == hipSuccess) W->empty = false;
        if (e != hipSuccess) {
            rc = fail(DSIM_ERR_HIP, "phase GEMM: %s", hipGetErrorString(e));
            break;
        }
        HIP_TRY(hipEventRecord(ev[2], st));
        if (traj_out) {
            // rows [3 * len][n] out of the spin tiles' 16-byte k chunks
            const size_t tile = (size_t)3 * len * dsim::kTrajTile;  // floats per tile
            std::vector<float> h(tile * (W->n_pad / dsim::kTrajTile));
            HIP_TRY(hipMemcpyAsync(h.data(), W->traj.p, h.size() * 4, hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
            for (uint32_t r = 0; r < 3 * len; ++r) {
                float *dst = traj_out + ((size_t)3 * c + r) * W->n;
                const size_t kc = (size_t)(r / dsim::kTrajChunk) * dsim::kTrajTile * dsim::kTrajChunk +
                                  r % dsim::kTrajChunk;
                for (uint32_t s = 0; s < W->n; ++s)
                    dst[s] = h[(s / dsim::kTrajTile) * tile + kc +
                               (size_t)(s % dsim::kTrajTile) * dsim::kTrajChunk];
            }
        }
        HIP_TRY(hipEventSynchronize(ev[2]));
        float a = 0.f, b = 0.f;
        HIP_TRY(hipEventElapsedTime(&a, ev[0], ev[1]));
        HIP_TRY(hipEventElapsedTime(&b, ev[1], ev[2]));
        W->walk_ms += a;
        W->gemm_ms += b;
        W->done += len;
        c += len;
    }
    for (auto &e : ev) (void)hipEventDestroy(e);
    if (rc) return rc;
    return dsim_sync(W->sim);
}

extern "C" int dsim_waveforms_signal(dsim_waveforms *W, double *out) {
    if (!W || !out) return fail(DSIM_ERR_ARG, "NULL argument");
    const float *mag, *x0;
    const uint32_t *label, *id;
    dsim_host::sim_readout_fields(W->sim, &mag, &label, &x0, &id);
    hipStream_t st = dsim_host::sim_stream(W->sim);
    const uint32_t nb = std::max<uint32_t>(1, std::min<uint32_t>(kPhaseBlocks, W->n));
    if (int rc = clear_pairs(W, st)) return rc;
    hipError_t e = dsim::launch_phase_signal(W->n, W->phase.p, W->n_wpad, W->gsum, mag, label, x0, id,
                                             W->partial, nb, W->out, st);
    if (e != hipSuccess) return fail(DSIM_ERR_HIP, "phase readout: %s", hipGetErrorString(e));
    std::vector<double> v((size_t)W->n_wpad * 15);
    HIP_TRY(hipMemcpyAsync(v.data(), W->out, v.size() * 8, hipMemcpyDeviceToHost, st));
    if (int rc = dsim_sync(W->sim)) return rc;
    for (uint32_t w = 0; w < W->n_wave; ++w) {
        const double *q = &v[(size_t)w * 15];
        for (int k = 0; k < 5; ++k)
            out[(size_t)w * 5 + k] =
                q[10 + k] == 0.0 ? 0.0 : std::sqrt(q[k] * q[k] + q[5 + k] * q[5 + k]) / q[10 + k];
    }
    return DSIM_OK;
}

extern "C" int dsim_waveforms_get_phase(dsim_waveforms *W, float *phase, float *comp) {
    if (!W) return fail(DSIM_ERR_ARG, "NULL waveforms");
    if (int rc = dsim_sync(W->sim)) return rc;
    if (!W->n || (!phase && !comp)) return DSIM_OK;
    hipStream_t st = dsim_host::sim_stream(W->sim);
    if (int rc = clear_pairs(W, st)) return rc;
    // blocks of whole spin pairs, without the padded waveforms, through a
    // staging buffer: a copy of rows at a stride takes the runtime about 5 us
    // a row
    const uint64_t row = (uint64_t)W->n_wave * 4, both = row * ((phase ? 1 : 0) + (comp ? 1 : 0));
    const uint32_t rows = (uint32_t)std::min<uint64_t>((W->n + 1u) & ~1u,
                                                       std::max<uint64_t>(kStagingBytes / both & ~1ull, 2));
    PoolBuf<float> stage;
    if (int rc = stage.alloc(rows * both / 4))
        return rc == DSIM_ERR_NOMEM ? get_phase_strided(W, phase, comp) : rc;
    float *c_stage = stage.p + (phase ? (size_t)rows * W->n_wave : 0);
    hipError_t e = hipSuccess;
    for (uint32_t s0 = 0; s0 < W->n && e == hipSuccess; s0 += rows) {
        const uint32_t m = std::min(rows, W->n - s0);
        const size_t bytes = (size_t)m * row, at = (size_t)s0 * W->n_wave;
        e = dsim::launch_phase_rows(s0, m, W->phase.p, W->comp, W->n_wave, W->n_wpad,
                                    phase ? stage.p : nullptr, comp ? c_stage : nullptr, st);
        if (e == hipSuccess && phase)
            e = hipMemcpyAsync(phase + at, stage.p, bytes, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess && comp)
            e = hipMemcpyAsync(comp + at, c_stage, bytes, hipMemcpyDeviceToHost, st);
    }
    const hipError_t es = hipStreamSynchronize(st);
    if (e == hipSuccess) e = es;
    stage.release();
    if (e != hipSuccess) return fail(DSIM_ERR_HIP, "phase copy: %s", hipGetErrorString(e));
    return DSIM_OK;
}

extern "C" int dsim_waveforms_timing(dsim_waveforms *W, double *walk_ms, double *gemm_ms) {
    if (!W) return fail(DSIM_ERR_ARG, "NULL waveforms");
    if (walk_ms) *walk_ms = W->walk_ms;
    if (gemm_ms) *gemm_ms = W->gemm_ms;
    return DSIM_OK;
}
