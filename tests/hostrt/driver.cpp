// Checks of the library's host code over the host-memory runtime: one case by
// name, or all of them.
#include "stub_hip.h"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "../../dsim_amd/csrc/host_common.h"
#include "../../dsim_amd/csrc/sim_internal.h"
#include "../../include/dsim.h"
#include "../../include/dsim_phase.h"
#include "../../include/dsim_serve.h"

static int fails = 0;
#define EXPECT(c)                                                              \
    do {                                                                       \
        if (!(c)) {                                                            \
            fprintf(stderr, "FAILED %s:%d: %s (%s)\n", __FILE__, __LINE__, #c, \
                    dsim_last_error());                                        \
            ++fails;                                                           \
        }                                                                      \
    } while (0)

using dsim_host::PoolBuf;

static int device_of(const void *p) { return stub::blocks.at(const_cast<void *>(p)).device; }

static dsim_substrate *make_sub(uint32_t kind = DSIM_GRID_AABB, uint32_t n_tri = 0) {
    std::vector<float> v(3 * 3 * (size_t)n_tri);
    std::vector<uint32_t> t(3 * (size_t)n_tri), info(3 * (size_t)n_tri, 0);
    for (uint32_t k = 0; k < 3 * n_tri; ++k) {
        t[k] = k;
        for (int a = 0; a < 3; ++a) v[3 * k + a] = 0.1f * (float)((k * 7 + a * 3) % 11) - 0.5f;
    }
    dsim_mesh m{3 * n_tri, v.data(), n_tri, t.data(), info.data()};
    dsim_grid_params g{};
    g.kind = kind;
    for (int k = 0; k < 3; ++k) { g.dims[k] = 4; g.lo[k] = -1.0f; g.cell[k] = 0.5f; }
    dsim_substrate *s = nullptr;
    EXPECT(dsim_substrate_create(&m, &g, &s) == DSIM_OK);
    return s;
}

static dsim_params params(uint32_t sort = 0) {
    dsim_params p{};
    p.dt = 0.005f;
    for (int c = 0; c < 4; ++c) { p.std_dev[c] = 0.01f; p.t2[c] = INFINITY; }
    p.reflection_type = 1;
    p.mode = DSIM_MODE_PHYSICAL;
    p.boundary = DSIM_BOUNDARY_PERIODIC;
    p.rng = DSIM_RNG_PHILOX;
    p.sort_interval = sort;
    return p;
}

static dsim_sim *make_sim(dsim_substrate *s, uint32_t n, uint32_t sort = 0) {
    const dsim_params p = params(sort);
    dsim_sim *h = nullptr;
    EXPECT(dsim_sim_create(s, &p, n, &h) == DSIM_OK);
    return h;
}

// A block goes back under the device that it was allocated on, whatever device
// is current then.
static void pool_device() {
    dsim_host::pool_ref();
    PoolBuf<float> a, b, c;
    hipSetDevice(1);
    EXPECT(a.alloc(1000) == DSIM_OK);
    const void *on1 = a.p;
    hipSetDevice(0);
    a.release();
    EXPECT(b.alloc(1000) == DSIM_OK);
    EXPECT(device_of(b.p) == 0);
    hipSetDevice(1);
    EXPECT(c.alloc(1000) == DSIM_OK);
    EXPECT(c.p == on1 && device_of(c.p) == 1);
    hipSetDevice(0);
    b.release();
    c.release();
    dsim_host::pool_unref();
    EXPECT(stub::blocks.empty());
}

// Each device's idle blocks are held to its own share.
static void pool_bound() {
    dsim_host::pool_ref();
    const size_t lim[2] = {stub::total[0] / dsim_host::kPoolShare,
                           stub::total[1] / dsim_host::kPoolShare};
    std::vector<PoolBuf<uint8_t>> v[2];
    for (int d : {0, 1}) {
        hipSetDevice(d);
        v[d].resize(4);
        for (auto &b : v[d]) EXPECT(b.alloc(lim[d] / 3) == DSIM_OK);
    }
    for (int d : {0, 1}) {
        hipSetDevice(1 - d);  // the other device is current when they are given back
        for (auto &b : v[d]) b.release();
    }
    for (int d : {0, 1}) {
        EXPECT(stub::used[d] <= lim[d]);
        EXPECT(stub::used[d] >= lim[d] / 2);  // and one device does not push out the other's
    }
    hipSetDevice(0);
    dsim_host::pool_unref();
    EXPECT(stub::blocks.empty());
}

// Handles made and closed with different devices current.
static void handle_device() {
    hipSetDevice(0);
    dsim_substrate *s0 = make_sub();
    hipSetDevice(1);
    dsim_substrate *s1 = make_sub();
    dsim_sim *keep = make_sim(s1, 100), *h = make_sim(s1, 1000, 16);
    hipSetDevice(0);
    EXPECT(dsim_sim_destroy(h) == DSIM_OK);
    const size_t before = stub::used[1];
    dsim_sim *g = make_sim(s0, 1000, 16);
    EXPECT(stub::used[1] == before);
    size_t on0 = 0;
    for (auto &kv : stub::blocks) on0 += kv.second.device == 0 ? kv.second.bytes : 0;
    EXPECT(on0 >= 2 * 21 * 4 * 1000);  // both state blocks
    EXPECT(dsim_sim_destroy(g) == DSIM_OK);
    EXPECT(dsim_sim_destroy(keep) == DSIM_OK);
    EXPECT(dsim_substrate_destroy(s0) == DSIM_OK && dsim_substrate_destroy(s1) == DSIM_OK);
    EXPECT(stub::blocks.empty());
}

// Where the labeller's row lists put the triangles past the grid: never more
// than their 32-bit places hold, nor more than the grid's own size.
static void row_plan() {
    using namespace dsim_host;
    // a grid of the crossing bundles: 1600 axons
    EXPECT(row_plan(14'503'175, 16'000'000, 9'000, 60'000) == kRowsEnds);
    EXPECT(row_plan(1'000'000, 3'000'000, 0, 0) == kRowsEnds);
    // 1e5 walls across the far face of a grid of 4e4 rows: 4e9 entries
    EXPECT(row_plan(4'000'000, 3'000'000, 100'000, 4'000'000'000ull) == kRowsShared);
    // whose sum wraps to few in 32 bits
    EXPECT(row_plan(1ull << 28, 100'000'000, 1 << 20, (1ull << 32) + 5) == kRowsShared);
    EXPECT(row_plan(1ull << 28, 0xFFFFFF00ull - 10, 5, 11) == kRowsShared);
    EXPECT(row_plan(1ull << 28, 0xFFFFFF00ull - 10, 10, 10) == kRowsEnds);
    EXPECT(row_plan(1ull << 28, 0xFFFFFF00ull - 10, 11, 11) == kRowsNone);
    EXPECT(row_plan(1ull << 28, 0xFFFFFFFFull, 2, 2) == kRowsNone);
    EXPECT(row_plan(100, 50, 10, 150) == kRowsEnds);
    EXPECT(row_plan(100, 50, 10, 151) == kRowsShared);
    EXPECT(row_plan(1ull << 28, 1ull << 28, 10, kRowEndsMax) == kRowsEnds);
    EXPECT(row_plan(1ull << 28, 1ull << 28, 10, kRowEndsMax + 1) == kRowsShared);
}

// An error flag of a step comes out of the next call that waits, once: on its
// own, beside a signal's sums, in front of a state read in one copy (256 spins)
// or in several (100,000), and before the caller's arrays are written.
static void error_flags() {
    dsim_substrate *s = make_sub();
    for (uint32_t n : {256u, 100000u}) {
        std::vector<float> pos(3 * n);
        std::vector<dsim_spin_data> spins(n);
        for (uint32_t bits : {1u, 4u}) {
            const int code = bits == 1 ? DSIM_ERR_OVERFLOW : DSIM_ERR_STATE;
            const char *word = bits == 1 ? "4096 collisions" : "out of range";
            dsim_sim *h = make_sim(s, n);
            EXPECT(dsim_init_spins_uniform(h, 1.0f) == DSIM_OK);
            const float g[3] = {0, 0, 0};
            for (int how = 0; how < 6; ++how) {
                stub::flag_bits = bits;
                EXPECT(dsim_integrate(h, g, 0.0f, 1) == DSIM_OK);
                stub::flag_bits = 0;
                double sig[5] = {-1, -1, -1, -1, -1};
                pos.assign(3 * n, -7.0f);
                memset(spins.data(), 0x5A, n * sizeof spins[0]);
                const int rc = how == 0   ? dsim_sync(h)
                               : how == 1 ? dsim_signal(h, sig)
                               : how == 2 ? dsim_get_state_aos(h, pos.data(), spins.data(), nullptr)
                               : how == 3 ? dsim_get_state_aos(h, nullptr, spins.data(), nullptr)
                               : how == 4 ? dsim_get_state_aos(h, pos.data(), nullptr, nullptr)
                                          : dsim_get_state_aos(h, nullptr, nullptr, nullptr);
                EXPECT(rc == code && strstr(dsim_last_error(), word));
                EXPECT(sig[0] == -1 && pos[0] == -7.0f && pos[3 * n - 1] == -7.0f);
                EXPECT(spins[n - 1].insideFiber == 0x5A5A);
                EXPECT(dsim_sync(h) == DSIM_OK && dsim_signal(h, sig) == DSIM_OK);
                EXPECT(dsim_get_state_aos(h, pos.data(), spins.data(), nullptr) == DSIM_OK);
                EXPECT(pos[3 * n - 1] == (float)(n - 1) + 2.0f);
            }
            EXPECT(dsim_sim_destroy(h) == DSIM_OK);
        }
    }
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// Labelling takes no device memory of its own: it works on a full device, with
// spin counts that leave its per-spin words unaligned, and leaves the fields it
// does not end as they were.
static void label_on_a_full_device() {
    stub::keep_rows = true;
    dsim_substrate *s = make_sub();
    stub::keep_rows = false;
    for (uint32_t n : {1u, 2u, 7u, 1000u, 40001u}) {
        dsim_sim *h = make_sim(s, n);
        EXPECT(dsim_init_spins_uniform(h, 1.0f) == DSIM_OK && dsim_moment_reset(h) == DSIM_OK);
        const float *mag, *x0;
        const uint32_t *label, *id;
        dsim_host::sim_readout_fields(h, &mag, &label, &x0, &id);
        const size_t was = stub::capacity[0];
        const uint32_t rows = stub::n_label_rows;
        stub::capacity[0] = stub::used[0];
        uint32_t amb = 77;
        EXPECT(dsim_label_spins(h, 1, 1, 1, 3, &amb) == DSIM_OK && amb == 0);
        stub::capacity[0] = was;
        EXPECT(stub::n_label_rows == rows + 1);
        bool same = true;
        for (uint32_t i = 0; i < n; ++i)
            same &= mag[i] == 1.0f && label[i] == 7u << 8 && id[i] == i && x0[2 * n + i] == 0.25f;
        EXPECT(same);
        double sig[5];
        EXPECT(dsim_integrate_moment(h, 1.0f, 1) == DSIM_ERR_STATE);  // the moments have ended
        const float g[3] = {1, 0, 0};
        EXPECT(dsim_signal_moment(h, 1, g, 1.0f, sig) == DSIM_ERR_STATE);
        EXPECT(dsim_moment_reset(h) == DSIM_OK && dsim_integrate_moment(h, 1.0f, 1) == DSIM_OK);
        EXPECT(dsim_sim_destroy(h) == DSIM_OK);
    }
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// A labelling that finds no memory for the row lists of a large grid goes
// through the pass over all triangles, which needs none; no error stays behind.
static void label_without_lists() {
    dsim_substrate *s = make_sub();
    dsim_sim *h = make_sim(s, 1000);
    EXPECT(dsim_init_spins_uniform(h, 1.0f) == DSIM_OK);
    stub::row_bytes = 1 << 20;
    const size_t was = stub::capacity[0];
    const uint32_t rows = stub::n_label_rows, all = stub::n_label_all;
    for (size_t room : {(size_t)0, (size_t)100, (size_t)1 << 19}) {  // none, and for a part of them
        stub::capacity[0] = stub::used[0] + room;
        EXPECT(dsim_label_spins(h, 1, 1, 1, 3, nullptr) == DSIM_OK);
    }
    stub::capacity[0] = was;
    EXPECT(stub::n_label_rows == rows && stub::n_label_all == all + 3);
    EXPECT(dsim_label_spins(h, 1, 1, 1, 3, nullptr) == DSIM_OK);
    EXPECT(stub::n_label_rows == rows + 1 && stub::n_label_all == all + 3);
    EXPECT(dsim_sim_destroy(h) == DSIM_OK);
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// A server's budget holds for all that its requests' handles take: their own
// blocks, those that wait for the next handle, and row lists that a labelling
// makes; lists that the budget has no room for are gone without.
static void server_budget() {
    dsim_substrate *s = make_sub();
    const float lobe[1] = {1.0f}, g[60] = {1};
    const uint32_t steps[1] = {300};
    // the last: handles of 6100 spins in blocks that were of 8000, beside one of 8000
    for (uint64_t rows : {0ull, 200'000ull, 5'000'000ull, 1ull}) {
        stub::row_bytes = rows;
        const bool tight = rows == 1;
        dsim_params p = params();
        const uint64_t one = dsim_host::sim_footprint(8000, &p, 20);
        const uint64_t budget = tight ? one + dsim_host::sim_footprint(6100, &p, 20) + 1000
                                      : 2 * one + one / 2;
        dsim_server *S = nullptr;
        EXPECT(dsim_server_create(budget, 0, 0, &S) == DSIM_OK);
        uint32_t id = 0;
        EXPECT(dsim_server_add_substrate(S, s, &id) == DSIM_OK);
        std::vector<uint64_t> tickets;
        auto submit = [&](uint32_t n) {
            dsim_request q{};
            q.substrate = id;
            q.n_spins = n;
            q.dt = 0.005f;
            for (int c = 0; c < 4; ++c) { q.std_dev[c] = 0.01f; q.t2[c] = INFINITY; }
            q.boundary = DSIM_BOUNDARY_PERIODIC;
            q.start_box = 1.0f;
            for (int k = 0; k < 3; ++k) q.label_extent[k] = 1.0f;
            q.n_lobes = 1;
            q.lobe_weight = lobe;
            q.lobe_steps = steps;
            q.n_lines = 20;
            q.grads = g;
            tickets.emplace_back();
            EXPECT(dsim_server_submit(S, &q, &tickets.back()) == DSIM_OK);
        };
        submit(100);  // brings the job table, which is not a request's
        uint32_t active = 1, queued = 1;
        while (active || queued) EXPECT(dsim_server_round(S, &active, &queued) == DSIM_OK);
        dsim_host::pool_trim_to(0, 0);
        const size_t base = stub::used[0];
        stub::peak[0] = base;
        // falling and rising sizes: handles in blocks that were larger ones'
        const uint32_t builds = stub::n_row_builds, all = stub::n_label_all;
        for (uint32_t k = 0, u = 1; k < 200; ++k) {
            u = u * 1664525u + 1013904223u;
            submit(tight ? (k % 3 == 1 ? 6100 : 8000) : 1000 + (u >> 8) % 7001);
            if (tight && k % 3 == 0)
                for (active = 1; active;) EXPECT(dsim_server_round(S, &active, &queued) == DSIM_OK);
            if (tight && k % 3 == 1) EXPECT(dsim_server_round(S, &active, &queued) == DSIM_OK);
        }
        active = queued = 1;
        size_t rounds = 0;
        while (active || queued) {
            EXPECT(dsim_server_round(S, &active, &queued) == DSIM_OK);
            if (++rounds > 1000) break;
        }
        EXPECT(rounds <= 1000);
        EXPECT(stub::peak[0] - base <= budget);
        if (stub::peak[0] - base > budget)
            fprintf(stderr, "lists %llu: %zu of %llu\n", (unsigned long long)rows,
                    stub::peak[0] - base, (unsigned long long)budget);
        for (uint64_t t : tickets) EXPECT(dsim_server_wait(S, t, 0) == DSIM_OK);
        if (rows > budget) EXPECT(stub::n_row_builds == builds && stub::n_label_all == all + 200);
        else if (!tight) EXPECT(stub::n_row_builds > builds);
        EXPECT(dsim_server_destroy(S) == DSIM_OK);
    }
    stub::row_bytes = 0;
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// State read-back on a full device: the same words, in spin order too.
static void state_on_a_full_device() {
    dsim_substrate *s = make_sub();
    for (uint32_t n : {1u, 1000u, 100001u})
        for (uint32_t sort : {0u, 1u}) {
            dsim_sim *h = make_sim(s, n, sort);
            std::vector<float> pos(3 * n), p2(3 * n, -1.0f);
            std::vector<dsim_spin_data> spins(n), s2(n);
            for (uint32_t i = 0; i < n; ++i) {
                memset(&spins[i], 0, sizeof spins[i]);
                memset(&s2[i], 0x5A, sizeof s2[i]);
                for (int k = 0; k < 3; ++k) pos[3 * i + k] = (float)(i + k);
                spins[i].signalMagnitude = (float)i + 0.5f;
                spins[i].signalPhase = -(float)i;
                spins[i].compartmentType = i % 4;
                spins[i].insideFiber = (uint16_t)(i * 7);
            }
            EXPECT(dsim_set_state_aos(h, pos.data(), spins.data(), nullptr) == DSIM_OK);
            const float g[3] = {0, 0, 0};
            EXPECT(dsim_integrate(h, g, 0.0f, 3) == DSIM_OK);  // sorted: three reorders
            const size_t was = stub::capacity[0];
            stub::capacity[0] = stub::used[0];
            EXPECT(dsim_get_state_aos(h, p2.data(), s2.data(), nullptr) == DSIM_OK);
            EXPECT(pos == p2 && !memcmp(spins.data(), s2.data(), n * sizeof spins[0]));
            p2.assign(3 * n, -1.0f);
            EXPECT(dsim_get_state_aos(h, p2.data(), nullptr, nullptr) == DSIM_OK && pos == p2);
            EXPECT(dsim_sync(h) == DSIM_OK);
            stub::capacity[0] = was;
            memset(s2.data(), 0x5A, n * sizeof s2[0]);
            EXPECT(dsim_get_state_aos(h, nullptr, s2.data(), nullptr) == DSIM_OK);
            EXPECT(!memcmp(spins.data(), s2.data(), n * sizeof spins[0]));
            EXPECT(dsim_sim_destroy(h) == DSIM_OK);
        }
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// Phases read back through staging of at most 64 MB, whichever of the two
// arrays is asked for, and on a full device.
static void phases_read_back() {
    dsim_substrate *s = make_sub();
    for (uint32_t n : {1u, 8191u, 20001u}) {
        dsim_sim *h = make_sim(s, n);
        EXPECT(dsim_init_spins_uniform(h, 1.0f) == DSIM_OK && dsim_moment_reset(h) == DSIM_OK);
        const uint32_t nw = 1003;
        std::vector<float> g((size_t)32 * nw * 3, 1.0f);
        dsim_waveforms *W = nullptr;
        EXPECT(dsim_waveforms_create(h, nw, 32, g.data(), 1.0f, 32, &W) == DSIM_OK);
        EXPECT(dsim_waveforms_run(W, 32, nullptr) == DSIM_OK);
        dsim_host::pool_trim_to(0, 0);
        const size_t m = (size_t)n * nw, was = stub::capacity[0], used = stub::used[0];
        std::vector<float> p0(m), c0(m), p(m), c(m);
        stub::peak[0] = used;
        EXPECT(dsim_waveforms_get_phase(W, p0.data(), c0.data()) == DSIM_OK);
        EXPECT(stub::peak[0] - used <= 64 << 20);
        EXPECT(n < 8000 || stub::peak[0] - used > 60 << 20);
        for (bool full : {false, true})
            for (int which : {1, 2, 3}) {
                dsim_host::pool_trim_to(0, 0);
                stub::capacity[0] = full ? stub::used[0] : was;
                stub::peak[0] = stub::used[0];
                memset(p.data(), 0xA5, 4 * m);
                memset(c.data(), 0xA5, 4 * m);
                EXPECT(dsim_waveforms_get_phase(W, which & 1 ? p.data() : nullptr,
                                                which & 2 ? c.data() : nullptr) == DSIM_OK);
                EXPECT(stub::peak[0] - used <= (which == 3 || m > 16 << 20 ? 64u << 20 : 4 * (m + nw)));
                EXPECT(!(which & 1) || !memcmp(p.data(), p0.data(), 4 * m));
                EXPECT(!(which & 2) || !memcmp(c.data(), c0.data(), 4 * m));
                stub::capacity[0] = was;
            }
        EXPECT(dsim_waveforms_destroy(W) == DSIM_OK && dsim_sim_destroy(h) == DSIM_OK);
    }
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// Trajectory rows stand in their place however the steps are split into launches.
static void trajectory_launches() {
    dsim_substrate *s = make_sub();
    const uint32_t n = 200, steps = 96;
    for (uint32_t sort : {0u, 1u, 5u, 10u, 64u})
        for (uint32_t spl : {0u, 1u, 2u, 3u, 7u, 30u, 1000u}) {
            dsim_params p = params(sort);
            p.steps_per_launch = spl;
            dsim_sim *h = nullptr;
            dsim_waveforms *W = nullptr;
            EXPECT(dsim_sim_create(s, &p, n, &h) == DSIM_OK);
            EXPECT(dsim_init_spins_uniform(h, 1.0f) == DSIM_OK && dsim_moment_reset(h) == DSIM_OK);
            std::vector<float> g((size_t)2 * steps * 3, 1.0f), tr((size_t)steps * 3 * n, -1.0f);
            EXPECT(dsim_waveforms_create(h, 1, 2 * steps, g.data(), 1.0f, steps, &W) == DSIM_OK);
            for (uint32_t first : {0u, steps}) {
                EXPECT(dsim_waveforms_run(W, steps, tr.data()) == DSIM_OK);
                size_t bad = 0;
                for (size_t k = 0; k < tr.size(); ++k) bad += tr[k] != (float)(3 * first + k / n);
                EXPECT(bad == 0);
            }
            EXPECT(dsim_waveforms_destroy(W) == DSIM_OK && dsim_sim_destroy(h) == DSIM_OK);
        }
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK);
    dsim_host::pool_trim_to(0, 0);
    EXPECT(stub::blocks.empty());
}

// A waveform handle's device memory is what its header says; preparing its
// operands takes no more beside phases that are larger than the gradients.
static void waveforms_memory() {
    dsim_substrate *s = make_sub();
    for (uint32_t n : {20001u, 127u}) {
        dsim_sim *h = make_sim(s, n);
        EXPECT(dsim_init_spins_uniform(h, 1.0f) == DSIM_OK && dsim_moment_reset(h) == DSIM_OK);
        const uint32_t nw = 128, steps = 32;
        std::vector<float> g((size_t)steps * nw * 3, 1.0f);
        dsim_waveforms *W = nullptr;
        const size_t pad = (n + 127) / 128 * 128, used = stub::used[0];
        stub::peak[0] = used;
        EXPECT(dsim_waveforms_create(h, nw, steps, g.data(), 1.0f, 32, &W) == DSIM_OK);
        const size_t held = 6 * pad * nw + 4 * (size_t)nw * 3 * steps + 12 * pad * 32 +
                            8 * ((size_t)nw * 18 + 512 * (size_t)nw * 15);  // sums of the readout
        EXPECT(stub::used[0] - used == held);
        EXPECT(stub::peak[0] - used == held);
        std::vector<double> sig(5 * nw);
        EXPECT(dsim_waveforms_signal(W, sig.data()) == DSIM_OK);
        EXPECT(dsim_waveforms_destroy(W) == DSIM_OK && dsim_sim_destroy(h) == DSIM_OK);
    }
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// A buffer that cannot grow leaves the handle with one that works.
static void failed_growth() {
    dsim_substrate *s = make_sub();
    dsim_sim *h = make_sim(s, 1000);
    EXPECT(dsim_init_spins_uniform(h, 1.0f) == DSIM_OK && dsim_moment_reset(h) == DSIM_OK);
    const size_t was = stub::capacity[0];
    std::vector<float> g(3 * 4000, 1.0f);
    std::vector<double> sig(5 * 4000);
    double one[5] = {0};
    for (uint32_t lines : {4000u, 100u, 4000u}) {
        stub::capacity[0] = stub::used[0] + 100'000;  // room for the lines, not for their sums
        EXPECT(dsim_signal_moment(h, lines, g.data(), 1.0f, sig.data()) == DSIM_ERR_NOMEM);
        EXPECT(dsim_signal(h, one) == DSIM_OK && one[0] > 0);
        stub::capacity[0] = was;
        EXPECT(dsim_signal_moment(h, 90, g.data(), 1.0f, sig.data()) == DSIM_OK);
    }
    stub::capacity[0] = stub::used[0];
    EXPECT(dsim_label_spins(h, 1, 1, 1, 3, nullptr) == DSIM_OK);
    stub::capacity[0] = was;
    EXPECT(dsim_moment_reset(h) == DSIM_OK);
    std::vector<float> w((size_t)320 * 128 * 3, 1.0f);
    dsim_waveforms *W = nullptr;
    EXPECT(dsim_waveforms_create(h, 128, 320, w.data(), 1.0f, 32, &W) == DSIM_OK);
    EXPECT(dsim_waveforms_set_buffer(W, 64) == DSIM_OK);
    dsim_host::pool_trim_to(0, 0);
    stub::capacity[0] = stub::used[0];
    EXPECT(dsim_waveforms_set_buffer(W, 256) == DSIM_ERR_NOMEM);
    EXPECT(dsim_waveforms_run(W, 160, nullptr) == DSIM_OK);
    stub::capacity[0] = 0;  // not even the buffer that it had
    EXPECT(dsim_waveforms_set_buffer(W, 256) == DSIM_ERR_NOMEM);
    EXPECT(dsim_waveforms_run(W, 32, nullptr) == DSIM_ERR_NOMEM);
    stub::capacity[0] = was;
    EXPECT(dsim_waveforms_set_buffer(W, 32) == DSIM_OK);
    EXPECT(dsim_waveforms_run(W, 160, nullptr) == DSIM_OK);
    EXPECT(dsim_waveforms_destroy(W) == DSIM_OK && dsim_sim_destroy(h) == DSIM_OK);
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// The caller can have the waiting blocks given back, on every device, while
// handles are alive.
static void trim() {
    dsim_substrate *s = make_sub();
    dsim_sim *keep = make_sim(s, 10);
    size_t base[2];
    for (int d : {0, 1}) {
        hipSetDevice(d);
        base[d] = stub::used[d];
        PoolBuf<float> a, b;
        EXPECT(a.alloc(100'000) == DSIM_OK && b.alloc(1000) == DSIM_OK);
        a.release();
        b.release();
        EXPECT(stub::used[d] >= base[d] + 404'000);
    }
    hipSetDevice(0);
    EXPECT(dsim_trim_memory() == DSIM_OK);
    EXPECT(stub::used[0] == base[0] && stub::used[1] == base[1]);
    EXPECT(dsim_trim_memory() == DSIM_OK);
    EXPECT(dsim_sync(keep) == DSIM_OK && dsim_sim_destroy(keep) == DSIM_OK);
    EXPECT(dsim_substrate_destroy(s) == DSIM_OK && stub::blocks.empty());
}

// A server's handles lie on the device that was current at its creation, also
// when another thread runs its rounds.
static void server_device() {
    hipSetDevice(1);
    dsim_substrate *s = make_sub();
    dsim_server *S = nullptr;
    EXPECT(dsim_server_create(100 << 20, 0, 0, &S) == DSIM_OK);
    uint32_t id = 0;
    EXPECT(dsim_server_add_substrate(S, s, &id) == DSIM_OK);
    const float lobe[1] = {1.0f}, g[3] = {1, 0, 0};
    const uint32_t steps[1] = {300};
    for (bool background : {true, false}) {
        hipSetDevice(background ? 1 : 0);
        dsim_trim_memory();
        stub::peak[0] = stub::used[0];
        stub::peak[1] = stub::used[1];
        const size_t base = stub::used[1];
        dsim_request q{};
        q.substrate = id;
        q.n_spins = 5000;
        q.dt = 0.005f;
        for (int c = 0; c < 4; ++c) { q.std_dev[c] = 0.01f; q.t2[c] = INFINITY; }
        q.start_box = 1.0f;
        q.n_lobes = 1;
        q.lobe_weight = lobe;
        q.lobe_steps = steps;
        q.n_lines = 1;
        q.grads = g;
        uint64_t t = 0;
        EXPECT(dsim_server_submit(S, &q, &t) == DSIM_OK);
        if (background) {
            EXPECT(dsim_server_start(S) == DSIM_OK);
            EXPECT(dsim_server_wait(S, t, 30) == DSIM_OK);
            EXPECT(dsim_server_stop(S) == DSIM_OK);
        } else {
            uint32_t a = 1, n = 1;
            while (a || n) EXPECT(dsim_server_round(S, &a, &n) == DSIM_OK);
            int d = -1;
            EXPECT(hipGetDevice(&d) == hipSuccess && d == 0);
        }
        EXPECT(stub::peak[0] == 0 && stub::peak[1] >= base + 5000 * 21 * 4);
    }
    EXPECT(dsim_server_destroy(S) == DSIM_OK && dsim_substrate_destroy(s) == DSIM_OK);
    hipSetDevice(0);
    EXPECT(stub::blocks.empty());
}

int main(int argc, char **argv) {
    const std::pair<const char *, void (*)()> cases[] = {
        {"pool_device", pool_device},
        {"pool_bound", pool_bound},
        {"handle_device", handle_device},
        {"row_plan", row_plan},
        {"error_flags", error_flags},
        {"label_on_a_full_device", label_on_a_full_device},
        {"label_without_lists", label_without_lists},
        {"server_budget", server_budget},
        {"state_on_a_full_device", state_on_a_full_device},
        {"phases_read_back", phases_read_back},
        {"trajectory_launches", trajectory_launches},
        {"waveforms_memory", waveforms_memory},
        {"failed_growth", failed_growth},
        {"trim", trim},
        {"server_device", server_device},
    };
    for (auto &c : cases) {
        if (argc > 1 && strcmp(argv[1], c.first)) continue;
        const int was = fails;
        c.second();
        printf("%s: %s\n", c.first, fails == was ? "ok" : "FAILED");
    }
    return fails != 0;
}
