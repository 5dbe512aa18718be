// Controls and records of the host-memory HIP runtime (stub_hip.cpp).
#pragma once

#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>

namespace stub {
constexpr int kDevices = 2;
struct Block {
    int device;
    size_t bytes;
};
extern std::mutex mu;
extern std::map<void *, Block> blocks;  // live allocations
extern size_t used[kDevices], peak[kDevices];
extern size_t total[kDevices];     // as hipDeviceTotalMem says
extern size_t capacity[kDevices];  // allocations past it fail
extern uint64_t n_malloc, n_free;
extern uint32_t flag_bits;         // error flags the next step launches raise
extern uint32_t n_label_rows, n_label_all, n_row_builds;
extern uint64_t row_bytes;         // of the row lists a call builds
extern bool keep_rows;             // new substrates hold row lists
}  // namespace stub
