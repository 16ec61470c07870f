// stub_device.h -- what the tests set and read of the stand-in device.
#pragma once

#include <atomic>
#include <cstdint>

struct StubState {
    std::atomic<uint32_t> build_us{0}, prep_us{0}, gather_us{0}, copy_us{0};  // how long work takes
    std::atomic<int> fail_gather{-1};        // the launch_gather call that fails
    std::atomic<bool> fail_host_malloc{false};
    std::atomic<int> graphs{0}, gathers{0}, copies{0}, copies_done{0}, order_variant{-1};
};
extern StubState stub;

// digest of the rows that the stand-in kernels write for a target
uint64_t stub_digest(uint32_t W, uint32_t K, uint32_t layout);
