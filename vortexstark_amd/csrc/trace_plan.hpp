// Fibonacci traces: the steps a thread takes to its run of words, and the grid
// (host logic, shared with the kernel).
#pragma once
#include <stdint.h>

#include <algorithm>

namespace vx {

constexpr uint32_t FIB_RUN_LOG = 4, FIB_THREADS_LOG = 8;
// Workgroups along x: a launch has fewer than 2^32 threads along it, so longer
// traces (from 2^36 words on, 256 GiB) continue along z.
constexpr uint32_t FIB_GRID_LOG = 23;

// (F(2^b - 1), F(2^b)) mod 2^31 - 1 for every bit of a 64-bit word index.
struct FibSteps {
    uint32_t f[64][2] = {};
    constexpr FibSteps() {
        constexpr uint64_t M = 0x7FFFFFFFu;
        uint64_t x = 0, y = 1;
        for (int b = 0; b < 64; b++) {
            f[b][0] = (uint32_t)x;
            f[b][1] = (uint32_t)y;
            const uint64_t x2 = (x * x % M + y * y % M) % M, y2 = y * ((2 * x + y) % M) % M;
            x = x2;
            y = y2;
        }
    }
};

struct FibGrid {
    uint32_t x, z;
};
constexpr FibGrid fib_grid(uint64_t n) {
    const uint64_t blocks = ((n - 1) >> (FIB_RUN_LOG + FIB_THREADS_LOG)) + 1, row = 1ull << FIB_GRID_LOG;
    return {(uint32_t)std::min(blocks, row), (uint32_t)(((blocks - 1) >> FIB_GRID_LOG) + 1)};
}

}  // namespace vx
