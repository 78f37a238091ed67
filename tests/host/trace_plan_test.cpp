// Fibonacci trace steps and grid (csrc/trace_plan.hpp): every word index of a
// trace that fits a GPU has its step, and the grid covers it within HIP's limit
// of 2^32 threads along x.
#include <cstdio>
#include <cstdlib>

#include "../../vortexstark_amd/csrc/trace_plan.hpp"

using namespace vx;

#define CHECK(x)                                                        \
    do {                                                                \
        if (!(x)) {                                                     \
            std::printf("failed: %s (line %d)\n", #x, __LINE__);        \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

int main() {
    constexpr uint64_t M = 0x7FFFFFFFu;
    static constexpr FibSteps steps;
    constexpr uint32_t n_steps = sizeof(steps.f) / sizeof(steps.f[0]);
    // (F(2^b - 1), F(2^b)) by adding for small b, then F(i + j) = F(i - 1) F(j) + F(i) F(j + 1)
    uint64_t f0 = 0, f1 = 1;  // F(0), F(1)
    uint32_t b = 0;
    for (uint64_t i = 1; i <= 1u << 16; i++) {
        if (i == 1ull << b) {
            CHECK(steps.f[b][0] == f0 && steps.f[b][1] == f1);
            b++;
        }
        const uint64_t f2 = (f0 + f1) % M;
        f0 = f1;
        f1 = f2;
    }
    for (; b < n_steps; b++) {
        const uint64_t x = steps.f[b - 1][0], y = steps.f[b - 1][1], z = (x + y) % M;  // F(m-1), F(m), F(m+1)
        CHECK(steps.f[b][0] == (x * x % M + y * y % M) % M);
        CHECK(steps.f[b][1] == (x * y % M + y * z % M) % M);
    }
    for (uint32_t log_n = 0; log_n <= 40; log_n++) {
        const uint64_t n = 1ull << log_n;
        const FibGrid g = fib_grid(n);
        CHECK(log_n < n_steps);  // bits of the last word's index
        CHECK((uint64_t)g.x << FIB_THREADS_LOG < 1ull << 32);
        CHECK(g.z == 1 || g.x == 1u << FIB_GRID_LOG);
        CHECK(((((uint64_t)(g.z - 1) << FIB_GRID_LOG) + g.x) << (FIB_RUN_LOG + FIB_THREADS_LOG)) >= n);
        CHECK(((((uint64_t)(g.z - 1) << FIB_GRID_LOG) + g.x - 1) << (FIB_RUN_LOG + FIB_THREADS_LOG)) < n);
    }
    std::printf("trace plan: ok\n");
    return 0;
}
