// Points the NTT table kernel reads (csrc/table_plan.hpp): for every transform
// size and layer the table of step^(2^b) holds all of them.
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "../../vortexstark_amd/csrc/table_plan.hpp"

using namespace vx;

#define CHECK(x)                                                        \
    do {                                                                \
        if (!(x)) {                                                     \
            std::printf("failed: %s (line %d)\n", #x, __LINE__);        \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

// highest entry a layer of `len` words reads from its shift on: the step of the
// run itself, a whole workgroup's bits, and those of the last workgroup's number
static uint32_t top_entry(uint32_t shift, uint64_t len) {
    const uint64_t per_block = 1ull << (TABLE_RUN_LOG + TABLE_THREADS_LOG);
    uint32_t top = shift + TABLE_RUN_LOG + TABLE_THREADS_LOG - 1, b = shift + TABLE_RUN_LOG + TABLE_THREADS_LOG;
    for (uint64_t blk = (len - 1) / per_block; blk; blk >>= 1, b++) top = std::max(top, b);
    return top;
}

int main() {
    uint32_t top = 0;
    for (uint32_t log_n = 1; log_n <= NTT_LOG_MAX; log_n++) {
        const uint64_t n = 1ull << log_n;
        for (uint32_t l = 0; l + 1 < log_n; l++) top = std::max(top, top_entry(line_layer_shift(l), n >> (l + 1)));
        top = std::max(top, top_entry(0, n / 2));
        CHECK(top < NTT_TABLE_SQUARES);
    }
    CHECK(top == 70);  // the 2^31-point domain's last line layer
    std::printf("table points: ok\n");
    return 0;
}
