// Shapes of the Merkle stages (csrc/stage_plan.hpp): whatever the launch size,
// depth cap and tuned depth, a leaf stage stays inside the scratch the provers
// allocate for it and covers its items with whole waves.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "../../vortexstark_amd/csrc/stage_plan.hpp"

using namespace vx;

#define CHECK(x)                                                        \
    do {                                                                \
        if (!(x)) {                                                     \
            std::printf("failed: %s (line %d)\n", #x, __LINE__);        \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

static void check_shapes() {
    for (uint32_t l = 8; l <= 31; l++)
        for (uint32_t batch : {1u, 2u, 3u, 64u, 1000u})
            for (uint32_t cap : {2u, MERKLE_LOGC_MAX})
                for (bool nodes : {false, true}) {
                    const uint64_t n = 1ull << l;
                    const StageShape s = pick_stage(n, cap, batch, cap == MERKLE_LOGC_MAX, nodes);
                    CHECK(s.logc <= cap);
                    CHECK(s.logc == 0 || (n >> (7 + s.logc)) >= 2);
                    CHECK(s.keep >= 1 && s.keep <= 32 && (s.keep & (s.keep - 1)) == 0);
                    CHECK(!nodes || s.keep == 1);
                    // scratch: a leaf stage's nodes, and a node stage's (n / 128)
                    if (!nodes && n > 2048) CHECK((n >> (7 + s.logc)) * s.keep <= max_leaf_stage_nodes(n, 2048));
                    if (nodes && n > 2048) CHECK((n >> (7 + s.logc)) <= max_stage_nodes(n, 0));
                }
}

int main() {
    check_shapes();
    for (uint32_t c = 0; c <= MERKLE_LOGC_MAX; c++) {  // one tuned depth everywhere
        for (uint32_t i = 0; i < STAGE_PLAN_LOGS; i++) stage_plan_table()[i].store((uint8_t)(c + 1));
        check_shapes();
    }
    for (uint32_t i = 0; i < STAGE_PLAN_LOGS; i++) stage_plan_table()[i].store(0);
    // the lines of the default rule
    CHECK(pick_stage(1ull << 17, 5, 1, true, false).keep == 1 && pick_stage(1ull << 18, 5, 1, true, false).keep == 4);
    CHECK(pick_stage(1ull << 12, 5, 64, true, false).keep == 4);  // the launch counts, not the proof
    CHECK(pick_stage(1ull << 26, 5, 1, true, false).logc == 4 && pick_stage(1ull << 24, 5, 1, true, false).logc == 3);
    CHECK(pick_stage(1ull << 22, 2, 1, false, false).logc == 2);
    std::printf("stage shapes: ok\n");
    return 0;
}
