// The splits of sizes without a plan, general and blowup-4 evaluations: every size is covered by passes that
// have a kernel, and only the top one replicates.
#include <stdio.h>
#include <stdlib.h>

#include "../../vortexstark_amd/csrc/ntt_plan.hpp"

using namespace vx;
#define CHECK(c)                                     \
    if (!(c)) {                                      \
        printf("line %d, k = %u: %s\n", __LINE__, k, #c); \
        return 1;                                    \
    }

int main() {
    for (uint32_t k = 0; k <= 31; k++) {
        const std::vector<Pass> ps = default_lde_plan(k);
        CHECK(plan_valid(k, ps, true));
        for (size_t i = 0; i < ps.size(); i++) CHECK(ps[i].r == (k > NTT_LOW && i + 1 == ps.size()));
        for (const Pass& p : ps) CHECK(pass_rows(p) + p.c <= NTT_LOW_MAX);
        CHECK(ps.size() == (k == 0 ? 0 : k <= 12 ? 1 : k <= 24 ? 2 : 3));
        if (k > 12) CHECK(ps[0].m == std::min(12u, k - 3));
        const std::vector<Pass> us = untuned_plan(k);
        CHECK(plan_valid(k, us));
        if (k <= 23) CHECK(us.size() == (k == 0 ? 0 : k <= 12 ? 1 : 2));
        for (const Pass& p : us) CHECK(p.m + p.c <= NTT_LOW_MAX);
    }
    printf("lde plans: ok\n");
    return 0;
}
