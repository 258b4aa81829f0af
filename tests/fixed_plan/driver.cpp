// Plans of the one-group GEMMs (fixed_plan.h): reads lines "T N pair cb stages
// max_splits blocks", prints "m_tiles tile_rows n_tiles ksplit most_rows cols".
#include <cstdio>

#include "fixed_plan.h"

int main() {
    int T, N, pair, cb, stages, most, blocks;
    while (std::scanf("%d %d %d %d %d %d %d", &T, &N, &pair, &cb, &stages, &most, &blocks) == 7) {
        const hf::FixedPlan p = hf::plan_fixed_gemm(T, N, pair != 0, cb, stages, most, blocks);
        std::printf("%d %d %d %d %d %d\n", p.m_tiles, p.tile_rows, p.n_tiles, p.ksplit, hf::fixed_tile_rows(cb),
                    hf::fixed_tile_cols(cb, pair != 0));
    }
    return 0;
}
