// Checks lbm_amd/csrc/tile_plan.h (host code only) for tests/test_tile_plan.py:
// every plan of a call of n steps has launches of allowed lengths that add up to n.
//   tile_plan_check NX NY N [N ...]    ("ok" and the f32 / binary16 / FP64 launches, or what is wrong)
#include <cstdio>
#include <cstdlib>

#include "../../lbm_amd/csrc/tile_plan.h"

static bool adds_up(uint32_t n, uint32_t launches, uint32_t least) {
    const uint32_t low = n / launches, more = n % launches;
    return low >= least && low + (more != 0) <= (uint32_t)kTileMaxSteps;
}

int main(int argc, char **argv) {
    if (argc < 4) return 2;
    const int X = std::atoi(argv[1]), Y = std::atoi(argv[2]);
    for (int i = 3; i < argc; ++i) {
        const uint32_t n = (uint32_t)std::strtoull(argv[i], nullptr, 10);
        uint32_t found[2] = {0, 0};
        if (n >= 2)
            for (int precision : {LBM_PRECISION_F32, LBM_PRECISION_F16S})
                for (int first : {0, 1})
                    for (int last = first; last < 2; ++last)
                        for (bool even : {false, true}) {
                            const TilePlan p = tile_plan(precision, first, last, n, even, [&](int s, int steps) {
                                const TileShape &sh = tile_shape(precision, s);
                                return (int64_t)tile_nbx(X, steps) * tile_nby(Y, sh.waves * sh.m, steps);
                            });
                            // (two or three steps in an even number of launches: none)
                            const bool ok = p.launches ? adds_up(n, p.launches, 2) && p.shape >= first && p.shape <= last
                                                       : n <= 3 && even;
                            if (!ok || (even && p.launches % 2)) {
                                std::printf("n %u precision %d shapes %d..%d even %d: shape %d, %u launches\n", n,
                                            precision, first, last, even, p.shape, p.launches);
                                return 1;
                            }
                            found[precision != LBM_PRECISION_F32] = p.launches;
                        }
        const TilePlan q = plan64(X, Y, n);
        if (!q.launches || q.launches % 2 == 0 || !adds_up(n, q.launches, 1)) {
            std::printf("n %u FP64: shape %d, %u launches\n", n, q.shape, q.launches);
            return 1;
        }
        std::printf("%u: %u %u %u\n", n, found[0], found[1], q.launches);
    }
    std::printf("ok\n");
    return 0;
}
