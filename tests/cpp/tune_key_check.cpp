// Drives the keys and the entry check of lbm_amd/csrc/tune_cache.h (host code
// only) for tests/test_tune_keys.py:
//   tune_key_check grid DEVICE NX NY PRECISION ref|zg VARIANTS
//   tune_key_check batch DEVICE DOMAINS CELLS PRECISION ref|zg VARIANTS
//   tune_key_check answers ENTRY_VARIANT ENTRY_STEPS STEPS ALL_FROM VARIANTS   prints 0 / 1
#include <cstdio>
#include <cstdlib>
#include <string>

#include "../../lbm_amd/csrc/tune_cache.h"

int main(int argc, char **argv) {
    const std::string cmd = argc > 1 ? argv[1] : "";
    auto num = [&](int i) { return std::strtoull(argv[i], nullptr, 10); };
    if (cmd == "grid" && argc == 8) {
        std::printf("%s\n", tune_cache::grid_key(argv[2], (uint32_t)num(3), (uint32_t)num(4), argv[5],
                                                 std::string(argv[6]) == "ref", std::atoi(argv[7])).c_str());
    } else if (cmd == "batch" && argc == 8) {
        std::printf("%s\n", tune_cache::batch_key(argv[2], (uint32_t)num(3), num(4), argv[5],
                                                  std::string(argv[6]) == "ref", std::atoi(argv[7])).c_str());
    } else if (cmd == "answers" && argc == 7) {
        tune_cache::Entry e;
        e.variant = std::atoi(argv[2]);
        e.steps = (uint32_t)num(3);
        std::printf("%d\n", tune_cache::answers(e, (uint32_t)num(4), (uint32_t)num(5), std::atoi(argv[6])));
    } else {
        return 2;
    }
    return 0;
}
