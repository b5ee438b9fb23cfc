// Sizes and matcher choices of the plans, for a build whose host code carries
// AddressSanitizer; no device is needed and none is used.
//
//   plan_sizes                      sizes every allowed block, step, range and group
//   plan_sizes S R G W H N ...      the matcher kind chosen for each six numbers: block 8,
//                                   step S, range R, group G, W x H planes, N references
//   plan_sizes tiles G S R N ...    the group filters' tile for each four numbers: group G,
//                                   step S, range R, N references ("0 0": the atomic path)
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../vapoursynth-nssfactory_amd/csrc/instance.hpp"

using namespace nsship;

int main(int argc, char** argv) {
    if (argc > 1 && !std::strcmp(argv[1], "tiles")) {
        for (int i = 2; i + 3 < argc; i += 4) {
            const TileShape t = gram_tile_shape(8, std::atoi(argv[i]), std::atoi(argv[i + 1]), std::atoi(argv[i + 2]),
                                                std::atoll(argv[i + 3]));
            std::printf("%d %d\n", t.tw, t.th);
        }
        return 0;
    }
    if (argc > 1) {
        for (int i = 1; i + 5 < argc; i += 6) {
            int v[6];
            for (int k = 0; k < 6; ++k) v[k] = std::atoi(argv[i + k]);
            size_t lds = 0;
            std::printf("%d\n", choose_match_kind(8, v[0], v[1], v[2], v[3], v[4], v[5], &lds));
        }
        return 0;
    }
    long long shapes = 0, fits = 0, failures = 0;
    for (int block : {1, 2, 4, 8, 12, 16, 32})
        for (int step = 1; step <= block; ++step)
            for (int range = 1; range <= 64; ++range)
                for (int group : {1, 2, 4, 8, 16, 32, 64}) {
                    const size_t lds = match_mfma_lds_bytes(step, range, group);
                    const bool f = match_mfma_fits(block, group, step, range, 640, 480);
                    ++shapes;
                    fits += f;
                    // what is said to fit does, and the sizes of block 8 all do
                    failures += f && lds > 160 * 1024;
                    failures += block == 8 && group <= 32 && !f;
                    size_t chosen = 0;
                    const int kind = choose_match_kind(block, step, range, group, 640, 480, 1 << 20, &chosen);
                    failures += kind == 3 && (!f || chosen != lds);
                }
    std::printf("%lld shapes, %lld for the MFMA matcher; %lld failure(s)\n", shapes, fits, failures);
    return failures ? 1 : 0;
}
