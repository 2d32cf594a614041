// The host's rules by which launches choose their form, on 256 compute units, without a GPU.
//
//   launch_rules forms <width> <height> <samples> <max_iter> <reuse 0|1> <overlap 0..1>
//
// prints the vote groups a wave of the render kernels (1 or 2); `overlap` is the part of the
// image's width that an earlier one covers.
//
//   launch_rules lds <blocks> <from> <to> <per_cu>
//
// prints the bytes of LDS that a launch asks for to hold a CU to per_cu blocks.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../chaos-ultra_amd/csrc/host/engine_helpers.hpp"
#include "../../chaos-ultra_amd/csrc/host/render_form.hpp"

namespace cu {
int compute_units() { return 256; }
}  // namespace cu

int main(int argc, char **argv) {
    if (argc == 8 && std::strcmp(argv[1], "forms") == 0) {
        const cu::PlaneRect image{0, 0, 1, 1}, old{0, 0, atof(argv[7]), 1};
        std::printf("%d\n", cu::one_group_waves(atoll(argv[2]), atoll(argv[3]), (float)atof(argv[4]),
                                                (uint32_t)strtoul(argv[5], nullptr, 10),
                                                atoi(argv[6]) != 0, image, old)
                                ? 1
                                : 2);
        return 0;
    }
    if (argc == 6 && std::strcmp(argv[1], "lds") == 0) {
        std::printf("%u\n", cu::spread_lds(strtoull(argv[2], nullptr, 10), (uint32_t)atoi(argv[3]),
                                           (uint32_t)atoi(argv[4]), (uint32_t)atoi(argv[5])));
        return 0;
    }
    return 2;
}
