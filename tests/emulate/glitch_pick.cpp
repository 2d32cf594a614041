// The pixel picked for a deep frame's next reference: the flags come as W x H bytes on
// standard input.
//
//   glitch_pick <W> <H>
//
// prints the count of set flags, and the pixel if there is one.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../chaos-ultra_amd/csrc/host/glitch_pick.hpp"

int main(int argc, char **argv) {
    if (argc != 3) return 2;
    const uint32_t W = (uint32_t)atoi(argv[1]), H = (uint32_t)atoi(argv[2]);
    std::vector<unsigned char> flags((size_t)W * H);
    if (std::fread(flags.data(), 1, flags.size(), stdin) != flags.size()) return 2;
    uint32_t px = 0, py = 0, count = 0;
    if (cu::pick_secondary(flags.data(), W, H, px, py, count))
        std::printf("%u %u %u\n", count, px, py);
    else
        std::printf("%u\n", count);
    return 0;
}
