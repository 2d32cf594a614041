// glitch_pick.hpp — which pixel of a deep frame without rebasing gets the next reference.
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstring>

namespace cu {

// f(x, y) for every pixel whose flag is set, row by row.  Eight flags at a time, since few
// are set: 1920x1080 frames of 4 to 8 references take 1.4 to 3.4 ms.  With a test and a
// branch for each flag they took 3.8 to 9.0 or 5.0 to 11.3 ms, by where in the library the
// loop stood.
template <class F>
void each_flagged(const unsigned char *flags, uint32_t W, uint32_t H, F &&f) {
    for (uint32_t y = 0; y < H; ++y) {
        const unsigned char *row = flags + (size_t)y * W;
        uint32_t x = 0;
        for (; W - x >= 8; x += 8) {
            uint64_t eight;
            std::memcpy(&eight, row + x, 8);
            if (eight == 0) continue;
            for (uint32_t k = 0; k < 8; ++k)
                if (row[x + k]) f(x + k, y);
        }
        for (; x < W; ++x)
            if (row[x]) f(x, y);
    }
}

// The glitched pixel nearest the centroid of all glitched pixels, the first of several.
inline bool pick_secondary(const unsigned char *flags, uint32_t W, uint32_t H, uint32_t &px,
                           uint32_t &py, uint32_t &count) {
    double sx = 0, sy = 0;
    uint32_t set = 0;
    each_flagged(flags, W, H, [&](uint32_t x, uint32_t y) {
        sx += x;
        sy += y;
        ++set;
    });
    count = set;
    if (set == 0) return false;
    const double cx = sx / set, cy = sy / set;
    double best = -1;
    each_flagged(flags, W, H, [&](uint32_t x, uint32_t y) {
        const double d2 = (x - cx) * (x - cx) + (y - cy) * (y - cy);
        if (best < 0 || d2 < best) {
            best = d2;
            px = x;
            py = y;
        }
    });
    return true;
}

}  // namespace cu
