// render_form.hpp — the forms in which the fractal modules' render kernels are launched
// by the renderer layer and the serving loop (kernels/render_generic.hip): blocks that
// cover 32 x 4 pixels, with two vote groups a wave (*Strip, 32 x 4 threads) or one
// (*Group, 32 x 8 threads).  Pixels, vote groups and results are the same.
#pragma once

#include <algorithm>
#include <cstdint>

#include "common.hpp"

namespace cu {

constexpr int kStripRows = 4;   // rows of pixels of a block in either form
constexpr int kGroupTRows = 8;  // thread rows of a *Group block

// Thread rows of a compose block, on the reference's grid of ceil(W/32) x ceil(H/32).
// The compose of a module with the forms above strides over its block's 32 rows: a
// 1024-thread block only starts on a CU with 16 free wave slots, which other sessions'
// renders leave late (beside them compose took 207 us a frame on average, 5 us alone).
// Any other module's is the reference's kernel, one thread a pixel.
inline int compose_rows(bool forms) { return forms ? 8 : 32; }

struct PlaneRect {
    double lbx, lby, rtx, rty;
};

// Whether at least half of `image` lies in `old`.
inline bool mostly_inside(const PlaneRect &image, const PlaneRect &old) {
    const double w = std::min(image.rtx, old.rtx) - std::max(image.lbx, old.lbx);
    const double h = std::min(image.rty, old.rty) - std::max(image.lby, old.lby);
    return w > 0 && h > 0 && w * h >= 0.5 * (image.rtx - image.lbx) * (image.rty - image.lby);
}

// One vote group a wave halves what the waves with the most work do and doubles the
// number of waves, with half of their lanes idle where a pixel takes one sample.  So it
// is for launches that wait for their longest waves: frames that reuse most of an earlier
// one (only the fovea and the new edges are sampled), and frames of at most 60 waves a CU
// in the two-group form.  What it gives there depends on the image, at most half of the
// longest wave's chain of max_iter steps a sample; what it costs, on its size, however
// shallow the image (1920x1080 zoom frames 59 -> 81 us, 4K 154 -> 240; a Julia dust of
// 800x480 143 -> 155).  So max_iter has to be in proportion to the pixels.  Two groups / one,
// us: FP64 at width 1e-4, maxIter 5000, 4 samples, zoom frames 1080p 368 / 283, 720p 303 /
// 205, whole frames 720p 318 / 225, 800x480 301 / 194; below the line Julia zoom frames
// of maxIter 900, 720p 46 / 54, whole ones 800x480 48 / 57, and FP64 4K zooms 550 / 441 the
// other way.  Over 780 frames (64x48 to 4K, 10 views, 1 to 8 samples) zooms are 5 % faster than
// with this form always, whole frames even, and none is more than 16 % slower than with two.
inline bool one_group_waves(int64_t width, int64_t height, float max_ss, uint32_t max_iter,
                            bool reuse, const PlaneRect &image, const PlaneRect &old) {
    if (!(max_ss >= 2.0f)) return false;  // single samples: 184 -> 207 us
    const double pixels = (double)width * (double)height;
    if (reuse && mostly_inside(image, old)) return pixels <= 800.0 * max_iter;
    return (width + 15) / 16 * ((height + 3) / 4) <= 60ll * std::max(1, compute_units()) &&
           pixels <= 400.0 * max_iter;
}

}  // namespace cu
