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
// one (only the fovea and the new edges are sampled), and frames of at most 40 waves a CU
// in the two-group form.  FP64 at width 1e-4, 4 samples: 1080p zoom frames 420 -> 305 us,
// 720p 302 -> 208 us; whole frames 640x360 276 -> 189 us, 300x200 221 -> 162 us; the FP32
// home view 1024x576 209 -> 165 us.  Beyond, frames that fill the GPU with samples lose
// (a Julia dust 1280x720 at 5 samples 223 -> 230 us, a 4K frame 1521 -> 1818 us), as do
// single samples (1080p zoom frames 184 -> 207 us).
inline bool one_group_waves(int64_t width, int64_t height, float max_ss, bool reuse,
                            const PlaneRect &image, const PlaneRect &old) {
    if (!(max_ss >= 2.0f)) return false;
    return (width + 15) / 16 * ((height + 3) / 4) <= 40ll * std::max(1, compute_units()) ||
           (reuse && mostly_inside(image, old));
}

}  // namespace cu
