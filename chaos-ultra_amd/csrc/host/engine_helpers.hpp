// engine_helpers.hpp — helpers shared by the escape-family launchers (engine.cpp, frame.cpp).
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "../../../include/chaosultra.h"
#include "common.hpp"

namespace cu {

constexpr uint32_t kMaxPersistentTiles = 1024;  // tile tables staged in LDS

cu_function function(cu_engine e, const std::string &name);
void launch(cu_engine e, cu_function f, dim3 grid, dim3 block, void **params, cu_stream s,
            bool timed, uint32_t lds = 0);
// Bytes of LDS, not used by the kernel, that let a CU hold `per_cu` blocks of it at once,
// for launches of `from` to `to` blocks per CU; 0 for others.
//
// Blocks go to the CUs before their lengths are known.  A launch of a few blocks per
// wave slot that fills every slot has most of its blocks placed at the start, and its
// time is that of the CU that drew the long ones; held to fewer at once, which issue
// nearly as much in FP64 (two waves per SIMD reach 93 % of eight's rate), more blocks go where
// others have ended.  Launches of fewer blocks have nothing to hold back, those of many even
// out by themselves, shallow ones (and FP32, whose waves need each other more: 5 to 20 %
// slower at any size) only lose.
//
// Grid kernel, FP64, all slots -> 4 blocks, us: 8 blocks per CU home 53 -> 57; 10 to 28 per
// CU 3 % over six views and two sample counts (16: home 70 -> 63, the set's edge 155 -> 143,
// width 1e-4 123 -> 110), two streams of 1024^2 home tiles 125 -> 103 us a pair; from 34 on
// 1 to 6 % slower, and at any size outside the set (maxIter 300, 10 to 15 %): from 10 to 28
// blocks per CU and from maxIter 500.  Direct deep frames, 8 -> 6 blocks: 8 per CU 115 -> 128
// at width 1e-4, 26 -> 29 at 2; 10 to 32 per CU up to 6 % faster (1920x1080 at 1e-4 183 -> 171),
// even at 2 and, from 13 on, at 1e-6.  Pass 1 of the pipeline, FP64: 0.99 of the time on average
// at 10 to 12 blocks per CU (the set's edge 0.92), 0.96 at 16, 1.01 from 20 on: from 10 to 18 and
// from maxIter 500; not in FP32 (1.05 to 1.2 of the time).
inline uint32_t spread_lds(uint64_t blocks, uint32_t from, uint32_t to, uint32_t per_cu) {
    constexpr uint32_t kLdsPerCu = 160u << 10, kGranule = 1280;
    const uint64_t cus = (uint64_t)std::max(1, compute_units());
    if (blocks < from * cus || blocks > to * cus) return 0;
    return kLdsPerCu / per_cu / kGranule * kGranule;
}
// An event that only marks a time inside a sequence: nothing waits for it, so it needs no
// system-scope fence (a full one is a packet of about 4 us; a 256x256 tile and its
// compose, two sequences: 28.0 -> 25.5 us).  The last event of a sequence, which callers wait for, is a
// full one.
hipEvent_t mark_event();
// 256-thread blocks of `f` that a CU holds at once, by its registers and LDS (asked once)
uint32_t resident_blocks(cu_function f);
const char *real_name(int precision);
bool fused_safe(const cu_tile_desc &t, int precision);
void validate_tile(const cu_tile_desc &t);
void validate_tune(const cu_tune &tn);
// the checks cu_deep_create runs on a deep-frame description (CU_ERR_ILLEGAL_ARGUMENT)
void validate_deep(const cu_deep_desc &d, int method);
bool pick_fused(int variant, const cu_tile_desc &t, int precision);
void *device_alloc(size_t bytes);  // hipMalloc, nullptr for 0 bytes; throws CuError
// fill `words` u32 at p with `value` by the fillU32 kernel (safe under graph capture)
void fill_u32(cu_engine e, cu_stream s, void *p, uint32_t value, uint64_t words);

// C = log2(log2(R^2)), the per-tile term of the smooth value
// n + 1 - (log2(log2(|z|^2)) - C) computed by the kernels.
inline double smooth_constant(double bailout_sq) { return std::log2(std::log2(bailout_sq)); }

}  // namespace cu
