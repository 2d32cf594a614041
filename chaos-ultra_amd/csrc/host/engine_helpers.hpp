// engine_helpers.hpp — helpers shared by the escape-family launchers (engine.cpp, frame.cpp).
#pragma once
#include <hip/hip_runtime_api.h>

#include <cmath>
#include <string>

#include "../../../include/chaosultra.h"

namespace cu {

constexpr uint32_t kMaxPersistentTiles = 1024;  // tile tables staged in LDS

cu_function function(cu_engine e, const std::string &name);
void launch(cu_engine e, cu_function f, dim3 grid, dim3 block, void **params, cu_stream s,
            bool timed, uint32_t lds = 0);
// Bytes of LDS, not used by the kernel, that let a CU hold `per_cu` blocks of it at once.
//
// Blocks go to the CUs before their lengths are known.  A launch of a few blocks per
// wave slot that fills every slot has most of its blocks placed at the start, and its
// time is that of the CU that drew the long ones; held to fewer at once, which issue
// nearly as much (two waves per SIMD reach 93 % of eight's rate), more blocks go where
// others have ended.  Launches of many blocks per slot even out by themselves and lose
// a few per cent.  Measured, grid kernel / pass 1, us, all slots -> 4 blocks per CU:
// 1024^2, 1 spp, FP64 (16 blocks per CU) whole set 77 -> 68 / 78 -> 59, the set's edge
// 181 -> 153 / 167 -> 141; 2048^2 (64 per CU) at width 1e-4 349 -> 351 / 186 -> 173 (169
// with 5); 4096^2, 4 spp (1024 per CU) 3535 -> 4042 / 2376 -> 2498.
uint32_t lds_for(uint32_t per_cu);
bool few_blocks(dim3 grid);  // at most 32 per CU
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
