// hip_runtime.h — as much of the device language as kernels/escape_core.hpp and
// kernels/perturb_core.hpp use, for a host compiler: one wave of 64 lanes whose operations
// across lanes are those of simt.hpp.  Found before the real header by -I.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../simt.hpp"

#define __device__
#define __global__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)

using std::max;
using std::min;
struct double2 {
    double x, y;
};

#define threadIdx (simt::Index{(unsigned)simt::lane(), 0})
#define blockIdx (simt::Index{0, 0})
#define blockDim (simt::Index{64, 1})
#define gridDim (simt::Index{1, 1})

#define __ballot(p) simt::ballot(p)
#define __lane_id() ((unsigned)simt::lane())
#define __syncthreads() simt::barrier()
#define __builtin_amdgcn_readfirstlane(v) ((unsigned)simt::read_lane(v, 0))
#define __builtin_amdgcn_readlane(v, l) ((unsigned)simt::read_lane(v, l))
#define __builtin_amdgcn_inverse_ballot_w64(mask) (((mask) >> simt::lane() & 1) != 0)
#define __builtin_amdgcn_frexp_exp(v) simt::frexp_exp(v)
#define __builtin_amdgcn_frexp_mant(v) simt::frexp_mant(v)
#define __builtin_amdgcn_rcp(v) (1.0 / (v))
inline unsigned long long atomicAdd(unsigned long long *p, unsigned long long v) {
    const unsigned long long old = *p;
    *p += v;
    return old;
}
// the one instruction that the headers write by name (cu::lanes)
#define asm(...) n = (uint)__builtin_popcountll(mask)
