// escape_family.hip — planar escape-time kernels of the quadratic family for gfx950.
//
// These serve the throughput forms that have no counterpart in the reference:
// tiles of pixel-centre or seeded-jitter samples with any bailout radius and a
// smooth value, a persistent launch over many tiles of uneven depth, and a
// palette compose of the smooth plane.  Mandelbrot and Julia tiles mix freely
// (per-tile `kind`); the orbit rounding is the reference's (escape_core.hpp).
//
// Kernels (all extern "C", bound by name from escape_family.hsaco):
//   escapeTile{Double,Float}{Exact,Fused}      thread per pixel, one tile
//   escapeTilesPersistent{Double,Float}{Exact,Fused}
//                                              lane-refill work queue, many tiles
//   composeSmooth                              smooth plane -> RGBA8, LDS palette
//   fillU32                                    device fill (graph-capture safe)
#include "cu_types.hpp"
#include "escape_core.hpp"

#pragma clang fp contract(off)

namespace {

constexpr uint kMaxLdsTiles = 1024;
constexpr uint kPaletteLds = 4096;

// Start sample `sample_id` = (py * width + px) * spp + s of tile t (pixel (px, py)):
// z0 and c for the tile's kind.
template <class Real>
__device__ __forceinline__ void begin_sample_of(const cu_tile_desc &t, uint px, uint py,
                                                uint64_t sample_id, Real &x, Real &y, Real &cx,
                                                Real &cy) {
    double dx, dy;
    cu::sample_offset_of(t, sample_id, dx, dy);
    Real X, Y;
    cu::tile_point<Real>(t, px, py, dx, dy, X, Y);
    if (t.kind == CU_FRACTAL_JULIA) {
        x = X;
        y = Y;
        cx = (Real)t.julia_cx;
        cy = (Real)t.julia_cy;
    } else {
        x = 0;
        y = 0;
        cx = X;
        cy = Y;
    }
}

// Start sample s of pixel (px, py) of tile t: z0 and c for the tile's kind.
template <class Real>
__device__ __forceinline__ void begin_sample(const cu_tile_desc &t, uint px, uint py, uint s,
                                             Real &x, Real &y, Real &cx, Real &cy) {
    begin_sample_of<Real>(t, px, py, ((uint64_t)py * t.width + px) * t.spp + s, x, y, cx, cy);
}

__device__ __forceinline__ bool tile_blocks_valid(const cu_tile_desc &t) {
    return cu::blocks_valid(t.bailout_sq, t.kind == CU_FRACTAL_JULIA, t.julia_cx, t.julia_cy);
}

// ---------------------------------------------------------------------------
// thread per pixel over one tile (any spp; samples in sequence)
// ---------------------------------------------------------------------------
template <class Real, int K, bool kFused>
__device__ void escape_tile(const cu_tile_desc &t, double smooth_c, uint *counts, double *smooth,
                            unsigned long long *iters) {
    const uint px = cu::skewed_block_x() * blockDim.x + threadIdx.x;
    const uint py = blockIdx.y * blockDim.y + threadIdx.y;
    uint64_t executed = 0;
    if (px < t.width && py < t.height) {
        const bool blocks = tile_blocks_valid(t);
        const Real bsq = (Real)t.bailout_sq;
        const bool julia = t.kind == CU_FRACTAL_JULIA;
        uint count_sum = 0;
        double smooth_sum = 0;
        for (uint s = 0; s < t.spp; ++s) {
            Real x, y, cx, cy;
            begin_sample<Real>(t, px, py, s, x, y, cx, cy);
            const cu::Orbit<Real> o =
                cu::escape_orbit<Real, K, kFused>(x, y, cx, cy, t.max_iter, bsq, blocks);
            executed += o.n;
            count_sum += o.escaped ? o.n : (julia ? t.max_iter : 0u);
            smooth_sum += o.escaped ? cu::smooth_value(o.n, (double)o.mag2, smooth_c) : 0.0;
        }
        const uint64_t o = t.out_offset + (uint64_t)py * t.out_pitch + px;
        counts[o] = count_sum / t.spp;
        if (smooth) smooth[o] = smooth_sum / (double)t.spp;
    }
    cu::add_iterations(iters, executed);
}

// ---------------------------------------------------------------------------
// one sample per lane over one tile (spp a power of two <= 64)
// ---------------------------------------------------------------------------
// A wave covers 64/spp pixels as a near-square block (spp 4: 4x4 pixels x 4
// samples), so neighbouring lanes iterate neighbouring points and the wave's
// longest orbit stays close to its mean; per-sample setup and the smooth value
// run on all lanes at once.  The spp lanes of a pixel sum their counts and
// smooth values in sample order (lane s==0 adds lanes 1..spp-1 in turn), the
// same order as a sequential loop.  Block: 256 threads = 4 waves in 2x2.
//
// Bound by the waves with the longest orbits and how they share out over the SIMDs
// (VALU issue 0.39).  Whole set, 1024^2, maxIter 1000, FP64, kernel alone 92 -> 71 us
// with the cycle test (0.41 of the loop's steps left, 0.6 of its longest orbits per
// wave) and 62 us with run_blocks' loop and 4 blocks per CU (spread_lds); 777x613 FP32
// Julia set, 3 spp (escape_tile) with compose 74-95 -> 39-50 us.  Tried and not kept: a
// wave taking 2 to 4 blocks as one pool whose lanes refill (101 us: a wave then runs
// several long orbits one after another).
// shape 0 is the near-square block; each further shape is twice as wide (capped
// at one row of 64/spp pixels).
__device__ __forceinline__ void wave_pixel_block(uint spp, uint &bw, uint &bh, uint shape = 0) {
    const uint ppw = 64u / spp;
    const uint lg = 31u - __clz(ppw);
    bw = min(ppw, 1u << (((lg + 1u) >> 1) + shape));
    bh = ppw / bw;
}

template <class Real, int K, bool kFused>
__device__ void escape_tile_samples(const cu_tile_desc &t, double smooth_c, uint *counts,
                                    double *smooth, unsigned long long *iters) {
    const uint spp = t.spp;
    const uint lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint bw, bh;
    wave_pixel_block(spp, bw, bh);
    const uint pix = lane / spp, s = lane % spp;
    const uint px = (cu::skewed_block_x() * 2u + (wave & 1u)) * bw + pix % bw;
    const uint py = (blockIdx.y * 2u + (wave >> 1)) * bh + pix / bw;
    const bool inside = px < t.width && py < t.height;
    const bool julia = t.kind == CU_FRACTAL_JULIA;
    uint count = 0;
    double sm = 0;
    uint64_t executed = 0;
    if (inside) {
        Real x, y, cx, cy;
        begin_sample<Real>(t, px, py, s, x, y, cx, cy);
        const cu::Orbit<Real> o = cu::escape_orbit<Real, K, kFused>(
            x, y, cx, cy, t.max_iter, (Real)t.bailout_sq, tile_blocks_valid(t));
        executed = o.n;
        count = o.escaped ? o.n : (julia ? t.max_iter : 0u);
        sm = o.escaped ? cu::smooth_value(o.n, (double)o.mag2, smooth_c) : 0.0;
    }
    uint count_sum = count;
    double smooth_sum = sm;
    for (uint j = 1; j < spp; ++j) {  // wave-uniform: every lane takes part in the shuffles
        const uint cj = __shfl(count, (int)(lane + j), 64);
        const double sj = __shfl(sm, (int)(lane + j), 64);
        count_sum += cj;
        smooth_sum += sj;
    }
    if (inside && s == 0) {
        const uint64_t o = t.out_offset + (uint64_t)py * t.out_pitch + px;
        counts[o] = count_sum / spp;
        if (smooth) smooth[o] = smooth_sum / (double)spp;
    }
    cu::add_iterations(iters, executed);
}

// ---------------------------------------------------------------------------
// persistent lane-refill launch over many tiles
// ---------------------------------------------------------------------------
// Every wave keeps 64 independent samples in flight.  Lanes run unchecked blocks
// of K steps in lock step (cu::run_blocks); a lane whose block fails its end test,
// whose remaining budget is below K or whose orbit has become a cycle of states
// becomes pending.  Once `refill` lanes are pending or idle, the pending lanes locate
// the exact escape step in the half of their last block that holds it
// (cu::locate_escape), finish their sample, start the next sample of the same
// pixel or write the pixel, and idle lanes take new pixels from a wave-private
// chunk of the global pixel queue (one atomic per at most `chunk` pixels).  Pixels of
// one tile are numbered row-major from the tile's work_offset.  There is no
// barrier after the tile table is staged, and every wave leaves once the queue
// is exhausted and its lanes are idle.
//
// Bound by VALU issue, then by the longest orbits at the end (a lone wave takes about
// 17 ns a step, so 65536 of them 1.1 ms).  Batches of 32 and 24 uneven tiles, FP64,
// tune 32/32/256/16: 7.7 -> 2.8 and 10.0 -> 2.2 ms (1.8e10 and 2.3e10 loop iterations)
// with the cycle test, scalar lane masks and cursor and one resident set of waves (98
// VGPRs, four blocks per CU); 32 tiles in FP32
// 9.4 -> 1.8 ms.  Giving waves with old orbits issue priority (s_setprio) made no
// batch faster and frames' tails up to 8 % slower.
// A grab of the queue is of at least this many steps, at its tile's max_iter (as far as
// `chunk` allows).  The counter takes an atomic every 13 ns, so 4096 waves must not come more
// often than every 50 us, and pixels seldom run to max_iter.  With 64-pixel grabs at every
// depth and with these: 16 tiles of 256^2, maxIter 50, 212 / 41 us, one of 1024^2, maxIter
// 1000, 242 / 118, the headline frame's view there, maxIter 5000, 307 / 200; the other way, 1000
// tiles of 8 to 40 pixels a side, maxIter 256 to 1024, 260 / 346.  Four times as many steps
// leave waves with late deep grabs: 256 tiles of 50 to 200 pixels a side, maxIter 256 to
// 65536, FP32, 5.0 -> 7.2 ms; half and twice as many are even.
constexpr uint kGrabSteps = 1024u << 10;

// From this max_iter on, batches that the waves' first grabs cover are put in order too (a
// deep wave beside another on its SIMD takes twice as long; the first of the order go to
// SIMDs of their own) and spread over half of the waves: 32 tiles of 8 to 97 pixels a side
// 0.82 -> 0.69 ms.  Shallower ones are spread over all of them (maxIter up to 1024, 400
// tiles of 8 to 40 pixels a side 211 -> 169 us) and not worth the order's time.
constexpr uint kOrderDepth = 4096;

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Classes of max_iter, the deepest first: two to an octave, a lane of a wave each.
__device__ __forceinline__ uint depth_class(uint depth) {
    depth = max(depth, 1u);
    const uint octave = 31u - __clz(depth);
    return 63u - (2u * octave + (octave ? (depth >> (octave - 1)) & 1u : 0u));
}

// The queue's order of n tiles, by a block's four waves: from the deepest class of max_iter
// down, so that the longest orbits do not start last, in a class as they come (24 batches
// of 32 tiles of very different depth, 3.9 -> 3.2 ms on average, 0.6 to 1.14 of the time each:
// which wave is the last changes with any order; 512 tiles 5.0 -> 3.1, 1024 8.1 -> 4.7).  word[k] is tile k's size and depth; order[p] becomes the
// tile at place p, offset[p] the sizes of the places before it; returns the sum of all
// sizes times depths.  Each wave counts, places and adds up a quarter of the tiles.  Every
// block of the launch does it, so what counts is instructions: 1024 tiles take about 10 us,
// where counting each tile's place out against all others took 1150 us (256 tiles 76 us).
struct OrderLds {
    uint next[4][64];  // per wave and class: tiles, then the next one's place
    uint64_t sizes[4];
    float steps[4];
};
__device__ float order_by_depth(const uint64_t *word, uint n, OrderLds &lds, ushort *order,
                                uint64_t *offset) {
    const uint lane = cu::lane_id(), wave = threadIdx.x >> 6;
    const uint64_t lanes_below = (1ull << lane) - 1ull;
    const uint each = (n + 255) / 256 * 64;
    const uint lo = min(wave * each, n), hi = min(lo + each, n);
    lds.next[wave][lane] = 0;
    wave_fence();
    for (uint k = lo + lane; k < hi; k += 64)
        atomicAdd(&lds.next[wave][depth_class((uint)(word[k] >> 32))], 1u);
    __syncthreads();
    uint count = 0, place = 0;  // of the class `lane`, in all waves and in those before
#pragma unroll
    for (uint w = 0; w < 4; ++w) {
        const uint here = lds.next[w][lane];
        count += here;
        if (w < wave) place += here;
    }
    uint upto = count;
#pragma unroll
    for (uint d = 1; d < 64; d *= 2) {
        const uint below = __shfl_up(upto, d, 64);
        if (lane >= d) upto += below;
    }
    __syncthreads();
    lds.next[wave][lane] = upto - count + place;
    wave_fence();
    for (uint from = lo; from < hi; from += 64) {
        const bool have = from + lane < hi;
        const uint c = have ? depth_class((uint)(word[from + lane] >> 32)) : 0u;
        uint64_t alike = cu::ballot(have);  // the lanes with a tile of this lane's class
#pragma unroll
        for (uint bit = 0; bit < 6; ++bit) {
            const uint64_t set = cu::ballot((c >> bit) & 1u);
            alike &= (c >> bit) & 1u ? set : ~set;
        }
        const uint at = lds.next[wave][c] + (uint)__popcll(alike & lanes_below);
        wave_fence();
        if (have) {
            order[at] = (ushort)(from + lane);
            if ((alike >> lane) == 1) lds.next[wave][c] = at + 1;  // its last lane
        }
        wave_fence();
    }
    __syncthreads();
    uint64_t base = 0;
    float steps = 0;
    for (uint from = lo; from < hi; from += 64) {
        const bool have = from + lane < hi;
        const uint64_t w = have ? word[order[from + lane]] : 0u;
        const uint64_t size = (uint)w;
        steps += (float)size * (float)(uint)(w >> 32);
        unsigned long long through = size;
#pragma unroll
        for (uint d = 1; d < 64; d *= 2) {
            const unsigned long long below = __shfl_up(through, d, 64);
            if (lane >= d) through += below;
        }
        if (have) offset[from + lane] = base + through - size;
        base += __shfl(through, 63, 64);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) steps += __shfl_xor(steps, off, 64);
    if (lane == 0) {
        lds.sizes[wave] = base;
        lds.steps[wave] = steps;
    }
    __syncthreads();
    base = 0;
    for (uint w = 0; w < wave; ++w) base += lds.sizes[w];
    for (uint k = lo + lane; k < hi; k += 64) offset[k] += base;
    return lds.steps[0] + lds.steps[1] + lds.steps[2] + lds.steps[3];
}

template <class Real, int K, bool kFused>
__device__ void escape_tiles_persistent(const cu_tile_desc *__restrict__ tiles, uint n_tiles,
                                        uint64_t total, uint *counts, double *smooth,
                                        unsigned long long *iters, unsigned long long *queue,
                                        uint chunk, uint refill) {
    __shared__ uint64_t lds_offset[kMaxLdsTiles];
    __shared__ uint64_t lds_word[kMaxLdsTiles];  // smooth constant; size and depth for order_by_depth
    __shared__ ushort lds_order[kMaxLdsTiles];
    __shared__ OrderLds lds_ordering;
    __shared__ uint lds_deepest;
    if (threadIdx.x == 0) lds_deepest = 0;
    __syncthreads();
    uint deepest = 0;
    for (uint k = threadIdx.x; k < n_tiles; k += blockDim.x) {
        const uint64_t offset = tiles[k].work_offset;
        lds_offset[k] = offset;
        lds_order[k] = (ushort)k;
        lds_word[k] = __double_as_longlong(cu::smooth_constant(tiles[k].bailout_sq));
        deepest = max(deepest, tiles[k].max_iter);
    }
    atomicMax(&lds_deepest, deepest);
    __syncthreads();
    deepest = __builtin_amdgcn_readfirstlane(lds_deepest);
    const uint waves = gridDim.x * (blockDim.x >> 6);
    const uint least = min(chunk, 64u);
    // The fewest items of a grab at this depth, and a wave's first ones.
    auto floor_at = [&](uint depth) { return max(min(kGrabSteps / max(depth, 1u), chunk), least); };
    uint first = floor_at(deepest);
    if (total < (uint64_t)waves * first && total >> 32 == 0) {
        const uint spread = deepest < kOrderDepth ? waves : waves / 2u;
        first = min(first, (((uint)total - 1u) / (spread * 64u) + 1u) * 64u);
    }
    const uint64_t first_items = (uint64_t)waves * first;
    bool in_turn = false;  // the table is a tile after the other from 0 on
    bool sorted = false;   // and in more than one class
    float steps = (float)total * (float)deepest;
    if (first_items < total || deepest >= kOrderDepth) [[unlikely]] {
        auto size_of = [&](uint k) {
            return (k + 1 < n_tiles ? tiles[k + 1].work_offset : total) - tiles[k].work_offset;
        };
        int broken = lds_offset[0] != 0, uneven = 0;
        for (uint k = threadIdx.x; k < n_tiles; k += blockDim.x) {
            broken |= size_of(k) >> 32 != 0;
            uneven |= depth_class(tiles[k].max_iter) != depth_class(deepest);
        }
        in_turn = __syncthreads_or(broken) == 0;
        sorted = __syncthreads_or(uneven) != 0 && in_turn;
        if (sorted) {
            for (uint k = threadIdx.x; k < n_tiles; k += blockDim.x)
                lds_word[k] = size_of(k) | (uint64_t)tiles[k].max_iter << 32;
            __syncthreads();
            steps = order_by_depth(lds_word, n_tiles, lds_ordering, lds_order, lds_offset);
            __syncthreads();
            for (uint k = threadIdx.x; k < n_tiles; k += blockDim.x)
                lds_word[k] = __double_as_longlong(cu::smooth_constant(tiles[k].bailout_sq));
            __syncthreads();
        }
    }

    const uint lane = cu::lane_id();
    const uint64_t lanes_below = (1ull << lane) - 1ull;

    uint64_t run = 0, failed = 0, ended = 0;  // lanes by state (cu::run_blocks); the rest are idle
    uint64_t able = 0;                        // lanes whose tile can use unchecked blocks
    cu::LaneOrbit<Real> o = {};
    Real bsq = 4;
    uint tile = 0, px = 0, py = 0, s = 0, count_sum = 0;
    double smooth_sum = 0;
    uint max_iter = 0;
    uint64_t executed = 0;

    // The place in the queue's order of an item: the last with an offset <= item.
    auto place_of = [&](uint64_t item) {
        uint lo = 0, hi = n_tiles - 1;
        while (lo < hi) {
            const uint mid = (lo + hi + 1) >> 1;
            if (lds_offset[mid] <= item) lo = mid; else hi = mid - 1;
        }
        return lo;
    };

    // Wave-uniform chunk cursor.  A wave's first items follow from its number, so the
    // launch does not start with every wave's atomic on the one counter; the counter
    // hands out the items after all of the first ones.  A grab takes `chunk` items
    // while that is at most half of what the launch's waves would each get of the
    // rest, and fewer towards the end: one wave's last 256 pixels of deep orbits would
    // outlast every other wave.  For the same reason the steps its pixels may take are at
    // most an eighth of a wave's share of the batch's.  But not fewer than floor_at: the
    // counter takes an atomic every 12 ns, whatever the number of waves, so grabs of
    // shallow pixels must not be small.
    const uint64_t wave_global = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) +
                                                                (threadIdx.x >> 6));
    const uint share = 33u - __clz(waves);  // log2 of at least twice the waves
    steps /= (float)(8u * waves);             // an eighth of a wave's share
    auto grab_size = [&](uint64_t rest) {
        uint64_t part = rest >> share;
        uint depth = deepest;
        if (sorted && rest != 0) depth = tiles[lds_order[place_of(total - rest)]].max_iter;
        if (in_turn) part = min(part, (uint64_t)fminf(steps / (float)max(depth, 1u), 65536.0f));
        const uint size = part >= chunk ? chunk : max((uint)part, floor_at(depth));
        return (uint)__builtin_amdgcn_readfirstlane(size);
    };
    // `left` of the items from `cur` on are this wave's; scalars, so that the branches
    // on them leave the lane masks scalar too.
    uint64_t cur = wave_global * first;
    auto items_from = [&](uint64_t at, uint size) {
        const uint n = at < total ? (uint)min((uint64_t)size, total - at) : 0u;
        return (uint)__builtin_amdgcn_readfirstlane(n);
    };
    uint left = items_from(cur, first);
    bool exhausted = false;

    for (;;) {
        // ---- refill idle lanes ----
        uint64_t idle = ~(run | ended);
        while (idle != 0 && !exhausted) {
            if (left == 0) {
                const uint size = grab_size(cur < total ? total - cur : 0u);
                unsigned long long base = 0;
                if (lane == 0 && first_items < total) base = atomicAdd(queue, (unsigned long long)size);
                cur = first_items + cu::first_lane(base);
                left = items_from(cur, size);
                if (left == 0) {
                    exhausted = true;
                    break;
                }
            }
            const uint take = min(cu::lanes(idle), left);
            const uint rank = (uint)__popcll(idle & lanes_below);
            const uint64_t taken = idle & cu::ballot(rank < take);
            bool blocks = false;
            if (cu::in_mask(taken)) {
                const uint64_t item = cur + rank;
                const uint place = place_of(item);
                tile = lds_order[place];
                const cu_tile_desc &t = tiles[tile];
                const uint local = (uint)(item - lds_offset[place]);  // a tile holds < 2^32 pixels
                px = local % t.width;
                py = local / t.width;
                s = 0;
                count_sum = 0;
                smooth_sum = 0;
                max_iter = t.max_iter;
                bsq = (Real)t.bailout_sq;
                begin_sample<Real>(t, px, py, 0, o.x, o.y, o.cx, o.cy);
                o.i = 0;
                o.template begin<K>(max_iter, cu::kCycleFirstMixed);
                blocks = tile_blocks_valid(t) && max_iter >= (uint)K;
            }
            const uint64_t ok = cu::ballot(blocks);
            able = (able & ~taken) | ok;
            run |= ok;
            ended |= taken & ~ok;
            cur += take;
            left -= take;
            idle &= ~taken;
        }
        if ((run | ended) == 0) break;

        cu::run_blocks<Real, K, kFused, false>(o, run, failed, ended,
                                               exhausted ? run | ended : ~0ull, refill, max_iter,
                                               bsq);

        // ---- pending lanes: locate the escape or run checked steps, finish the sample ----
        bool another = false;
        if (cu::in_mask(failed | ended)) {
            Real mag2;
            const bool escaped = cu::finish_orbit<Real, K, kFused>(o, failed, max_iter, bsq, mag2);
            const cu_tile_desc &t = tiles[tile];
            executed += o.i;
            count_sum += escaped ? o.i : (t.kind == CU_FRACTAL_JULIA ? max_iter : 0u);
            smooth_sum += escaped ? cu::smooth_value(o.i, (double)mag2,
                                                      __longlong_as_double(lds_word[tile])) : 0.0;
            ++s;
            if (s < t.spp) {
                begin_sample<Real>(t, px, py, s, o.x, o.y, o.cx, o.cy);
                o.i = 0;
                o.template begin<K>(max_iter, cu::kCycleFirstMixed);
                another = true;
            } else {
                const uint64_t at = t.out_offset + (uint64_t)py * t.out_pitch + px;
                counts[at] = count_sum / t.spp;
                if (smooth) smooth[at] = smooth_sum / (double)t.spp;
            }
        }
        const uint64_t more = cu::ballot(another);
        run |= more & able;
        ended = more & ~able;
        failed = 0;
    }
    cu::add_iterations(iters, executed);
}

}  // namespace

#define CU_TILE_KERNELS(NAME, REAL, FUSED)                                                      \
    extern "C" __global__ __launch_bounds__(256) void escapeTile##NAME(                         \
        cu_tile_desc tile, double smooth_c, uint *counts, double *smooth,                       \
        unsigned long long *iters) {                                                            \
        escape_tile<REAL, 16, FUSED>(tile, smooth_c, counts, smooth, iters);                    \
    }                                                                                           \
    extern "C" __global__ __launch_bounds__(256) void escapeTileSamples##NAME(                  \
        cu_tile_desc tile, double smooth_c, uint *counts, double *smooth,                       \
        unsigned long long *iters) {                                                            \
        escape_tile_samples<REAL, 16, FUSED>(tile, smooth_c, counts, smooth, iters);            \
    }                                                                                           \
    extern "C" __global__ __launch_bounds__(256) void escapeTileSamples##NAME##K8(              \
        cu_tile_desc tile, double smooth_c, uint *counts, double *smooth,                       \
        unsigned long long *iters) {                                                            \
        escape_tile_samples<REAL, 8, FUSED>(tile, smooth_c, counts, smooth, iters);             \
    }                                                                                           \
    extern "C" __global__ __launch_bounds__(256) void escapeTilesPersistent##NAME##K8(          \
        const cu_tile_desc *tiles, uint n_tiles, uint64_t total, uint *counts, double *smooth,  \
        unsigned long long *iters, unsigned long long *queue, uint chunk, uint refill) {        \
        escape_tiles_persistent<REAL, 8, FUSED>(tiles, n_tiles, total, counts, smooth, iters,   \
                                                queue, chunk, refill);                          \
    }                                                                                           \
    extern "C" __global__ __launch_bounds__(256) void escapeTilesPersistent##NAME##K16(         \
        const cu_tile_desc *tiles, uint n_tiles, uint64_t total, uint *counts, double *smooth,  \
        unsigned long long *iters, unsigned long long *queue, uint chunk, uint refill) {        \
        escape_tiles_persistent<REAL, 16, FUSED>(tiles, n_tiles, total, counts, smooth, iters,  \
                                                 queue, chunk, refill);                         \
    }                                                                                           \
    extern "C" __global__ __launch_bounds__(256) void escapeTilesPersistent##NAME##K32(         \
        const cu_tile_desc *tiles, uint n_tiles, uint64_t total, uint *counts, double *smooth,  \
        unsigned long long *iters, unsigned long long *queue, uint chunk, uint refill) {        \
        escape_tiles_persistent<REAL, 32, FUSED>(tiles, n_tiles, total, counts, smooth, iters,  \
                                                 queue, chunk, refill);                         \
    }

CU_TILE_KERNELS(DoubleExact, double, false)
CU_TILE_KERNELS(DoubleFused, double, true)
CU_TILE_KERNELS(FloatExact, float, false)
CU_TILE_KERNELS(FloatFused, float, true)

// Palette compose of a smooth plane: idx = L - (round(v) mod L) - 1 (the
// colorize of mandelbrot.cu:27-35 applied to the smooth value; v <= 0 as 0).
extern "C" __global__ __launch_bounds__(256) void composeSmooth(
    const double *smooth, uint smooth_pitch, uint *rgba, uint rgba_pitch, uint width,
    uint height, const uint *palette, uint palette_length) {
    __shared__ uint lds_palette[kPaletteLds];
    const bool staged = palette_length <= kPaletteLds;
    const uint nthreads = blockDim.x * blockDim.y;
    const uint tid = threadIdx.x + threadIdx.y * blockDim.x;
    if (staged)
        for (uint k = tid; k < palette_length; k += nthreads) lds_palette[k] = palette[k];
    __syncthreads();
    const uint *pal = staged ? lds_palette : palette;
    for (uint y = blockIdx.y * blockDim.y + threadIdx.y; y < height; y += gridDim.y * blockDim.y)
        for (uint x = blockIdx.x * blockDim.x + threadIdx.x; x < width;
             x += gridDim.x * blockDim.x) {
            rgba[(size_t)y * rgba_pitch + x] =
                pal[cu::palette_slot(smooth[(size_t)y * smooth_pitch + x], palette_length)];
        }
}

// Order-sensitive checksum of n words: sum of p[i] * (2i + 1) mod 2^64, added to
// *out (integer addition, so the result does not depend on the schedule).  p is
// 16-byte aligned (an allocation's start).  All blocks add to one address, about 10 ns
// each: with an atomic per wave of 2048 blocks a 1280x720 image took 100-115 us, with
// one per block of at most 512 and four words per load it takes 8.5 us.
extern "C" __global__ __launch_bounds__(256) void checksumU32(const uint *p, uint64_t n,
                                                              unsigned long long *out) {
    __shared__ unsigned long long part[4];
    const uint4 *q = reinterpret_cast<const uint4 *>(p);
    const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint64_t acc = 0;
    for (uint64_t k = first; k < n / 4; k += (uint64_t)gridDim.x * blockDim.x) {
        const uint4 v = q[k];
        const uint64_t w = 8ull * k + 1ull;
        acc += v.x * w + v.y * (w + 2ull) + v.z * (w + 4ull) + v.w * (w + 6ull);
    }
    const uint64_t last = n / 4 * 4 + first;  // the words after the last whole four
    if (last < n) acc += (uint64_t)p[last] * (2ull * last + 1ull);
    acc = __ockl_wfred_add_u64(acc);
    if (cu::lane_id() == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, part[0] + part[1] + part[2] + part[3]);
}

extern "C" __global__ __launch_bounds__(256) void fillU32(uint *p, uint value, uint64_t n) {
    for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (uint64_t)gridDim.x * blockDim.x)
        p[k] = value;
}

// The straggler-compaction frame pipeline shares this module's helpers.
#include "escape_pipeline.hip"
// The deep-zoom perturbation form likewise.
#include "perturb.hip"
