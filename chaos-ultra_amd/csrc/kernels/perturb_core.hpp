// perturb_core.hpp — the deep-zoom perturbation form's device code: the
// double-double reference orbit, the perturbation step with rebasing and
// glitch detection, and the per-pixel frame kernels' bodies.  Included by
// perturb.hip (the escape_family module's entry points) and by the library's
// allocation-free deep render (csrc/host/deep_static.hip).
//
// Below a pixel of ~1e-13 of the plane the reference's double kernel cannot
// tell pixels apart (cudarenderer/RenderingKernel.java:124-138 and
// cudarenderer/CudaFractalRenderer.java:217-220 stop there).  This form
// iterates every pixel as a small delta around one reference orbit:
//
//   z_n = Z_m + d_n,   d_{n+1} = (2 Z_m + d_n) d_n + dc,   m <- m + 1
//
// The reference orbit Z is computed once per frame on the GPU by one lane in
// double-double (FP64 error-free transformations, ~106-bit significand): an
// orbit computed in plain FP64 drifts from the true orbit long before the
// pixel scale of a 1e-20 frame.  It is stored rounded to the delta type,
// each entry {Zx, Zy, |Z|^2/2, 0}.  Deltas are FP32 (twice the FP64 issue rate
// on gfx950) or FP64 (far more precise).
//
// Rebasing (Zhuoran): when |z| < |d| — tested as fma(Zx, dx, Zy dy) <
// -|Z|^2/2 — or when the pixel outlives the reference (m == M), the pixel
// restarts the reference from Z_0 = 0 with d = z.  Without rebasing,
// Pauldelbrot's test |z|^2 < eps |Z|^2 marks a pixel glitched and the host
// re-renders glitched pixels around a secondary reference.
//
// Hot loop: blocks of K steps (one orbit load and 9 VALU ops per step).  Where all
// lanes of a wave stand at the same orbit entry and none rebases, the entries come
// through the scalar cache; otherwise each lane reads its own and takes its rebases
// inside the block.  Escape is tested once, at the block's end (escape is permanent
// for bailout_sq >= 4, |c| <= 2), and the blocks with an escape are replayed, all
// lanes' together, with checked steps — the oracle's operation sequence.
#pragma once
#include "cu_types.hpp"
#include "escape_core.hpp"

#pragma clang fp contract(off)

namespace {

// ---- double-double (Dekker / Knuth error-free transformations) ----
struct DD {
    double hi, lo;
};

__device__ __forceinline__ DD dd_two_sum(double a, double b) {
    const double s = a + b;
    const double bb = s - a;
    return {s, (a - (s - bb)) + (b - bb)};
}
// dd_two_sum(2a, b): doubling is exact, so it folds into each operation on 2a.
__device__ __forceinline__ DD dd_two_sum_twice(double a, double b) {
    const double s = __builtin_fma(2.0, a, b);
    const double bb = __builtin_fma(-2.0, a, s);
    return {s, __builtin_fma(2.0, a, -(s - bb)) + (b - bb)};
}
__device__ __forceinline__ DD dd_quick_two_sum(double a, double b) {
    const double s = a + b;
    return {s, b - (s - a)};
}

__device__ __forceinline__ DD dd_two_prod(double a, double b) {
    const double p = a * b;
    return {p, __builtin_fma(a, b, -p)};  // double operands
}

// One step Z <- Z^2 + C of the reference orbit, compensated rather than composed
// from dd_mul and dd_add: the leading products are split exactly, the sums of
// leading terms are exact (two-sums), and the low-order terms (the products'
// errors, the cross terms 2 xh xl - 2 yh yl and 2 (xh yl + xl yh), C's low parts)
// are summed in plain double before one renormalisation; terms of order xl^2 are
// dropped.  The absolute error per step is a few units of 2^-104 |Z|^2, as for
// the composed form, in about half its instructions: the orbit is one lane's
// serial chain, issued one instruction at a time.  Doublings are exact and folded
// into the operation that follows (the same roundings, in 5 instructions fewer).
__device__ __forceinline__ void dd_orbit_step(DD &x, DD &y, DD cx, DD cy) {
    const DD px = dd_two_prod(x.hi, x.hi), py = dd_two_prod(y.hi, y.hi);
    const DD pxy = dd_two_prod(x.hi, y.hi);
    const DD s1 = dd_two_sum(px.hi, -py.hi);
    const DD s2 = dd_two_sum(s1.hi, cx.hi);
    const double u = __builtin_fma(x.hi, x.lo, -(y.hi * y.lo));
    const double xlo = ((s1.lo + s2.lo) + (px.lo - py.lo)) + __builtin_fma(2.0, u, cx.lo);
    const DD s3 = dd_two_sum_twice(pxy.hi, cy.hi);
    const double w = __builtin_fma(x.hi, y.lo, x.lo * y.hi);
    const double ylo = __builtin_fma(2.0, pxy.lo, s3.lo) + __builtin_fma(2.0, w, cy.lo);
    x = dd_quick_two_sum(s2.hi, xlo);
    y = dd_quick_two_sum(s3.hi, ylo);
}

template <class Real>
struct alignas(4 * sizeof(Real)) OrbitEntry {
    Real x, y, h;  // Z_m and |Z_m|^2 / 2
    Real quiet;    // 0, or where a block starts (m % kPlainSteps == 0) its quiet_bound
};

// Steps of the pixel kernels' blocks.
constexpr int kPlainSteps = 32;

// Pointers into LDS and global memory typed with their address spaces, so that
// loads through them stay LDS or global (or scalar) loads: through untyped
// pointers the compiler may merge reads from different branches into one
// generic (flat) load of a selected address.
template <class T>
using lds_ptr = const T __attribute__((address_space(3))) *;
template <class T>
using global_ptr = const T __attribute__((address_space(1))) *;

template <class Real, class Ptr>
__device__ __forceinline__ OrbitEntry<Real> load_entry(Ptr p) {
    OrbitEntry<Real> e;
    e.x = p->x;
    e.y = p->y;
    e.h = p->h;
    e.quiet = 0;
    return e;
}

// The reference orbit as the pixel kernels read it: entries below `staged`
// from the block's LDS copy, the rest (an orbit longer than the LDS budget)
// from global memory.
template <class Real>
struct OrbitView {
    global_ptr<OrbitEntry<Real>> global;
    lds_ptr<OrbitEntry<Real>> lds;
    uint staged;
    __device__ __forceinline__ OrbitEntry<Real> at(uint m) const {
        OrbitEntry<Real> e = load_entry<Real>(lds + (m < staged ? m : 0u));
        if (m >= staged) e = load_entry<Real>(global + m);
        return e;
    }
};

// A state of the orbit where its entry goes: the leading parts of Z_m, in FP64.
typedef double OrbitState __attribute__((ext_vector_type(2), may_alias));

// States 0 .. M of the orbit of C, and M, the first index whose |Z|^2 fails the bailout
// test, or max_iter.
//
// One lane's serial chain.  Alone on its SIMD it issues an instruction about every 5
// cycles, dependent or not, and a taken branch costs it about 30, so what counts is
// instructions and branches: kOrbitRun steps run without a test, each storing its state,
// and when the last one's end fails the test they are taken again one by one from their
// start (escape is permanent: bailout_sq >= 4, |C| <= 2; what is stored past M is not read,
// and lies within the max_iter + 1 entries there are).  Entries are made of the states
// afterwards, by the whole wave: 3088 of them 0.37 -> 0.32 ms, against a test and the
// entry's |Z|^2 and conversions in every step.
constexpr uint kOrbitRun = 8;

template <class Real>
__device__ uint orbit_states(double cx_hi, double cx_lo, double cy_hi, double cy_lo,
                             uint max_iter, double bailout_sq, OrbitEntry<Real> *orbit) {
    const DD cx{cx_hi, cx_lo}, cy{cy_hi, cy_lo};
    DD x{0.0, 0.0}, y{0.0, 0.0};
    uint n = 0;
    auto store = [&](uint at) { *(OrbitState *)(orbit + at) = OrbitState{x.hi, y.hi}; };
    auto inside = [&] {
        const double x2 = x.hi * x.hi;
        const double y2 = y.hi * y.hi;
        return x2 + y2 < bailout_sq;
    };
    while (max_iter - n >= kOrbitRun) {
        const DD x0 = x, y0 = y;
#pragma unroll
        for (uint k = 0; k < kOrbitRun; ++k) {
            store(n + k);
            dd_orbit_step(x, y, cx, cy);
        }
        if (!inside()) {
            x = x0;
            y = y0;
            break;
        }
        n += kOrbitRun;
    }
    for (;;) {
        store(n);
        if (!inside() || n == max_iter) return n;
        dd_orbit_step(x, y, cx, cy);
        ++n;
    }
}

// The entries of states 0 .. M, by one wave.
template <class Real>
__device__ void orbit_entries(OrbitEntry<Real> *orbit, uint M) {
    constexpr uint kTogether = 8;
    for (uint from = threadIdx.x; from <= M; from += 64 * kTogether) {
        OrbitState z[kTogether];
#pragma unroll
        for (uint j = 0; j < kTogether; ++j)
            z[j] = *(const OrbitState *)(orbit + min(from + 64 * j, M));
#pragma unroll
        for (uint j = 0; j < kTogether; ++j) {
            const double x2 = z[j].x * z[j].x;
            const double y2 = z[j].y * z[j].y;
            OrbitEntry<Real> e;
            e.x = (Real)z[j].x;
            e.y = (Real)z[j].y;
            e.h = (Real)(0.5 * (x2 + y2));
            e.quiet = 0;
            if (from + 64 * j <= M) orbit[from + 64 * j] = e;
        }
    }
}

// The reference orbit as the pixel kernels need it beside its entries: the index of the
// last one, and the cycle it ends in: entries m and m + period are the same for all m
// from `start` on (as far as entries go; period 0: no cycle was found, or the orbit
// escapes).
struct OrbitInfo {
    uint last, period, start, pad;
};

// A point inside the set settles into a cycle, and rounded to the delta type its entries
// repeat exactly long before the double-double values do.  One wave looks back from the
// last entry for an equal one, at most kPeriodMax before it, then for the first pair a
// period apart that differs.  For 50001 entries about 0.1 ms, where the orbit took 5 ms.
constexpr uint kPeriodMax = 4096;

template <class Real>
__device__ void orbit_cycle(const OrbitEntry<Real> *orbit, uint M, uint &period, uint &start) {
    const uint lane = threadIdx.x;
    auto alike = [&](uint a, uint b) {
        const OrbitEntry<Real> e = orbit[a], f = orbit[b];
        return e.x == f.x && e.y == f.y && e.h == f.h;
    };
    period = start = 0;
    const uint longest = min(M, kPeriodMax);
    for (uint d = 1; d <= longest; d += 64) {
        const uint64_t hit = cu::ballot(d + lane <= longest && alike(M - min(d + lane, M), M));
        if (hit != 0) {
            period = d + (uint)__builtin_ctzll(hit);
            break;
        }
    }
    if (period == 0) return;
    constexpr uint kAhead = 4;  // wave-widths of entries looked at together
    for (uint top = M - period + 1; top != 0;) {  // indices from `top` on have been found alike
        uint64_t differ[kAhead];
#pragma unroll
        for (uint j = 0; j < kAhead; ++j) {
            const uint back = j * 64 + lane + 1;
            const uint m = top - min(back, top);
            differ[j] = cu::ballot(back <= top && !alike(m, m + period));
        }
#pragma unroll
        for (uint j = 0; j < kAhead; ++j)
            if (differ[j] != 0) {
                start = top - j * 64 - (uint)__builtin_ctzll(differ[j]);
                return;
            }
        top -= min(top, kAhead * 64);
    }
}

// The bound C with which no rebase test fires in the block of kPlainSteps steps from entry
// m, whatever the lane, if (|d| + |dc|) C < 1 at its start.  While |d_j| <= |Z_j| / 4, a
// step gives |d'| <= (2 |Z| + |Z| / 4) |d| + |dc|, so with E = |d| + |dc| at the start
// |d_k| <= E U_k for U_0 = 1, U_k+1 = 2.25 |Z_k| U_k + 1; and at |d| <= |Z| / 4 the test,
// Z.d < -|Z|^2 / 2, is far from firing.  C is the largest 4 U_k / |Z_k|.  The margins of 4 %
// a step are many times the roundings of a step and of this sum, in FP32 too.  Where |Z| is
// small (the orbit starts at 0) there is no bound.
template <class Real>
__device__ float quiet_bound(const OrbitEntry<Real> *orbit, uint m) {
    float u = 1, c = 0;
#pragma unroll 8
    for (int k = 0; k < kPlainSteps; ++k) {
        const float x = (float)orbit[m + k].x, y = (float)orbit[m + k].y;
        const float z = sqrtf(x * x + y * y);
        c = z > 1e-6f ? fmaxf(c, 4.16f * u / z) : __builtin_inff();
        u = 2.35f * z * u + 1.04f;
    }
    return c;
}

// One wave: its first lane computes the orbit, all look for the cycle and for the blocks'
// quiet bounds.
template <class Real>
__device__ void reference_orbit(double cx_hi, double cx_lo, double cy_hi, double cy_lo,
                                uint max_iter, double bailout_sq, OrbitEntry<Real> *orbit,
                                OrbitInfo *info) {
    if (blockIdx.x != 0) return;
    uint n = 0;
    if (threadIdx.x == 0)
        n = orbit_states<Real>(cx_hi, cx_lo, cy_hi, cy_lo, max_iter, bailout_sq, orbit);
    __syncthreads();
    const uint M = __builtin_amdgcn_readfirstlane(n);
    orbit_entries<Real>(orbit, M);
    __syncthreads();
    uint period = 0, start = 0;
    if (M == max_iter && M != 0) orbit_cycle<Real>(orbit, M, period, start);
    for (uint b = threadIdx.x; b < M / kPlainSteps; b += 64)
        orbit[b * kPlainSteps].quiet = (Real)quiet_bound<Real>(orbit, b * kPlainSteps);
    if (threadIdx.x == 0) *info = {M, period, start, 0};
}

struct DeepArgs {
    const void *orbit;         // OrbitEntry<Real>[M + 1]
    const OrbitInfo *info;
    uint *counts;              // W x H, row-major
    double *smooth;
    unsigned char *glitch;     // 1 = glitched (Pauldelbrot) in the last pass over the pixel
    uint *rgba;                // optional palette colour
    const uint *palette;
    unsigned long long *iters; // CU_ITER_SLOTS slots
    double centre_x, centre_y; // direct form only: c = centre + offset
    double pixel_w, pixel_h;
    double ref_ox, ref_oy;     // reference point - frame centre (plane units)
    double bailout_sq;
    double smooth_c;           // log2(log2(bailout_sq))
    uint width, height, max_iter, flags;
    uint palette_length;
    float glitch_eps;
    uint only_glitched;        // 1: pixels whose glitch flag is set, others untouched
    uint pad;
};
static_assert(sizeof(DeepArgs) == 160, "DeepArgs layout");

constexpr uint kDeepRebase = 1u;

__device__ __forceinline__ void deep_offset(const DeepArgs &a, uint px, uint py, double &ox,
                                            double &oy) {
    ox = ((double)px + 0.5 - (double)a.width * 0.5) * a.pixel_w;
    oy = ((double)a.height * 0.5 - ((double)py + 0.5)) * a.pixel_h;
}

// The rebase test |Z + d| < |d|, i.e. |Z|^2 + 2 Z.d < 0, evaluated as
// Zx dx + Zy dy < -h with h = |Z|^2 / 2 from the orbit entry: one product, one
// FMA and a compare.  Every operand taken from the orbit enters a different
// instruction, so a wave that reads the orbit through scalar registers needs no
// copies into vector registers.  At Z = 0 (m = 0, h = 0) the sum is a zero and
// the test does not fire for finite d.
template <class Real>
__device__ __forceinline__ bool rebase_test(Real Zx, Real Zy, Real h, Real dx, Real dy) {
    return cu::fma_r(Zx, dx, Zy * dy) < -h;
}

// The delta of an earlier rebase, for the cycle test.  After a rebase the reference
// index is 0, so the pixel's future is a function of its delta alone: a delta that
// comes back makes the orbit a cycle that never escapes, and the checked loop's result
// is the one at max_iter.  (-0 compares equal to 0: a zero's sign changes no later
// magnitude.)  Before the first rebase the pixel's start is held, a delta of 0 at index
// 0.  Pixels of the set's interior rebase every few hundred steps; by a count on the CPU
// (1e-6 frame, maxIter 50000, three quarters interior) the test leaves 0.48 of the steps
// with FP64 deltas and 0.28 with FP32 ones.
template <class Real>
struct HeldDelta {
    Real x = 0, y = 0;
    __device__ __forceinline__ bool is(Real dx, Real dy) const { return dx == x && dy == y; }
    __device__ __forceinline__ void take(Real dx, Real dy) {
        x = dx;
        y = dy;
    }
};

// One checked step of the perturbation loop (the oracle's or_perturb_pixel
// body).  Returns 0 to continue, 1 escaped (mag set), 2 max_iter, 3 glitched.
template <class Real>
__device__ __forceinline__ int checked_step(const OrbitView<Real> &Z, uint M, Real &dx, Real &dy,
                                            uint &m, uint &n, Real dcx, Real dcy, uint max_iter,
                                            Real bsq, bool rebase, Real geps, Real &mag_out) {
    const OrbitEntry<Real> e = Z.at(m);
    Real Zx = e.x, Zy = e.y;
    const Real zx = Zx + dx;
    const Real zy = Zy + dy;
    const Real mag = cu::fma_r(zx, zx, zy * zy);
    if (!(n < max_iter)) return 2;
    if (!(mag < bsq)) {
        mag_out = mag;
        return 1;
    }
    if (rebase) {
        if (rebase_test(Zx, Zy, e.h, dx, dy) || m == M) {
            dx = zx;
            dy = zy;
            m = 0;
            Zx = 0;
            Zy = 0;
        }
    } else if (m == M) {
        dx = zx;
        dy = zy;
        m = 0;
        Zx = 0;
        Zy = 0;
    } else if (m > 0 && mag < geps * (e.h + e.h)) {
        mag_out = mag;
        return 3;
    }
    const Real ax = cu::fma_r((Real)2, Zx, dx);
    const Real ay = cu::fma_r((Real)2, Zy, dy);
    const Real ndx = cu::fma_r(ax, dx, cu::fma_r(-ay, dy, dcx));
    const Real ndy = cu::fma_r(ax, dy, cu::fma_r(ay, dx, dcy));
    dx = ndx;
    dy = ndy;
    ++m;
    ++n;
    return 0;
}

// K unchecked steps from orbit entry zp[0], the same for all lanes; returns the ballot of
// lanes whose rebase test fired at any of the K states.  No branches: the orbit loads of
// the whole block can be issued ahead of the arithmetic.  Entries are read 64 bytes at a
// time, one scalar load for two FP64 or four FP32 ones: in 1e-10 and 1e-20 frames with
// FP64 deltas 3 % less time than with two loads an entry, 1 to 3 % at 1e-6 (the other
// waves cover the loads' latency; asking one group ahead was slower by a tenth).
//
// Without kTest it leaves the tests out and returns 0, for blocks in which none can fire
// (quiet_bound): 6 VALU instructions a step against 9.
template <class Real, int K, bool kTest>
__device__ __forceinline__ uint64_t unchecked_block(global_ptr<OrbitEntry<Real>> zp, Real &dx,
                                                    Real &dy, Real dcx, Real dcy) {
    constexpr int kTogether = 64 / (int)sizeof(OrbitEntry<Real>);
    typedef Real Entries __attribute__((ext_vector_type(4 * kTogether), aligned(4 * sizeof(Real))));
    uint64_t flagged = 0;
#pragma unroll
    for (int k = 0; k < K; k += kTogether) {
        const Entries z = *(global_ptr<Entries>)(zp + k);
#pragma unroll
        for (int j = 0; j < kTogether; ++j) {
            const Real x = z[4 * j], y = z[4 * j + 1], h = z[4 * j + 2];
            if constexpr (kTest) flagged |= cu::ballot(rebase_test(x, y, h, dx, dy));
            const Real ax = cu::fma_r((Real)2, x, dx);
            const Real ay = cu::fma_r((Real)2, y, dy);
            const Real ndx = cu::fma_r(ax, dx, cu::fma_r(-ay, dy, dcx));
            const Real ndy = cu::fma_r(ax, dy, cu::fma_r(ay, dx, dcy));
            dx = ndx;
            dy = ndy;
        }
    }
    return flagged;
}

// K steps in which each lane takes its own rebases: lane's index is m at step 0, and
// a lane whose test fires (or, kEnd, whose index is M) restarts the reference there
// with d = z and takes the step from Z_0 = 0, as the checked loop does, while the
// others go on.  So a step costs what an unchecked one does, plus a branch and, where
// some lane rebases, a few masked instructions; entries come one step ahead of their
// use, and a rebased lane's next one is Z_1, the same for all.  Every read lies in
// [0, m + K], clamped to M with kEnd.  Returns the running lanes that rebased, with the delta of
// each one's last rebase in (rx, ry); `end` is the entry at the final index.
template <class Real, int K, bool kEnd, class Ptr>
__device__ __forceinline__ uint64_t rebasing_block(Ptr orbit, uint M, const OrbitEntry<Real> &z1,
                                                   uint64_t running, uint &m, Real &dx, Real &dy,
                                                   Real dcx, Real dcy, Real &rx, Real &ry,
                                                   OrbitEntry<Real> &end) {
    uint64_t rebased = 0;
    int first = (int)m;  // the lane's index at step k is first + k
    OrbitEntry<Real> e = load_entry<Real>(orbit + first);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        int ahead = first + (k + 1);
        if constexpr (kEnd) ahead = min(ahead, (int)M);
        OrbitEntry<Real> next = load_entry<Real>(orbit + ahead);
        bool fire = rebase_test(e.x, e.y, e.h, dx, dy);
        if constexpr (kEnd) fire = fire || first + k == (int)M;
        const uint64_t firing = cu::ballot(fire) & running;
        if (firing != 0) {
            cu::seldom();
            rebased |= firing;
            if (cu::in_mask(firing)) {
                dx = rx = e.x + dx;
                dy = ry = e.y + dy;
                e.x = 0;
                e.y = 0;
                next = z1;
                first = -k;
            }
        }
        const Real ax = cu::fma_r((Real)2, e.x, dx);
        const Real ay = cu::fma_r((Real)2, e.y, dy);
        const Real ndx = cu::fma_r(ax, dx, cu::fma_r(-ay, dy, dcx));
        const Real ndy = cu::fma_r(ax, dy, cu::fma_r(ay, dx, dcy));
        dx = ndx;
        dy = ndy;
        e = next;
    }
    m = (uint)(first + K);
    end = e;
    return rebased;
}

// Whole pixel; lanes whose `active` is false only take part in the ballots.
//
// With rebasing, the running lanes take blocks of K steps together, so their
// iteration count n is one scalar.  While they all read the same orbit entries (same
// m) a block reads them through the scalar cache and only collects whether a rebase
// test fired; if one did, it is run again as a rebasing_block, which is taken at once
// where lanes stand at different entries or the last two blocks had to be rerun.
// Escape is tested at a block's end (it is permanent for bailout_sq >= 4, |c| <= 2):
// a lane that left inside a block keeps that block's start, and when no lane runs any
// more all such lanes replay theirs together with checked steps, the oracle's loop
// body; the last max_iter % K steps are checked ones too.  A lane whose rebase delta
// has come back is at a cycle's end (HeldDelta).
//
// A lane that does not rebase, with the reference inside the set, is the other kind of
// cycle: along the reference's own cycle its future is a function of its delta and its
// place in the cycle.  Lanes that are on it when a delta is to be held hold their present
// one (`along`), and it is looked for again a whole number of periods later, at the block
// ends `stride` apart.  (A pixel's index is never above its iteration count, so with a
// reference that runs to max_iter the end of the entries is not reached before the last
// iteration, and entries a period apart are the same entry to it.)
//
// Without rebasing every step is a checked one (the glitch test needs each).
//
// Bound by VALU issue, and by the longest waves once the others have ended; 1920x1080,
// without the reference orbit's time, FP32 / FP64 deltas: 1e-10 (each pixel rebases on
// its own) 1.50 / 2.24 -> 1.00 / 1.73 ms, a shallow frame of width 1 2.85 / 3.80 ->
// 0.44 / 0.73 ms (0.70 / 1.15 without the cycles along the reference's), 1e-20 (few
// rebases) 1.20 / 2.03 -> 0.80 / 1.39 ms (1.14 / 1.88 with the tests in every block);
// before, a block stopped for the whole wave at its first rebase, and each escape was
// replayed as it came, 32 checked steps for one lane.  1e-6, three quarters interior,
// 18.7 / 32.7 -> 8.8 / 19.1 ms, 11.0 / 22.0 of it by the cycle test.
template <class Real, int K>
__device__ int perturb_pixel(const OrbitView<Real> &Z, const OrbitInfo &info, Real dcx,
                             Real dcy, uint max_iter, Real bsq, bool rebase, Real geps,
                             bool active, uint &n_out, Real &mag_out) {
    const uint M = info.last;
    Real dx = 0, dy = 0;
    uint m = 0, n_lane = 0;
    int state = active ? 0 : 4;
    mag_out = 0;
    // Where the reference escapes within a block most pixels do too, and a block with its
    // replay is the longer way (1080p frames beside the set, FP32 / FP64 55 / 86 -> 26 / 31
    // us): checked steps until it has.
    uint n = 0;                          // iterations of the running lanes
    if (rebase && M < (uint)K)
        for (; n < M + 2u && cu::ballot(state == 0) != 0; ++n)
            if (state == 0)
                state = checked_step<Real>(Z, M, dx, dy, m, n_lane, dcx, dcy, max_iter, bsq, rebase,
                                           geps, mag_out);
    if (rebase) {
        uint64_t run = cu::ballot(state == 0), failed = 0;
        Real sx = 0, sy = 0;             // block start
        uint sm = 0;
        Real rx = 0, ry = 0;             // delta of the lane's last rebase
        HeldDelta<Real> held;
        uint hold = 0;                   // iteration count from which the next one is held
        uint64_t along = 0;              // lanes that hold their delta on the reference's cycle
        uint due = 0;                    // iteration count at which theirs is looked for
        const uint stride = info.period * ((uint)K >> __builtin_ctz(info.period | (uint)K));
        uint bounded = 0;                // entry whose quiet_bound, if it has one, is loaded
        Real quiet = __builtin_inff();   // (ahead of its use: a load here would be waited for)
        uint streak = 0;                 // consecutive blocks rerun for a rebase
        const OrbitEntry<Real> z1 = load_entry<Real>(Z.global + min(1u, M));
        while (run != 0 && max_iter - n >= (uint)K) {
            if (cu::in_mask(run)) {
                sx = dx;
                sy = dy;
                sm = m;
            } else {
                m = 0;  // lanes that do not run compute along from entry 0, for no effect
            }
            const uint mu = __builtin_amdgcn_readlane(m, (int)__builtin_ctzll(run));
            const bool same = (cu::ballot(m != mu) & run) == 0;
            const bool near = (cu::ballot(M - m < (uint)K) & run) != 0;
            OrbitEntry<Real> e;
            uint64_t rebased = 0;
            bool plain = same && !near && streak < 2;
            if (plain) {
                const Real bx = dx, by = dy;
                bool none = false;  // whether no test can fire in this block
                if (mu == bounded && mu % (uint)K == 0) {
                    const Real size = __builtin_fabs(dx) + __builtin_fabs(dy) +
                                      (__builtin_fabs(dcx) + __builtin_fabs(dcy));
                    none = (run & ~cu::ballot(size * quiet < 1)) == 0;
                }
                if (none)
                    unchecked_block<Real, K, false>(Z.global + mu, dx, dy, dcx, dcy);
                else
                    plain = (unchecked_block<Real, K, true>(Z.global + mu, dx, dy, dcx, dcy) &
                             run) == 0;
                if (plain) {
                    e = load_entry<Real>(Z.global + (mu + (uint)K));
                    bounded = mu + (uint)K;
                    quiet = Z.global[bounded].quiet;
                    m += (uint)K;
                    streak = 0;
                } else {
                    dx = bx;
                    dy = by;
                    ++streak;
                }
            }
            if (!plain) {
                if (near)
                    rebased = rebasing_block<Real, K, true>(Z.global, M, z1, run, m, dx, dy, dcx,
                                                            dcy, rx, ry, e);
                else if ((cu::ballot(m + (uint)K >= Z.staged) & run) == 0)
                    rebased = rebasing_block<Real, K, false>(Z.lds, M, z1, run, m, dx, dy, dcx,
                                                             dcy, rx, ry, e);
                else
                    rebased = rebasing_block<Real, K, false>(Z.global, M, z1, run, m, dx, dy, dcx,
                                                             dcy, rx, ry, e);
                if (rebased == 0) streak = 0;
            }
            const Real zx = e.x + dx;
            const Real zy = e.y + dy;
            const uint64_t out = run & ~cu::ballot(cu::fma_r(zx, zx, zy * zy) < bsq);
            if (out != 0) {
                cu::seldom();
                failed |= out;
                run &= ~out;
                if (cu::in_mask(out)) n_lane = n;  // where its block starts
            }
            n += (uint)K;
            rebased &= run;
            if (rebased != 0) {
                cu::seldom();
                const uint64_t cycle = rebased & ~along & cu::ballot(held.is(rx, ry));
                if (cu::in_mask(cycle)) {
                    n_lane = max_iter;
                    state = 2;
                }
                run &= ~cycle;
                if (cu::in_mask(along & rebased)) held.take(rx, ry);
                along &= ~rebased;
            }
            if (n == due) {
                cu::seldom();
                const uint64_t cycle = run & along & cu::ballot(held.is(dx, dy));
                if (cu::in_mask(cycle)) {
                    n_lane = max_iter;
                    state = 2;
                }
                run &= ~cycle;
                due += stride;
            }
            if (n >= hold) {
                cu::seldom();
                along = stride != 0 ? run & cu::ballot(m >= info.start) : 0;
                if (cu::in_mask(along))
                    held.take(dx, dy);
                else
                    held.take(rx, ry);
                due = n + stride;
                hold = n + n / 2;
            }
        }
        if (cu::in_mask(run)) n_lane = n;
        if (cu::in_mask(failed)) {
            dx = sx;
            dy = sy;
            m = sm;
        }
    }
    while (cu::ballot(state == 0) != 0)
        if (state == 0)
            state = checked_step<Real>(Z, M, dx, dy, m, n_lane, dcx, dcy, max_iter, bsq, rebase,
                                       geps, mag_out);
    n_out = n_lane;
    return state;
}

__device__ __forceinline__ void deep_write(const DeepArgs &a, uint64_t o, int state, uint n,
                                           double mag) {
    const uint count = (state == 1 || state == 3) ? n : 0u;  // Mandelbrot: max_iter -> 0
    const double sm = state == 1 ? cu::smooth_value(n, mag, a.smooth_c) : 0.0;
    a.counts[o] = count;
    if (a.smooth) a.smooth[o] = sm;
    if (a.glitch) a.glitch[o] = state == 3 ? 1 : 0;
    if (a.rgba) {
        a.rgba[o] = a.palette[cu::palette_slot(sm, a.palette_length)];
    }
}

// A block of WX x WY waves, each wave 8 x 8 pixels.
template <uint WX, uint WY>
__device__ __forceinline__ void deep_pixel_coords(uint &px, uint &py) {
    const uint lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    px = (blockIdx.x * WX + (wave % WX)) * 8u + (lane & 7u);
    py = (blockIdx.y * WY + (wave / WX)) * 8u + (lane >> 3);
}

// Perturbation blocks stage the first LdsBytes of the orbit in LDS and share it
// among their WX x WY waves.  A CU holds 160 KB of LDS and 32 waves, and a
// block's wave slots only free up when its slowest wave ends, so smaller blocks
// keep more waves resident; larger copies keep more of the orbit in LDS.
//   FP32: 2 x 2 waves (16 x 16 pixels, 256 threads), 20 KB = 1280 entries, 8 blocks per CU
//   FP64: 4 x 2 waves (32 x 16 pixels, 512 threads), 40 KB = 1280 entries, 4 blocks per CU
template <class Real, int K, uint WX, uint WY, uint LdsBytes>
__device__ void perturb_frame(const DeepArgs a, const OrbitEntry<Real> *__restrict__ orbit) {
    static_assert(K == kPlainSteps, "the orbit's quiet bounds are for blocks of that length");
    __shared__ OrbitEntry<Real> lds[LdsBytes / sizeof(OrbitEntry<Real>)];
    const OrbitInfo info = *a.info;
    const uint staged = min(info.last + 1u, LdsBytes / (uint)sizeof(OrbitEntry<Real>));
    for (uint k = threadIdx.x; k < staged; k += blockDim.x) lds[k] = orbit[k];
    __syncthreads();
    const OrbitView<Real> view{(global_ptr<OrbitEntry<Real>>)orbit,
                               (lds_ptr<OrbitEntry<Real>>)lds, staged};
    uint px, py;
    deep_pixel_coords<WX, WY>(px, py);
    const uint64_t o = (uint64_t)py * a.width + px;
    bool active = px < a.width && py < a.height;
    if (active && a.only_glitched) active = a.glitch[o] != 0;
    Real dcx = 0, dcy = 0;
    if (active) {
        double ox, oy;
        deep_offset(a, px, py, ox, oy);
        dcx = (Real)(ox - a.ref_ox);
        dcy = (Real)(oy - a.ref_oy);
    }
    uint n = 0;
    Real mag = 0;
    const int state = perturb_pixel<Real, K>(
        view, info, dcx, dcy, a.max_iter, (Real)a.bailout_sq,
        (a.flags & kDeepRebase) != 0, (Real)a.glitch_eps, active, n, mag);
    if (active) deep_write(a, o, state, n, (double)mag);
    cu::add_iterations(a.iters, active ? (uint64_t)n : 0u);
}

// Direct FP64 at c = centre + offset: the reference loop with bailout_sq.
template <int K, bool kFused>
__device__ void deep_direct(const DeepArgs a) {
    uint px, py;
    deep_pixel_coords<2, 2>(px, py);
    const bool active = px < a.width && py < a.height;
    uint64_t executed = 0;
    if (active) {
        double ox, oy;
        deep_offset(a, px, py, ox, oy);
        const double cx = a.centre_x + ox, cy = a.centre_y + oy;
        const cu::Orbit<double> r = cu::escape_orbit<double, K, kFused>(
            0.0, 0.0, cx, cy, a.max_iter, a.bailout_sq, a.bailout_sq >= 4.0);
        executed = r.n;
        deep_write(a, (uint64_t)py * a.width + px, r.escaped ? 1 : 2, r.n, r.mag2);
    }
    cu::add_iterations(a.iters, executed);
}

}  // namespace
