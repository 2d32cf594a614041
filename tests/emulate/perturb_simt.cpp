// The perturbation kernels' device code (chaos-ultra_amd/csrc/kernels/perturb_core.hpp), as it
// is, on the CPU: 64 lanes in lockstep at their operations across lanes (simt/simt.hpp).
// The reference orbit, its cycle and the blocks' bounds are compared with the oracle's orbit
// and with plain restatements; 8x8-pixel waves of a frame are compared with the oracle's
// checked loop, bit for bit.  Entries lie against pages that cannot be read, so a read past
// the last one stops the program.
//
//   perturb_simt <32|64> <centre_x> <centre_y> <width> <max_iter> <limit> <waves> <seed>
//
// An orbit of max_iter steps serves frames of `limit` (at most max_iter), as a kept one does.
// Each wave runs four times: with all shortcuts; without the reference's cycle; without the
// blocks that leave their tests out; and with those taken everywhere.  Prints counts:
//   entries, period, start, bounds  mismatches with the oracle's orbit and the restatements
//   pixels                          mismatches in the first three runs
//   operations, uncycled            operations across lanes with all shortcuts and without the cycle
//   tested, unsound                 pixels that differ when no test runs at all, and so
//                                   whether the blocks without tests are reached
//   last, first_period              the orbit's last index and its period
#include <sys/mman.h>
#include <unistd.h>

#include <cstring>

#include "hip/hip_runtime.h"

#include "../../chaos-ultra_amd/csrc/kernels/perturb_core.hpp"
#undef asm
#include "../../oracle/chaos_oracle.h"

extern "C" unsigned long long __ockl_wfred_add_u64(unsigned long long v) { return v; }

namespace {

constexpr uint32_t kWidth = 1920, kHeight = 1080;
constexpr double kBailout = 256.0;

// n entries that end where a page that cannot be read begins.
template <class T>
T *guarded(size_t n) {
    const size_t page = (size_t)sysconf(_SC_PAGESIZE), bytes = (n * sizeof(T) + page - 1) / page * page;
    char *p = (char *)mmap(nullptr, bytes + page, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    mprotect(p + bytes, page, PROT_NONE);
    return (T *)(p + bytes) - n;
}

template <class Real>
uint32_t oracle_orbit(double cx, double cy, uint32_t mi, Real *out) {
    return sizeof(Real) == 4 ? or_reference_orbit_f(cx, 0, cy, 0, mi, kBailout, (float *)out)
                             : or_reference_orbit_d(cx, 0, cy, 0, mi, kBailout, (double *)out);
}

struct Pixel {
    uint32_t n;
    int state;
    double mag;
    bool operator==(const Pixel &o) const {
        return n == o.n && state == o.state && (state != 1 || std::memcmp(&mag, &o.mag, sizeof mag) == 0);
    }
};

template <class Real>
int run(double cx, double cy, double width, uint32_t mi, uint32_t limit, int waves, unsigned seed) {
    typedef OrbitEntry<Real> Entry;
    std::vector<Real> want(4 * ((size_t)mi + 2));
    const uint32_t M = oracle_orbit<Real>(cx, cy, mi, want.data());
    Entry *whole = guarded<Entry>((size_t)mi + 1);
    OrbitInfo info{};
    simt::run([&] { reference_orbit<Real>(cx, 0, cy, 0, mi, kBailout, whole, &info); });
    // the pixels read a copy of the entries there are
    Entry *orbit = guarded<Entry>((size_t)M + 1);
    std::memcpy(orbit, whole, ((size_t)M + 1) * sizeof(Entry));

    uint64_t entries = info.last != M, period = 0, start = 0, bounds = 0;
    for (uint32_t m = 0; m <= M; ++m)
        entries += orbit[m].x != want[4 * m] || orbit[m].y != want[4 * m + 1] || orbit[m].h != want[4 * m + 2];
    auto alike = [&](uint32_t a, uint32_t b) {
        return orbit[a].x == orbit[b].x && orbit[a].y == orbit[b].y && orbit[a].h == orbit[b].h;
    };
    uint32_t p = 0, from = 0;
    if (M == mi)
        for (uint32_t d = 1; d <= M && d <= kPeriodMax && p == 0; ++d)
            if (alike(M - d, M)) p = d;
    if (p != 0)
        for (from = M - p; from != 0 && alike(from - 1, from - 1 + p);) --from;
    period = info.period != p;
    start = info.start != from;
    uint32_t bounded = 0;
    for (uint32_t m = 0; m <= M; ++m) {
        float u = 1, c = 0;
        if (m % kPlainSteps == 0 && m + kPlainSteps <= M)
            for (int k = 0; k < kPlainSteps; ++k) {
                const float x = (float)orbit[m + k].x, y = (float)orbit[m + k].y, z = std::sqrt(x * x + y * y);
                c = z > 1e-6f ? std::fmax(c, 4.16f * u / z) : INFINITY;
                u = 2.35f * z * u + 1.04f;
            }
        bounds += orbit[m].quiet != (Real)c;
        bounded += c > 0 && c < INFINITY;
    }

    constexpr uint32_t kStaged = 1280;
    const uint32_t staged = std::min(M + 1, kStaged);
    Entry *lds = guarded<Entry>(staged);
    const double pw = width / kWidth;
    srand(seed);
    uint64_t pixels = 0, operations = 0, uncycled = 0, tested = 0, untested = 0, unsound = 0;
    for (int w = 0; w < waves; ++w) {
        const uint32_t wx = (uint32_t)(rand() % (kWidth / 8)) * 8, wy = (uint32_t)(rand() % (kHeight / 8)) * 8;
        Real dcx[64], dcy[64];
        Pixel right[64], got[64];
        for (int l = 0; l < 64; ++l) {
            double ox, oy;
            or_deep_offset(wx + (l & 7), wy + (l >> 3), kWidth, kHeight, pw, pw, &ox, &oy);
            dcx[l] = (Real)ox;
            dcy[l] = (Real)oy;
            Real mag = 0;
            if constexpr (sizeof(Real) == 4)
                right[l].n = or_perturb_pixel_f(want.data(), M, dcx[l], dcy[l], limit, (float)kBailout, 1u, 1e-6f, &mag, &right[l].state);
            else
                right[l].n = or_perturb_pixel_d(want.data(), M, dcx[l], dcy[l], limit, kBailout, 1u, 1e-6, &mag, &right[l].state);
            right[l].mag = mag;
        }
        auto differing = [&](const OrbitInfo &with) {
            std::memcpy(lds, orbit, staged * sizeof(Entry));
            simt::run([&] {
                const int l = simt::lane();
                const OrbitView<Real> view{(global_ptr<Entry>)orbit, (lds_ptr<Entry>)lds, staged};
                Real mag = 0;
                uint n = 0;
                const int state = perturb_pixel<Real, 32>(view, with, dcx[l], dcy[l], limit, (Real)kBailout,
                                                          true, (Real)1e-6, true, n, mag);
                got[l] = Pixel{n, state, (double)mag};
            });
            uint64_t bad = 0;
            for (int l = 0; l < 64; ++l) bad += !(got[l] == right[l]);
            return bad;
        };
        uint64_t before = simt::g_operations;
        pixels += differing(info);
        operations += simt::g_operations - before;
        before = simt::g_operations;
        pixels += differing(OrbitInfo{M, 0, 0, 0});
        uncycled += simt::g_operations - before;
        std::vector<Real> quiet((size_t)M / kPlainSteps + 1);
        for (uint32_t m = 0; m <= M; m += kPlainSteps) quiet[m / kPlainSteps] = orbit[m].quiet;
        for (uint32_t m = 0; m <= M; m += kPlainSteps) orbit[m].quiet = INFINITY;
        before = simt::g_operations;
        pixels += differing(info);
        tested += simt::g_operations - before;
        for (uint32_t m = 0; m <= M; m += kPlainSteps) orbit[m].quiet = 0;
        before = simt::g_operations;
        unsound += differing(info);
        untested += simt::g_operations - before;
        for (uint32_t m = 0; m <= M; m += kPlainSteps) orbit[m].quiet = quiet[m / kPlainSteps];
    }
    printf("entries %llu period %llu start %llu bounds %llu pixels %llu operations %llu uncycled %llu "
           "tested %llu untested %llu unsound %llu last %u first_period %u from %u bounded %u\n",
           (unsigned long long)entries, (unsigned long long)period, (unsigned long long)start,
           (unsigned long long)bounds, (unsigned long long)pixels, (unsigned long long)operations,
           (unsigned long long)uncycled, (unsigned long long)tested, (unsigned long long)untested,
           (unsigned long long)unsound, M, info.period, info.start, bounded);
    return entries + period + start + bounds + pixels != 0;
}

}  // namespace

int main(int argc, char **argv) {
    if (argc != 9) return 2;
    const double cx = atof(argv[2]), cy = atof(argv[3]), width = atof(argv[4]);
    const uint32_t mi = (uint32_t)strtoul(argv[5], nullptr, 10), limit = (uint32_t)strtoul(argv[6], nullptr, 10);
    const int waves = atoi(argv[7]);
    const unsigned seed = (unsigned)strtoul(argv[8], nullptr, 10);
    return atoi(argv[1]) == 32 ? run<float>(cx, cy, width, mi, limit, waves, seed)
                               : run<double>(cx, cy, width, mi, limit, waves, seed);
}
