// A CPU model of the perturbation kernel's blocks (perturb_pixel and rebasing_block in
// chaos-ultra_amd/csrc/kernels/perturb_core.hpp), checked pixel by pixel against the
// oracle's checked loop (oracle/deep_oracle.cpp, or_perturb_pixel_f/_d).
//
// 64 lanes take blocks of K steps together; a lane whose rebase test fires, or whose
// index is the orbit's last, restarts the reference inside the block; escape is
// tested at a block's end and replayed from its start with checked steps; a lane whose
// rebase delta equals a held one ends at max_iter.  The model also checks that every
// orbit entry it reads exists.
//
//   perturb_rebasing <32|64> <centre_x> <centre_y> <width_plane> <max_iter> <waves> <seed>
//
// prints "mismatches N outside O cycles C rebases R" and exits 1 when N or O > 0.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../oracle/chaos_oracle.h"

namespace {

constexpr int K = 32;  // steps per block
constexpr uint32_t kWidth = 1920, kHeight = 1080;

inline float fma_r(float a, float b, float c) { return fmaf(a, b, c); }
inline double fma_r(double a, double b, double c) { return fma(a, b, c); }

template <class Real>
struct Wave {
    const std::vector<Real> &Z;  // {x, y, |Z|^2/2, 0} per entry
    uint32_t M, max_iter;
    uint64_t outside = 0, cycles = 0, rebases = 0;

    struct Lane {
        Real dcx, dcy, dx = 0, dy = 0, sx = 0, sy = 0, rx = 0, ry = 0, hx = 0, hy = 0;
        uint32_t m = 0, sm = 0, n = 0;
        int state = 0;  // 0 running or to be finished with checked steps, 2 max_iter
        bool run = true;
    };

    Real at(int64_t m, int field) {
        if (m < 0 || m > (int64_t)M) {
            ++outside;
            return 0;
        }
        return Z[4 * (size_t)m + (size_t)field];
    }

    void block(Lane &l, bool &rebased) {
        int64_t first = l.m;
        const bool end = M - l.m < (uint32_t)K;
        for (int k = 0; k < K; ++k) {
            Real Zx = at(first + k, 0), Zy = at(first + k, 1);
            if (fma_r(Zx, l.dx, Zy * l.dy) < -at(first + k, 2) || (end && first + k == (int64_t)M)) {
                l.dx = l.rx = Zx + l.dx;
                l.dy = l.ry = Zy + l.dy;
                Zx = Zy = 0;
                first = -k;
                rebased = true;
                ++rebases;
            }
            const Real ax = fma_r((Real)2, Zx, l.dx), ay = fma_r((Real)2, Zy, l.dy);
            const Real nx = fma_r(ax, l.dx, fma_r(-ay, l.dy, l.dcx));
            const Real ny = fma_r(ax, l.dy, fma_r(ay, l.dx, l.dcy));
            l.dx = nx;
            l.dy = ny;
        }
        l.m = (uint32_t)(first + K);
    }

    void go(Lane (&L)[64]) {
        uint32_t n = 0, hold = 0;
        auto running = [&] { return std::any_of(L, L + 64, [](const Lane &l) { return l.run; }); };
        while (running() && max_iter - n >= (uint32_t)K) {
            for (Lane &l : L) {
                if (!l.run) continue;
                l.sx = l.dx;
                l.sy = l.dy;
                l.sm = l.m;
                bool rebased = false;
                block(l, rebased);
                const Real zx = at(l.m, 0) + l.dx, zy = at(l.m, 1) + l.dy;
                if (!(fma_r(zx, zx, zy * zy) < (Real)256)) {  // replayed from the start
                    l.run = false;
                    l.n = n;
                    l.dx = l.sx;
                    l.dy = l.sy;
                    l.m = l.sm;
                } else if (rebased && l.rx == l.hx && l.ry == l.hy) {
                    l.run = false;
                    l.n = max_iter;
                    l.state = 2;
                    ++cycles;
                }
            }
            n += (uint32_t)K;
            if (n >= hold) {
                for (Lane &l : L) {
                    l.hx = l.rx;
                    l.hy = l.ry;
                }
                hold = n + n / 2;
            }
        }
        for (Lane &l : L)
            if (l.run) l.n = n;
    }
};

// The oracle's loop from (dx, dy, m, n) on.
template <class Real>
int finish(const std::vector<Real> &Z, uint32_t M, uint32_t max_iter, Real &dx, Real &dy, uint32_t m,
           uint32_t &n, Real dcx, Real dcy, Real &mag) {
    for (;;) {
        Real Zx = Z[4 * m], Zy = Z[4 * m + 1];
        const Real x = Zx + dx, y = Zy + dy, mg = fma_r(x, x, y * y);
        if (!(n < max_iter)) return 2;
        if (!(mg < (Real)256)) {
            mag = mg;
            return 1;
        }
        if (fma_r(Zx, dx, Zy * dy) < -Z[4 * m + 2] || m == M) {
            dx = x;
            dy = y;
            m = 0;
            Zx = Zy = 0;
        }
        const Real ax = fma_r((Real)2, Zx, dx), ay = fma_r((Real)2, Zy, dy);
        const Real nx = fma_r(ax, dx, fma_r(-ay, dy, dcx)), ny = fma_r(ax, dy, fma_r(ay, dx, dcy));
        dx = nx;
        dy = ny;
        ++m;
        ++n;
    }
}

template <class Real>
int run(double cx, double cy, double width_plane, uint32_t max_iter, int waves, unsigned seed) {
    std::vector<Real> Z(4 * ((size_t)max_iter + 2), 0);
    const uint32_t M = sizeof(Real) == 4
                           ? or_reference_orbit_f(cx, 0, cy, 0, max_iter, 256.0, (float *)Z.data())
                           : or_reference_orbit_d(cx, 0, cy, 0, max_iter, 256.0, (double *)Z.data());
    const double pw = width_plane / kWidth;
    srand(seed);
    uint64_t bad = 0;
    Wave<Real> w{Z, M, max_iter};
    for (int k = 0; k < waves; ++k) {
        const uint32_t wx = (uint32_t)(rand() % (kWidth / 8)) * 8, wy = (uint32_t)(rand() % (kHeight / 8)) * 8;
        typename Wave<Real>::Lane L[64];
        for (int l = 0; l < 64; ++l) {
            double ox, oy;
            or_deep_offset(wx + (l & 7), wy + (l >> 3), kWidth, kHeight, pw, pw, &ox, &oy);
            L[l].dcx = (Real)ox;
            L[l].dcy = (Real)oy;
        }
        w.go(L);
        for (auto &l : L) {
            Real mag = 0, want_mag = 0;
            if (l.state == 0)
                l.state = finish<Real>(Z, M, max_iter, l.dx, l.dy, l.m, l.n, l.dcx, l.dcy, mag);
            int state = 0;
            uint32_t n;
            if constexpr (sizeof(Real) == 4)
                n = or_perturb_pixel_f(Z.data(), M, l.dcx, l.dcy, max_iter, 256.f, 1u, 1e-6f, &want_mag, &state);
            else
                n = or_perturb_pixel_d(Z.data(), M, l.dcx, l.dcy, max_iter, 256.0, 1u, 1e-6, &want_mag, &state);
            if (n != l.n || state != l.state || (state == 1 && std::memcmp(&mag, &want_mag, sizeof mag) != 0)) ++bad;
        }
    }
    printf("mismatches %llu outside %llu cycles %llu rebases %llu\n", (unsigned long long)bad,
           (unsigned long long)w.outside, (unsigned long long)w.cycles, (unsigned long long)w.rebases);
    return bad != 0 || w.outside != 0;
}

}  // namespace

int main(int argc, char **argv) {
    if (argc != 8) return 2;
    const double cx = atof(argv[2]), cy = atof(argv[3]), width = atof(argv[4]);
    const uint32_t max_iter = (uint32_t)strtoul(argv[5], nullptr, 10);
    const int waves = atoi(argv[6]);
    const unsigned seed = (unsigned)strtoul(argv[7], nullptr, 10);
    return atoi(argv[1]) == 32 ? run<float>(cx, cy, width, max_iter, waves, seed)
                               : run<double>(cx, cy, width, max_iter, waves, seed);
}
