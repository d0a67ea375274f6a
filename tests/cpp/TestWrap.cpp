// Wrapping, z-bins, lattice images and grid points of any position (csrc/atm_wrap.h), on the host.
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "atm_wrap.h"

using namespace atm;

static int failures = 0;
#define CHECK(ok, ...)                                  \
    do {                                                \
        if (!(ok) && ++failures < 20) {                 \
            printf("%s:%d: ", #ok, __LINE__);           \
            printf(__VA_ARGS__);                        \
            printf("\n");                               \
        }                                               \
    } while (0)

static std::vector<float> numbers(std::mt19937& rng, int n) {
    std::vector<float> v = {0.f, -0.f, 1e-45f, -1e-45f, 3.4028235e38f, -3.4028235e38f, INFINITY, -INFINITY, NAN};
    std::uniform_real_distribution<double> u(0.0, 1.0);
    for (int k = 0; k < n; ++k) {
        float x;
        uint32_t bits = rng();
        std::memcpy(&x, &bits, 4);  // every exponent and sign
        v.push_back(x);
        v.push_back((float)std::ldexp(u(rng) * 2 - 1, (int)(rng() % 60) - 10));
        v.push_back((float)(std::floor(20 * (u(rng) - 0.5) * 1048576.0) / 1048576.0));  // the 2^-20 grid
    }
    return v;
}

int main() {
    std::mt19937 rng(5);
    const std::vector<float> x = numbers(rng, 20000);
    for (float L : {1.8f, 3.1f, 8.8f, 41.37f}) {
        const float invL = (float)(1.0 / L);
        for (float v : x) {
            const float w = wrap_coord(v, L, invL);
            if (!std::isfinite(v)) { CHECK(std::isnan(w), "%g -> %g in %g", v, w, L); continue; }
            CHECK(w >= 0.f && w <= L, "%g -> %g in %g", v, w, L);
            // an image of the position itself, to the rounding of one step
            if (std::fabs(v) < 1e6f) {
                const double r = std::remainder((double)v - (double)w, (double)L);
                CHECK(std::fabs(r) <= 1.2e-7 * L, "%.9g -> %.9g in %g: off by %g", v, w, L, r);
            }
        }
        const float Lt[3] = {L, 0.9f * L, 1.1f * L}, inv[3] = {(float)(1.0 / Lt[0]), (float)(1.0 / Lt[1]), (float)(1.0 / Lt[2])};
        for (float s : {0.5f, -0.5f, 0.23f, 0.f}) {
            const float tilt[3] = {s * Lt[0], -s * Lt[0], s * Lt[1]};
            for (size_t k = 0; k + 2 < x.size(); ++k) {
                const float p[3] = {x[k], x[(7 * k + 1) % x.size()], x[(13 * k + 2) % x.size()]};
                float a = p[0], b = p[1], c = p[2];
                wrap_tri(Lt, inv, tilt, a, b, c);
                CHECK(!(a < 0.f || a > Lt[0] || b < 0.f || b > Lt[1] || c < 0.f || c > Lt[2]), "%g %g %g -> %g %g %g", p[0],
                      p[1], p[2], a, b, c);
                if (std::fabs(p[0]) + std::fabs(p[1]) + std::fabs(p[2]) < 1e3f) {  // back by whole lattice vectors
                    const double nc = std::round(((double)p[2] - c) / Lt[2]), nb = std::round((p[1] - b - nc * tilt[2]) / Lt[1]);
                    const double ry = p[1] - b - nc * tilt[2] - nb * Lt[1], rz = p[2] - c - nc * Lt[2];
                    const double rx = std::remainder(p[0] - a - nc * tilt[1] - nb * tilt[0], (double)Lt[0]);
                    CHECK(std::fabs(rx) + std::fabs(ry) + std::fabs(rz) < 2e-3, "%g %g %g: off by %g %g %g", p[0], p[1], p[2], rx, ry, rz);
                }
            }
        }
        for (size_t k = 0; k + 1 < x.size(); ++k) {
            const float d = x[k], reach = std::fabs(x[k + 1]);
            int n0, n1;
            image_range(d, reach, invL, n0, n1);
            CHECK(n0 >= -8 && n1 <= 8, "d %g reach %g: %d..%d", d, reach, n0, n1);
            if (!(std::fabs(d) <= 3 * L && reach <= 2 * L)) continue;  // differences and boxes inside the cell
            for (int n = -20; n <= 20; ++n)
                CHECK(std::fabs((double)d - n * (double)L) >= reach || (n >= n0 && n <= n1), "d %g reach %g: image %d missed (%d..%d)",
                      d, reach, n, n0, n1);
        }
        for (int nz : {1, 2, 3, 5, 17, 64, 333, 4096}) {
            const float invZe = (float)(nz / (double)L);
            for (size_t k = 0; k < x.size(); k += 11) {
                const float z = x[k];  // wrapped or not: the indices stay inside
                for (float hz : {0.f, 1e-6f, 0.3f * L, 0.4999f * L, 0.5f * L, 0.501f * L}) {
                    int a0, a1, b0, b1;
                    z_bins(z, hz, invZe, L, nz, a0, a1, b0, b1);
                    CHECK(0 <= a0 && a0 <= a1 && a1 < nz, "z %g hz %g nz %d: %d %d", z, hz, nz, a0, a1);
                    CHECK(b0 > b1 || (0 <= b0 && b1 < nz && (b0 > a1 || b1 < a0)), "z %g hz %g nz %d: %d %d | %d %d", z, hz, nz, a0, a1, b0, b1);
                    if (!(z >= 0.f && z <= L) || nz > 64) continue;
                    for (int q = 0; q < nz; ++q) {  // a bin within hz of z under some image is in a range
                        bool near = false;
                        for (int n = -1; n <= 1; ++n) {
                            const double lo = (double)L * q / nz + n * (double)L, hi = (double)L * (q + 1) / nz + n * (double)L;
                            near |= lo <= z + hz && hi >= z - hz;
                        }
                        CHECK(!near || (q >= a0 && q <= a1) || (q >= b0 && q <= b1), "z %g hz %g nz %d: bin %d missed", z, hz, nz, q);
                    }
                }
            }
        }
    }
    for (double L : {3.05, 4.217, 41.37}) {
        const double invL = 1.0 / L;
        for (int k = 0; k < 200000; ++k) {
            double v;
            uint64_t bits = (uint64_t)rng() << 32 | rng();
            std::memcpy(&v, &bits, 8);  // every exponent and sign
            if (k & 1) v = std::ldexp((double)rng() / 4294967296.0 - 0.5, (int)(rng() % 90) - 10);
            const double f = grid_fraction(v, invL);
            for (int K : {5, 27, 35, 1024}) {
                const int g = (int)std::floor(f * K);
                CHECK(g >= -1 && g <= K, "%g: grid point %d of %d", v, g, K);
            }
            for (int m : {3, 4, 40}) {
                double w;
                const int c = wrap_cell(v, L, invL, m, &w);
                CHECK(c >= 0 && c < m && w >= 0.0 && w < L, "%g: cell %d of %d, %g", v, c, m, w);
                if (std::fabs(v) < 1e6) {
                    CHECK(std::fabs(std::remainder(v - w, L)) < 1e-9, "%.17g -> %.17g in %g", v, w, L);
                    const double df = f * L - w;
                    CHECK(std::fabs(std::remainder(df, L)) < 1e-9, "%.17g -> %.17g in %g: fraction %.17g", v, w, L, f);
                }
            }
        }
    }
    printf(failures ? "%d failures\n" : "Done\n", failures);
    return failures ? 1 : 0;
}
