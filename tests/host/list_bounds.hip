// CPU checks of the brick lists' sizes:
//   1. max_sections(): the offsets of the longest lists a launch may have (as
//      many sections as it allows, each in plane_hits() bricks, one work item
//      per pair and one per key) are ints, and one section more would not
//      fit, for every shape and box size.
//   2. plane_hits(): no section's plane hits more bricks, by the list
//      builders' own tests, for every shape and for random, axis-aligned,
//      diagonal and (within the host's 1e-4) not quite orthonormal rotations,
//      their normals formed as the builders form them.
// Exit status 0 when every check holds.
#include <climits>
#include <cmath>
#include <cstdio>
#include <random>

#include "insert.hpp"

using namespace spbp;

int main() {
    long fails = 0, checks = 0;
    for (int nx = 4; nx <= 1024; ++nx)
        for (int shape = 0; shape <= NSHAPES; ++shape) {
            const BrickGrid bg = shape_grid(nx, shape);
            const size_t n = max_sections(bg), hits = plane_hits(bg), keys = 2 * (size_t)bg.nb;
            ++checks;
            if (n < 1 || n * hits + keys > (size_t)INT_MAX || (n + 1) * hits + keys <= (size_t)INT_MAX) {
                if (fails < 10) std::fprintf(stderr, "nx %d shape %d: %zu sections of %zu bricks\n", nx, shape, n, hits);
                ++fails;
            }
        }
    std::mt19937_64 rng(17);
    std::uniform_real_distribution<double> uni(0.0, 1.0);
    std::normal_distribution<double> nd;
    for (int nx : {4, 5, 9, 10, 16, 33, 64, 75, 128})
        for (int shape = 0; shape <= NSHAPES; ++shape) {
            const BrickGrid bg = shape_grid(nx, shape);
            const int ns = ((bg.nbx + 1) / 2) * ((bg.nby + 1) / 2) * ((bg.nbz + 1) / 2);
            const size_t most = plane_hits(bg);
            for (int q = 0; q < 200; ++q) {
                const bool grid = q < 64;
                const double a = grid ? (q & 3) * M_PI / 4 : 2 * M_PI * uni(rng),
                             b = grid ? (q >> 2 & 3) * M_PI / 4 : q < 80 ? std::acos(1 / std::sqrt(3.0)) : std::acos(2 * uni(rng) - 1),
                             c = grid ? (q >> 4) * M_PI / 4 : q < 80 ? M_PI / 4 : 2 * M_PI * uni(rng);
                const double ca = std::cos(a), sa = std::sin(a), cb = std::cos(b), sb = std::sin(b), cc = std::cos(c), sc = std::sin(c);
                double d[6] = {cc * cb * ca - sc * sa, sc * cb * ca + cc * sa, -sb * ca,
                               -cc * cb * sa - sc * ca, -sc * cb * sa + cc * ca, sb * sa};
                if (q % 4 == 3)   // rows 1-2 with |r|^2 and r1 . r2 up to 1e-4 off
                    for (double& v : d) v += 2.5e-5 * std::fmax(-1.0, std::fmin(1.0, nd(rng)));
                float r[6];
                for (int k = 0; k < 6; ++k) r[k] = (float)d[k];
                const float4 g = section_plane(r, 0);
                size_t hits = 0;
                for (int s = 0; s < ns; ++s) {
                    const SuperBrick sbk = superbrick(bg, s, nx);
                    if (!superbrick_hit(sbk, nx, g)) continue;
                    for (int m = 0; m < 8; ++m) hits += sbk.b[m] >= 0 && member_hit(sbk, m, g);
                }
                ++checks;
                if (hits > most || hits < 1) {
                    if (fails < 10) std::fprintf(stderr, "nx %d shape %d rotation %d: %zu bricks, bound %zu\n", nx, shape, q, hits, most);
                    ++fails;
                }
            }
        }
    std::printf("%ld checks, %ld failures\n", checks, fails);
    if (fails) return 1;
    std::printf("list bound checks passed\n");
    return 0;
}
