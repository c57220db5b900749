// CPU checks of the unit-cell insertion's host-callable parts:
//   1. half_away(x) is roundf(x) for every float in [0, 5000);
//   2. the list builders keep every (brick, section) pair that holds a sample:
//      for random, axis-aligned and diagonal rotations, every lattice sample
//      of the disk lies in a brick (by the floor of its effective position)
//      whose member test and group test the section's plane passes.
// Exit status 0 when every check holds.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "insert_cells.hpp"

using namespace spbp;

int main() {
    long fails = 0, checks = 0;
    for (unsigned u = 0;; ++u) {
        float x;
        std::memcpy(&x, &u, 4);
        if (!(x < 5000.0f)) break;
        ++checks;
        if (half_away(x) != (int)roundf(x)) ++fails;
    }
    std::mt19937_64 rng(11);
    std::uniform_real_distribution<double> uni(0.0, 1.0);
    for (int nx : {4, 9, 16, 33, 64}) {
        BrickGrid bg;
        bg.bx = bg.by = bg.bz = CELL_EDGE;
        bg.own = 2;
        bg.nbx = (nx + bg.bx - 1) / bg.bx;
        bg.nby = (2 * nx - 1 + bg.by - 1) / bg.by;
        bg.nbz = (2 * nx - 1 + bg.bz - 1) / bg.bz;
        bg.nb = bg.nbx * bg.nby * bg.nbz;
        const int nsx = (bg.nbx + 1) / 2, nsy = (bg.nby + 1) / 2;
        for (int r = 0; r < 60; ++r) {
            const bool grid = r < 16;
            const double a = grid ? (r & 3) * M_PI / 4 : 2 * M_PI * uni(rng), b = grid ? (r >> 2) * M_PI / 4 : std::acos(2 * uni(rng) - 1),
                         c = grid ? 0.0 : 2 * M_PI * uni(rng);
            const double ca = std::cos(a), sa = std::sin(a), cb = std::cos(b), sb = std::sin(b), cc = std::cos(c), sc = std::sin(c);
            const float d[9] = {(float)(cc * cb * ca - sc * sa), (float)(sc * cb * ca + cc * sa), (float)(-sb * ca),
                                (float)(-cc * cb * sa - sc * ca), (float)(-sc * cb * sa + cc * ca), (float)(sb * sa),
                                (float)(sb * cc), (float)(sb * sc), (float)cb};
            const float4 n = make_float4(d[6], d[7], d[8], 0.0f);
            for (int I = 0; I <= nx; ++I)
                for (int J = -nx + 1; J <= nx; ++J) {
                    if (!(I * I + J * J < nx * nx) || (I == 0 && J < 0)) continue;
                    float e[3];
                    for (int k = 0; k < 3; ++k) {
                        volatile float u = (float)I * d[k], v = (float)J * d[3 + k];
                        e[k] = u + v;
                    }
                    if (e[0] < 0.0f)
                        for (float& q : e) q = -q;
                    const int i = (int)std::floor(e[0]), j = (int)std::floor(e[1]) + nx - 1, k = (int)std::floor(e[2]) + nx - 1;
                    // ONELINE's bounds keep the nearest voxel (and so the cell) inside the grid of bricks
                    const int q[3] = {(int)(e[0] + 0.5f + 2 * nx) - 2 * nx, (int)(e[1] + 0.5f + 2 * nx) - 2 * nx,
                                      (int)(e[2] + 0.5f + 2 * nx) - 2 * nx};
                    if (q[0] > nx - 3 || q[1] < -nx + 4 || q[1] > nx - 3 || q[2] < -nx + 4 || q[2] > nx - 3) continue;
                    const int bi = i / bg.bx, bj = j / bg.by, bk = k / bg.bz;
                    const int s = bi / 2 + nsx * (bj / 2 + nsy * (bk / 2)), m = (bi & 1) | (bj & 1) << 1 | (bk & 1) << 2;
                    const SuperBrick sbk = superbrick(bg, s, nx);
                    ++checks;
                    const int brick = bi + bg.nbx * (bj + bg.nby * bk);
                    if (j < 0 || k < 0 || bi >= bg.nbx || bj >= bg.nby || bk >= bg.nbz || sbk.b[m] != brick ||
                        member(bg, s, m) != brick || !member_hit(sbk, m, n) || !superbrick_hit(sbk, nx, n)) {
                        if (fails < 10)
                            std::fprintf(stderr, "nx %d: sample (%d, %d) at (%g %g %g): brick %d not listed\n", nx, I, J, e[0],
                                         e[1], e[2], brick);
                        ++fails;
                    }
                }
        }
    }
    std::printf("%ld checks, %ld failures\n", checks, fails);
    if (fails) return 1;
    std::printf("cell list checks passed\n");
    return 0;
}
