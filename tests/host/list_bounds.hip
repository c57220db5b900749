// CPU checks of the brick lists' sizes:
//   1. max_sections(): the offsets of the longest lists a launch may have (as
//      many sections as it allows, each in plane_hits() bricks, one work item
//      per pair and one per key) are ints, and one section more would not
//      fit, for every shape and box size.
// Exit status 0 when every check holds.
#include <climits>
#include <cstdio>

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
    std::printf("%ld checks, %ld failures\n", checks, fails);
    if (fails) return 1;
    std::printf("list bound checks passed\n");
    return 0;
}
