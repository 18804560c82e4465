// Grid of the tiled z-march (tm_grid) on host alone: reads "nx ny nz" lines,
// prints "grid.x grid.y grid.z zc" for each.
#include <cstdio>

#include "../../fluid-engine-dev_amd/csrc/jg_device.h"

int main() {
    jg::Dims d;
    while (std::scanf("%d %d %d", &d.nx, &d.ny, &d.nz) == 3) {
        dim3 grid;
        int zc = 0;
        jg::tm_grid(d, grid, zc);
        std::printf("%u %u %u %d\n", grid.x, grid.y, grid.z, zc);
        std::fflush(stdout);
    }
}
