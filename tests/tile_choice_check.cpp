// The 3+1D tile variant vh::mixed_tile_3d picks for one event of each size,
// and for events together: prints "nx ny nz variant" lines, then the two mixes.
#include <cstdio>

#include "../cpu-vh_amd/csrc/vh_kernels.hpp"

int main() {
    const int ny[] = {1, 4, 5, 6, 17, 65}, nz[] = {2, 3, 33};
    for (int nx = 1; nx <= 140; ++nx)
        for (int y : ny)
            for (int z : nz) std::printf("%d %d %d %d\n", nx, y, z, vh::mixed_tile_3d({{nx, y, z}}));
    std::printf("mix %d\n", vh::mixed_tile_3d({{17, 17, 17}, {101, 101, 41}}));
    std::printf("mix %d\n", vh::mixed_tile_3d({{17, 65, 33}, {17, 65, 33}, {16, 16, 3}}));
}
