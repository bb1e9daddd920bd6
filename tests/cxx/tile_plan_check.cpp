// Every tile has exactly one workgroup and round, for any number of resident workgroups and of tiles.
#include <cstdio>
#include <vector>

#include "tile_plan.hpp"

int main()
{
    for (size_t resident = 1; resident <= 3 * 304; resident++)
        for (size_t tiles : {1ul, 7ul, 8ul, 9ul, 500ul, 1000ul, 1816ul}) {
            const unsigned grid = rppa::plan_grid(resident, tiles);
            std::vector<int> seen(tiles, 0);
            if (grid > 8 && (grid > resident || grid >= tiles + 8)) return std::printf("grid %u of %zu, %zu tiles\n", grid, resident, tiles), 1;
            for (unsigned round = 0; static_cast<size_t>(round) * grid < tiles; round++)
                for (unsigned block = 0; block < grid; block++) {
                    const unsigned t = rppa::plan_tile(round, block, grid);
                    if (t < tiles) seen[t]++;
                }
            for (size_t t = 0; t < tiles; t++)
                if (seen[t] != 1) return std::printf("%zu resident, %zu tiles: tile %zu taken %d times\n", resident, tiles, t, seen[t]), 1;
        }
    std::puts("every tile once");
    return 0;
}
