// single_item_coord of odc_tiles.h against locate_tile, over every tile of launches of one item.
#include <cstdio>
#include <initializer_list>

#include "odc_tiles.h"

using namespace odc_tiles;

int main() {
  const uint32_t worlds[] = {1, 2, 3, 8, 12, 64}, tiles[] = {1, 2, 7, 64, 129};
  unsigned long checked = 0;
  for (uint32_t world : worlds)
    for (uint32_t per_rank : tiles)
      for (uint32_t order : {kRanksInterleaved, kItemMajor, kRankOutermost})
        for (uint32_t first_rank = 0; first_rank < world; ++first_rank) {
          TileTable tt;
          uint32_t next = 0;
          fill_tile_table(tt, world, 1, &next, kTileBytes, [&](uint32_t) { return (uint64_t)per_rank * kTileBytes; },
                          [](uint32_t, uint32_t) {});
          tt.order = order;
          tt.first_rank = first_rank;
          for (uint32_t t = 0; t < tt.n_tiles; ++t, ++checked) {
            TileCursor cur;
            TileCoord want;
            locate_tile(tt, t, cur, want);
            const TileCoord got = single_item_coord(tt, t);
            if (got.item != want.item || got.rank != want.rank || got.chunk != want.chunk) {
              printf("world %u tiles %u order %u first_rank %u tile %u\n", world, per_rank, order, first_rank, t);
              return 1;
            }
          }
        }
  printf("single items ok: %lu tiles\n", checked);
  return 0;
}
