// few_items_find and few_items_coord of odc_tiles.h against locate_tile, over every tile of launches of
// 1 to kFewItems items.
#include <cstdio>
#include <initializer_list>
#include <random>
#include <vector>

#include "odc_tiles.h"

using namespace odc_tiles;

int main() {
  std::mt19937_64 rng(11);
  unsigned long checked = 0;
  for (uint32_t n_items = 1; n_items <= kFewItems; ++n_items)
    for (uint32_t world : {1u, 2u, 3u, 8u, 12u, 64u})
      for (uint32_t order : {kRanksInterleaved, kItemMajor, kRankOutermost})
        for (uint64_t unit : {(uint64_t)kTileBytes, (uint64_t)kTileElems / kShortTileParts}) {
          std::vector<uint64_t> sizes;
          for (uint32_t i = 0; i < n_items; ++i)  // from one unit to a few tiles, on and off their edges
            sizes.push_back(rng() % 3 ? 1 + rng() % (5 * unit) : unit * (1 + rng() % 3));
          TileTable tt;
          uint32_t next = 0;
          fill_tile_table(tt, world, n_items, &next, unit, [&](uint32_t i) { return sizes[i]; }, [](uint32_t, uint32_t) {});
          tt.order = order;
          tt.first_rank = (uint32_t)(rng() % world);
          const FewItemsTable few = few_items_table(tt);
          for (uint32_t t = 0; t < tt.n_tiles; ++t, ++checked) {
            TileCursor cur;
            TileCoord want;
            locate_tile(tt, t, cur, want);
            const FewItemsTile f = few_items_find(few, few.tiles_before, t);
            const TileCoord got = few_items_coord(few, f, few.tiles_before[f.item], (uint32_t)tiles_for(sizes[f.item], unit));
            if (got.item != want.item || got.rank != want.rank || got.chunk != want.chunk) {
              printf("%u items world %u order %u first_rank %u tile %u\n", n_items, world, order, tt.first_rank, t);
              return 1;
            }
          }
        }
  // the largest launch there is: positions and table entries up to the last sign bit
  TileTable tt;
  uint32_t next = 0;
  const uint64_t most = (kMaxTilesPerLaunch - 1) / 2;
  fill_tile_table(tt, 1, 2, &next, 1, [&](uint32_t) { return most; }, [](uint32_t, uint32_t) {});
  tt.order = kItemMajor;
  tt.first_rank = 0;
  const FewItemsTable few = few_items_table(tt);
  for (uint32_t t : {0u, (uint32_t)most - 1, (uint32_t)most, tt.n_tiles - 1}) {
    const FewItemsTile f = few_items_find(few, few.tiles_before, t);
    const TileCoord got = few_items_coord(few, f, few.tiles_before[f.item], (uint32_t)most);
    if (got.item != (t >= most) || got.rank != 0 || got.chunk != t % most) return 1;
  }
  printf("few items ok: %lu tiles\n", checked);
  return 0;
}
