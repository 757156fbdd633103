// The item tables of odc_tiles.h (items_table, items_position, count_before, items_coord) against
// locate_tile, over every tile of launches of as many items as they hold and fewer.
#include <cstdio>
#include <initializer_list>
#include <random>
#include <vector>

#include "odc_tiles.h"

using namespace odc_tiles;

// As the kernels do it: the block of the table, then the item in it.
template <uint32_t kItems>
static TileCoord find(const ItemsTable<kItems>& table, uint32_t t, const std::vector<uint64_t>& sizes, uint64_t unit) {
  ItemsTile f = items_position(table, t);
  if (kItems != kFewItems) f.item = kFewItems * count_before<kItems / kFewItems>(table.block_before, f.position);
  f.item += count_before<kFewItems>(table.tiles_before + f.item, f.position);
  return items_coord(table, f, table.tiles_before[f.item], (uint32_t)tiles_for(sizes.at(f.item), unit));
}

static unsigned long checked = 0;

template <uint32_t kItems>
static bool check(uint32_t n_items, uint32_t world, uint32_t order, uint64_t unit, std::mt19937_64& rng) {
  std::vector<uint64_t> sizes;
  for (uint32_t i = 0; i < n_items; ++i)  // from one unit to a few tiles, on and off their edges
    sizes.push_back(rng() % 3 ? 1 + rng() % (5 * unit) : unit * (1 + rng() % 3));
  TileTable tt;
  uint32_t next = 0;
  fill_tile_table(tt, world, n_items, &next, unit, [&](uint32_t i) { return sizes[i]; }, [](uint32_t, uint32_t) {});
  tt.order = order;
  tt.first_rank = (uint32_t)(rng() % world);
  const ItemsTable<kItems> table = items_table<kItems>(tt);
  for (uint32_t t = 0; t < tt.n_tiles; ++t, ++checked) {
    TileCursor cur;
    TileCoord want;
    locate_tile(tt, t, cur, want);
    const TileCoord got = find(table, t, sizes, unit);
    if (got.item != want.item || got.rank != want.rank || got.chunk != want.chunk) {
      printf("%u of %u items world %u order %u first_rank %u tile %u\n", n_items, kItems, world, order, tt.first_rank, t);
      return false;
    }
  }
  return true;
}

int main() {
  std::mt19937_64 rng(11);
  for (uint32_t world : {1u, 2u, 3u, 8u, 12u, 64u})
    for (uint32_t order : {kRanksInterleaved, kItemMajor, kRankOutermost})
      for (uint64_t unit : {(uint64_t)kTileBytes, (uint64_t)kTileElems / kShortTileParts}) {
        for (uint32_t n_items = 1; n_items <= kFewItems; ++n_items)
          if (!check<kFewItems>(n_items, world, order, unit, rng)) return 1;
        for (uint32_t n_items : {1u, 15u, 16u, 17u, 31u, 32u, 33u, 48u, 49u, 63u, 64u})
          if (!check<kSomeItems>(n_items, world, order, unit, rng)) return 1;
      }
  // the largest launch there is: positions and table entries up to the last sign bit
  TileTable tt;
  uint32_t next = 0;
  const uint64_t most = (kMaxTilesPerLaunch - 1) / 2;
  fill_tile_table(tt, 1, 2, &next, 1, [&](uint32_t) { return most; }, [](uint32_t, uint32_t) {});
  tt.order = kItemMajor;
  tt.first_rank = 0;
  for (uint32_t t : {0u, (uint32_t)most - 1, (uint32_t)most, tt.n_tiles - 1}) {
    const TileCoord few = find(items_table<kFewItems>(tt), t, {most, most}, 1), some = find(items_table<kSomeItems>(tt), t, {most, most}, 1);
    for (const TileCoord& got : {few, some})
      if (got.item != (t >= most) || got.rank != 0 || got.chunk != t % most) return 1;
  }
  printf("few items ok: %lu tiles\n", checked);
  return 0;
}
