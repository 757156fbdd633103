// CPU check of the short tiles of odc_amd/csrc/odc_tiles.h: every unit of a segment is owned by
// exactly one role of exactly one tile, when the table is filled in short-tile units and the roles
// are those of kShortTileVecs vectors per tile. Built by tests/test_short_tiles.py with g++.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "odc_tiles.h"

using namespace odc_tiles;

static void require(bool ok, const char* what, uint64_t n, uint64_t address) {
  if (ok) return;
  std::printf("FAILED: %s (n %llu, address %llu)\n", what, (unsigned long long)n, (unsigned long long)address);
  std::exit(1);
}

static void check(uint64_t n, uint64_t address, uint32_t unit_bytes, uint32_t vec_units) {
  TileTable tt;
  uint32_t next = 0;
  const int items = fill_tile_table(tt, 1, 1, &next, (uint64_t)kShortTileVecs * vec_units, [&](uint32_t) { return n; },
                                    [](uint32_t, uint32_t) {});
  require(items == 1, "one item", n, address);
  const SegShape g = seg_shape<kShortTileVecs>((uintptr_t)address, n, unit_bytes, vec_units);
  std::vector<uint8_t> seen(n, 0);
  for (uint32_t t = 0; t < tt.n_tiles; ++t) {
    const TileWork w = tile_work<kShortTileVecs>(t, g);
    require(w.nv <= kShortTileVecs && is_whole<kShortTileVecs>(w) == (w.nv == kShortTileVecs), "whole", n, address);
    require(has_edges<kShortTileVecs>(w) == ((w.nv && w.nv != kShortTileVecs) || w.head || w.tail), "edges", n, address);
    if (w.head) for (uint64_t k = 0; k < g.head; ++k) seen.at(k)++;
    for (uint64_t k = 0; k < (uint64_t)w.nv * vec_units; ++k) seen.at(g.head + w.v0 * vec_units + k)++;
    if (w.tail) for (uint64_t k = 0; k < g.tail; ++k) seen.at(g.head + g.nvec * vec_units + k)++;
    require(w.nv == 0 || (address + (g.head + w.v0 * vec_units) * unit_bytes) % (vec_units * unit_bytes) == 0, "alignment", n, address);
  }
  for (uint64_t k = 0; k < n; ++k) require(seen[k] == 1, "owned once", n, address);
}

int main() {
  static const struct { uint32_t unit_bytes, vec_units; } kinds[] = {{1, 16}, {4, 4}, {2, 4}};
  long checks = 0;
  for (const auto& kind : kinds) {
    const uint64_t tile = (uint64_t)kShortTileVecs * kind.vec_units;
    for (uint64_t base : {uint64_t(1), uint64_t(kind.vec_units), tile - 1, tile, tile + 1, 3 * tile - 1, 4 * tile, 4 * tile + 5})
      for (uint64_t extra = 0; extra < 40; ++extra)
        for (uint64_t address = 0; address < 256; address += kind.unit_bytes, ++checks)
          check(base + extra * (extra & 1 ? 1 : 37), 4096 + address, kind.unit_bytes, kind.vec_units);
  }
  std::printf("short tiles ok: %ld segments\n", checks);
  return 0;
}
