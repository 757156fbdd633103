// odc_tiles.h — how a launch of libodc_hip.so is cut into tiles, and how a tile finds its work.
//
// Shared by the kernels (device), by the launch code (host) and by the CPU geometry test, which
// compiles this header with g++ alone and checks, by brute force, that every unit of every rank
// segment is owned by exactly one tile role and that no role reaches outside its segment.
//
// Vocabulary. A launch carries up to kMaxItems ITEMS (one shard of one tensor). An item has one
// SEGMENT per rank: `n` units (bytes or elements) at the same symmetric offset of every rank
// region. A segment is cut into TILES of kTileVecs vectors (or of kShortTileVecs, a launch of short
// ones); a workgroup of 64, 128, 256 or 512 threads does one tile at a time.
#ifndef ODC_TILES_H_
#define ODC_TILES_H_

#include <stdint.h>

#if defined(__HIPCC__)
#define ODC_HD __host__ __device__ __forceinline__
#else
#define ODC_HD inline
#endif

#ifndef ODC_TILE_THREADS
#define ODC_TILE_THREADS 256  // 4 wavefronts of 64 lanes
#endif
#ifndef ODC_TILE_UNROLL
#define ODC_TILE_UNROLL 4  // independent vector accesses per lane per stream before the stores
#endif
#ifndef ODC_BODY_ALIGN
#define ODC_BODY_ALIGN 128  // bytes: alignment of a segment's vector body on the written side
#endif
#ifndef ODC_MAX_ITEMS_PER_LAUNCH
#define ODC_MAX_ITEMS_PER_LAUNCH 112
#endif

namespace odc_tiles {

constexpr int kThreads = ODC_TILE_THREADS;
constexpr int kUnroll = ODC_TILE_UNROLL;
constexpr int kMaxItems = ODC_MAX_ITEMS_PER_LAUNCH;
constexpr uint32_t kTileVecs = kThreads * kUnroll;  // vectors per tile
constexpr uint32_t kTileBytes = kTileVecs * 16;     // gather / clear: 16 KiB of destination
constexpr uint32_t kTileElems = kTileVecs * 4;      // accumulate / cast / publish: 4096 elements
constexpr uint64_t kMaxTilesPerLaunch = 1ull << 31;
// Launches of short segments are cut finer: into quarters of a tile (wants_short_tiles and its
// neighbours in odc_host.cpp).
constexpr uint32_t kShortTileParts = 4;
constexpr uint32_t kShortTileVecs = kTileVecs / kShortTileParts;

// Tile order of a launch (TileTable::order).
//   kRanksInterleaved : item by item; within an item tile c of rank 0, of rank 1, ..., then c+1
//   kItemMajor        : item by item; within an item all of rank 0's tiles, then rank 1's
//   kRankOutermost    : rank by rank; within a rank item by item
enum TileOrder : uint32_t { kRanksInterleaved = 0, kItemMajor = 1, kRankOutermost = 2 };

// What a launch of any number of items says about its tiles; all there is to say about one item.
struct TileHead {
  uint32_t world;
  uint32_t n_items;
  uint32_t n_tiles;         // world * tiles_per_rank
  uint32_t order;           // TileOrder
  uint32_t first_rank;      // rotation of the rank walk (never changes the result)
  uint32_t tiles_per_rank;  // seg_prefix[n_items]
  uint32_t resident_below = 0;  // see is_resident
};

// Travels by value in the kernel-argument segment. seg_prefix[i] is the number of tiles that
// the items before item i have in ONE rank segment each, so item i has
// seg_prefix[i+1] - seg_prefix[i] tiles per rank segment and world times that in the launch.
// Entries past n_items hold tiles_per_rank, so a search never lands on them.
struct TileTable : TileHead {
  uint32_t seg_prefix[kMaxItems + 1];
};

struct TileCoord {
  uint32_t item, rank, chunk;  // chunk: tile index within the rank segment
};

// Largest i with seg_prefix[i] <= x, for x < tiles_per_rank (seg_prefix[0] is 0 and the entries
// are strictly increasing over the real items: empty items are never listed).
ODC_HD uint32_t find_item(const TileTable& tt, uint32_t x) {
  uint32_t lo = 0, hi = tt.n_items;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (tt.seg_prefix[mid] <= x) lo = mid; else hi = mid;
  }
  return lo;
}

// A cursor remembers the run of consecutive tile indices [lo, hi) that share the item (and, in
// rank-outermost order, the rank) of the last tile located, so a workgroup that walks many tiles
// with a grid-stride loop searches only when it leaves that run. Use:
//     if (!cursor_holds(cur, t)) {
//       cursor_seek(tt, t, cur);            // the search: sets cur.item
//       desc = launch.item[cur.item];       // the caller's per-item record ...
//       cursor_enter(tt, cur);              // ... and the run's bounds: independent loads
//     }
//     TileCoord c = cursor_coord(tt, cur, t);
struct TileCursor {
  uint32_t lo = 1, hi = 0;  // empty
  uint32_t item = 0;
  uint32_t rank = 0;  // kRankOutermost only: the (unrotated) rank of the run
  uint32_t tps = 1;   // tiles per rank segment of the item
};

ODC_HD bool cursor_holds(const TileCursor& cur, uint32_t t) { return t >= cur.lo && t < cur.hi; }

// The position of tile t along the items of one rank: seg_prefix[item] <= position < seg_prefix[item + 1].
ODC_HD uint32_t cursor_position(const TileHead& tt, uint32_t t, TileCursor& cur) {
  if (tt.order == kRankOutermost) {
    cur.rank = t / tt.tiles_per_rank;
    return t - cur.rank * tt.tiles_per_rank;
  }
  // item i owns tiles [seg_prefix[i] * world, seg_prefix[i+1] * world)
  cur.rank = 0;
  return t / tt.world;
}

ODC_HD void cursor_seek(const TileTable& tt, uint32_t t, TileCursor& cur) {
  cur.item = find_item(tt, cursor_position(tt, t, cur));
}

// The run's bounds, from the two entries of seg_prefix around cur.item.
ODC_HD void cursor_bounds(const TileHead& tt, uint32_t first, uint32_t next, TileCursor& cur) {
  cur.tps = next - first;
  if (tt.order == kRankOutermost) {
    cur.lo = cur.rank * tt.tiles_per_rank + first;
    cur.hi = cur.lo + cur.tps;
  } else {
    cur.lo = first * tt.world;
    cur.hi = next * tt.world;
  }
}

ODC_HD void cursor_enter(const TileTable& tt, TileCursor& cur) {
  cursor_bounds(tt, tt.seg_prefix[cur.item], tt.seg_prefix[cur.item + 1], cur);
}

// Tile t (inside the cursor's run) -> (item, rank, chunk). Everything here is wave-uniform.
ODC_HD TileCoord cursor_coord(const TileHead& tt, const TileCursor& cur, uint32_t t) {
  TileCoord c;
  const uint32_t lt = t - cur.lo;
  c.item = cur.item;
  if (tt.order == kRankOutermost) {
    c.rank = cur.rank;
    c.chunk = lt;
  } else if (tt.order == kItemMajor) {
    c.rank = lt / cur.tps;
    c.chunk = lt - c.rank * cur.tps;
  } else {
    c.chunk = lt / tt.world;
    c.rank = lt - c.chunk * tt.world;
  }
  c.rank += tt.first_rank;
  if (c.rank >= tt.world) c.rank -= tt.world;
  return c;
}

// The three steps in one call. Returns true when the cursor moved to another run.
ODC_HD bool locate_tile(const TileTable& tt, uint32_t t, TileCursor& cur, TileCoord& c) {
  const bool moved = !cursor_holds(cur, t);
  if (moved) {
    cursor_seek(tt, t, cur);
    cursor_enter(tt, cur);
  }
  c = cursor_coord(tt, cur, t);
  return moved;
}

// The same for the tiles of a launch of one item, whose two rank by rank orders are one.
ODC_HD TileCoord single_item_coord(const TileHead& tt, uint32_t t) {
  TileCoord c;
  c.item = 0;
  if (tt.order == kRanksInterleaved) {
    c.chunk = t / tt.world;
    c.rank = t - c.chunk * tt.world;
  } else {
    c.rank = t / tt.tiles_per_rank;
    c.chunk = t - c.rank * tt.tiles_per_rank;
  }
  c.rank += tt.first_rank;
  if (c.rank >= tt.world) c.rank -= tt.world;
  return c;
}

// A launch of up to kItems items with one workgroup per tile: the table is read in blocks of kFewItems
// entries, one scalar load each, and holds what the tile order needs, so that no tile divides twice: the tiles
// before item i in one rank segment each where ranks are outermost, in the whole launch where items
// are. Entries past the last item hold the total.
constexpr uint32_t kFewItems = 16;
constexpr uint32_t kSomeItems = 64;
template <uint32_t kItems>
struct ItemsTable : TileHead {
  uint32_t block_before[kItems / kFewItems];  // tiles_before of each block's first item
  uint32_t tiles_before[kItems];
};

template <uint32_t kItems>
inline ItemsTable<kItems> items_table(const TileTable& tt) {
  static_assert(kItems % kFewItems == 0 && kItems <= (uint32_t)kMaxItems, "whole blocks of the full table");
  ItemsTable<kItems> t;
  static_cast<TileHead&>(t) = tt;
  for (uint32_t i = 0; i < kItems; ++i) {
    t.tiles_before[i] = tt.seg_prefix[i] * (tt.order == kRankOutermost ? 1u : tt.world);
    if (i % kFewItems == 0) t.block_before[i / kFewItems] = t.tiles_before[i];
  }
  return t;
}

// A tile of such a launch: its item, its rank (rank outermost only) and its position, among all the launch's
// tiles or the rank's.
struct ItemsTile {
  uint32_t item, rank, position;
};

// Tile t's rank and position.
ODC_HD ItemsTile items_position(const TileHead& tt, uint32_t t) {
  ItemsTile f = {0, 0, t};
  if (tt.order == kRankOutermost) {
    f.rank = t / tt.tiles_per_rank;
    f.position = t - f.rank * tt.tiles_per_rank;
  }
  return f;
}

// The number of before[1] .. before[n - 1] that do not lie behind the position, for ascending values less than
// 2^31: counted by sign bits. before: in any form that can be indexed (the kernels hold it in scalar registers).
template <uint32_t n, class Before>
ODC_HD uint32_t count_before(const Before& before, uint32_t position) {
  static_assert(kMaxTilesPerLaunch <= 1ull << 31, "sign bits");
  uint32_t found = n - 1;
#pragma unroll
  for (uint32_t i = 1; i < n; ++i) found -= (position - before[i]) >> 31;
  return found;
}

// first: tiles_before of the item; per_rank: the item's tiles in one rank segment
ODC_HD TileCoord items_coord(const TileHead& tt, ItemsTile f, uint32_t first, uint32_t per_rank) {
  TileCoord c;
  c.item = f.item;
  f.position -= first;
  if (tt.order == kRankOutermost) {
    c.rank = f.rank;
    c.chunk = f.position;
  } else if (tt.order == kItemMajor) {
    c.rank = f.position / per_rank;
    c.chunk = f.position - c.rank * per_rank;
  } else {
    c.chunk = f.position / tt.world;
    c.rank = f.position - c.chunk * tt.world;
  }
  c.rank += tt.first_rank;
  if (c.rank >= tt.world) c.rank -= tt.world;
  return c;
}

// Shape of one rank segment of `n` units whose WRITTEN side starts at address D:
//     head  : the units before the first 128-byte line boundary of D (at most 127 bytes),
//     body  : nvec whole vectors, written with aligned 128-bit (64-bit for 16-bit outputs) stores,
//     tail  : what is left after the last whole vector.
// Tile c owns body vectors [c*kTileVecs, (c+1)*kTileVecs); tile 0 also does the head, and the
// tile holding the last body vector (tile 0 when there is none) the tail. The READ side takes
// whatever misalignment that leaves it with: gfx950 global loads accept any address.
struct SegShape {
  uint32_t head;  // units before the first line boundary of the written side (clipped to the segment)
  uint32_t tail;  // units after the last whole vector
  uint64_t nvec;  // whole vectors
  uint64_t last;  // tile that owns the tail
};

// unit_bytes: size of one unit on the written side; vec_units: units per vector; kVecs: vectors per
// tile of the launch
template <uint32_t kVecs = kTileVecs>
ODC_HD SegShape seg_shape(uintptr_t written_addr, uint64_t n, uint32_t unit_bytes, uint32_t vec_units) {
  // The body starts on a 128 B line of the written side, not merely on a vector boundary: a
  // wavefront's 64 vector stores then cover whole lines, none shared with the next wavefront.
  // (The head is at most kLine - 1 bytes. In bytes that can be more units than a workgroup of one wavefront has
  // lanes; each kernel asserts what it takes.)
  constexpr uint32_t kLine = ODC_BODY_ALIGN;
  static_assert(kLine >= 16, "whole vectors");
  SegShape g;
  uint64_t head = ((kLine - (uint32_t)(written_addr & (kLine - 1))) & (kLine - 1)) / unit_bytes;
  if (head > n) head = n;
  g.head = (uint32_t)head;
  g.nvec = (n - head) / vec_units;
  g.tail = (uint32_t)((n - head) - g.nvec * vec_units);
  g.last = g.nvec ? (g.nvec - 1) / kVecs : 0;
  return g;
}

// Number of tiles of a segment of n units when a tile is tile_units units. (Upper bound of what
// the shape needs: a head shifts the body by less than one vector line, never past the count.)
ODC_HD uint64_t tiles_for(uint64_t n, uint64_t tile_units) { return (n + tile_units - 1) / tile_units; }

// What tile `chunk` of a segment does.
struct TileWork {
  uint64_t v0;     // first body vector of the tile
  uint32_t nv;     // body vectors of the tile (0 .. kTileVecs)
  bool head, tail; // also does the segment's head / tail
};

template <uint32_t kVecs = kTileVecs>
ODC_HD TileWork tile_work(uint32_t chunk, const SegShape& g) {
  TileWork w;
  w.v0 = (uint64_t)chunk * kVecs;
  w.nv = w.v0 >= g.nvec ? 0u : (g.nvec - w.v0 >= kVecs ? kVecs : (uint32_t)(g.nvec - w.v0));
  w.head = chunk == 0 && g.head != 0;
  w.tail = chunk == g.last && g.tail != 0;
  return w;
}

// A tile is a whole run when all its vectors exist: the unrolled, unguarded loop.
template <uint32_t kVecs = kTileVecs>
ODC_HD bool is_whole(const TileWork& w) { return w.nv == kVecs; }
// True when the tile has anything else to do: a partial run, the head or the tail.
template <uint32_t kVecs = kTileVecs>
ODC_HD bool has_edges(const TileWork& w) { return (w.nv != 0 && w.nv != kVecs) || w.head || w.tail; }

// Whether the tile at this address of symmetric memory belongs to the part that stays in the last-level cache
// (resident_below in odc_host.cpp): its 16 KiB granule's place in a sequence that is spread evenly over
// [0, 2^32) lies below the line. A function of the address alone, so that launches of different kinds agree,
// spread so that every stretch of memory has its share; a lower line keeps a part of what a higher one does.
// The agreement is for speed only, and not complete. Asked is the address of a whole tile's first vector: where
// tiles do not start on granules (allocations of less than one, ragged heads) a whole tile and the four short
// ones of the same bytes can differ in the granule that they share with a neighbour. Left out are partial tiles,
// converting gathers, publishes, accumulates and stores of cached gradients, clears below their line, and the
// launches that read the whole table of their many items (FewTilesWalk).
ODC_HD bool is_resident(uintptr_t address, uint32_t below) {
  return (uint32_t)(address >> 14) * 0x9E3779B1u < below;
}

// Cuts items [*next, n_items) into one launch: at most kMaxItems non-empty items and fewer than
// kMaxTilesPerLaunch tiles. units(i) is item i's per-rank size in tile units (0 = skip);
// take(slot, i) copies item i's descriptor into slot `slot` of the launch. Returns the number of
// items taken (0 when only empty items were left), or -1 - i when item i alone is too large for
// one launch.
// (tile_units: a number, or an integral constant, which makes the division a shift)
template <class TileUnits, class Units, class Take>
inline int fill_tile_table(TileTable& tt, uint32_t world, uint32_t n_items, uint32_t* next,
                           TileUnits tile_units, Units units, Take take) {
  uint32_t n = 0;
  uint64_t tiles = 0, per_rank = 0;
  uint32_t i = *next;
  for (; i < n_items && n < (uint32_t)kMaxItems; ++i) {
    const uint64_t sz = units(i);
    if (sz == 0) continue;
    const uint64_t tps = tiles_for(sz, tile_units);
    if (tps * world >= kMaxTilesPerLaunch) return -1 - (int)i;
    if (tiles + tps * world >= kMaxTilesPerLaunch) break;
    tt.seg_prefix[n] = (uint32_t)per_rank;
    take(n, i);
    tiles += tps * world;
    per_rank += tps;
    ++n;
  }
  *next = i;
  for (uint32_t k = n; k <= (uint32_t)kMaxItems; ++k) tt.seg_prefix[k] = (uint32_t)per_rank;
  tt.world = world;
  tt.n_items = n;
  tt.n_tiles = (uint32_t)tiles;
  tt.tiles_per_rank = (uint32_t)per_rank;
  return (int)n;
}

}  // namespace odc_tiles

#endif  // ODC_TILES_H_
