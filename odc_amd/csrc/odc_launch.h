// odc_launch.h — what the host side of libodc_hip.so hands to its device side.
//
// The library is two translation units. odc_host.cpp is plain C++ (no HIP header): the C ABI,
// the symmetric arena, argument validation and launch planning. odc_kernels.hip holds the gfx950
// kernels and the few runtime calls (device queries, the one hipMalloc, the launches). They meet
// in this header: the per-launch descriptors, which travel BY VALUE in the kernel-argument
// segment, and the functions of namespace odc_device. A second implementation of odc_device that
// has no device (tests/cpu/no_device.cpp) lets the host side be built with g++ and run under
// AddressSanitizer / UBSan on bookkeeping-only and dry-run arenas.
#ifndef ODC_LAUNCH_H_
#define ODC_LAUNCH_H_

#include <stdint.h>

#include "odc_hip.h"
#include "odc_tiles.h"

namespace odc_launch {

using odc_tiles::kMaxItems;
using odc_tiles::kShortTileVecs;
using odc_tiles::kThreads;
using odc_tiles::kTileVecs;
using odc_tiles::TileTable;

// Whether a launch leaves what it reads / what it writes in the caches (plain accesses) or streams
// past them (nontemporal ones). For the gathers these are the shards and the output (OutputForm for
// the plain gather's).
struct CachePolicy {
  bool read = false;
  bool written = false;
};

// How a gather writes its output, an accumulate its accumulations or a clear its zeros: past the caches, through
// the L2 into the last-level cache, or with plain stores (store_output in odc_kernels.hip, output_form and
// those after it in odc_host.cpp).
enum OutputForm : uint32_t { kStream, kWriteThrough, kKeep };

// The same for an accumulate: "read" is the gradient, "written" the accumulations, which are read through the
// caches where they are written through or into them.
struct AccumPolicy {
  bool read = false;
  OutputForm written = kStream;
};

// How a launch is cut, and how its workgroups find their items (wants_short_tiles, table_form and tile_form in
// odc_host.cpp). kTinyTiles: kFewShortTiles by workgroups of one wavefront; kStreamTiles: short tiles of a long
// stream (stream_form there).
enum TileForm : uint32_t { kWholeTiles, kShortTiles, kFewShortTiles, kTinyTiles, kStreamTiles };

inline uint32_t tile_parts(TileForm form) { return form == kWholeTiles ? 1 : odc_tiles::kShortTileParts; }

// 16-bit gradients into fp32 accumulations are accumulated and stored in short tiles whatever the
// sizes. What bounds these streams is how reads and writes mix in HBM, and 16 workgroups of 128
// threads with 2 quads per lane in flight (98 KB of loads per CU) mix them better than 8 of 256 with
// 4 (196 KB), the more so the oftener the launch hops between segments. The decoder layer, us,
// 256 x 4 -> 128 x 2: accumulate 344 -> 341 at W = 8, 354 -> 349 at W = 16, 365 -> 352 at W = 32,
// 373 -> 352 at W = 64, 374 -> 370 at W = 128; a 525 M element embedding 863 -> 852; the store
// 206 -> 198 at W = 8, 209 -> 205 at W = 64. (128 x 1: 386, 64 x 2: 371, 64 x 4: 348 and 357 at
// W = 64, 128 x 4: 349 and 372, 256 x 1: 367, 256 x 2: 360.) fp32 gradients move the same bytes per
// lane in both streams and keep 256 x 4 (421; 128 x 2: 429); 16-bit accumulations have the shapes of
// kNarrowRmwThreads below. Where rank segments start on no line boundary neighbouring tiles share a
// line of gradient, and a short one holds a quarter of a whole one's: 1.4 % instead of 0.5 % more traffic
// over 40 uneven parameters at W = 12, which accumulate in 619 us instead of 631 (393 M elements) or in
// 259.4 instead of 257.5 (161 M, between gathers).
constexpr bool accum_streams_short(int grad_dtype, int acc_dtype) {
  return grad_dtype != ODC_DTYPE_F32 && acc_dtype == ODC_DTYPE_F32;
}

// Workgroup shape of the two gathers and of the scatter-store (the kernels that read one stream
// and write one) on whole tiles: 512 threads x 2 steps over the same 16 KiB tile as the 256 x 4 of
// the other kernels. Four such workgroups fill a CU's wave slots, which is the residency these kernels
// stream best at (measured: gathers +1.4..2.6 % over 256 x 4 with a residency cap of 4, which
// had to be enforced by claiming LDS; 256 x 4 without a cap loses 6..8 %; 1024 x 1 loses
// 20 %; short tiles lose 1 %). The read-modify-write with fp32 gradients keeps 256 x 4 (512 x 2:
// equal on long segments), and so does the clear (512 x 2: -25 % on per-parameter spans).
constexpr int kCopyThreads = 512;
constexpr int kCopyUnroll = (int)kTileVecs / kCopyThreads;  // 2 for the 16 KiB tile
constexpr int kStoreThreads = 512;
constexpr int kStoreUnroll = (int)kTileVecs / kStoreThreads;
static_assert(kCopyUnroll >= 1 && kStoreUnroll >= 1, "a tile holds at least one vector per thread");
// 16-bit gradients into 16-bit accumulations have 8-byte vectors in both streams, half a tile's bytes,
// and whole tiles take the other two shapes: the store 256 x 4 (64 KB of loads in flight per CU, as the
// gathers have; 512 x 2 has half of that), the read-modify-write 512 x 2 where its gradient is streamed
// (where the gradient is cached, up to 64 Mi elements, 256 x 4 is level or ahead). Graph-replayed
// launches, us, before -> after, then 128 x 8 for both: a decoder layer's store at W = 8 174 -> 136, 138;
// at W = 64 167 -> 140, 143; 12 uneven ranks 177 -> 141, 144; one of 525 M elements 326 -> 328, 333;
// 4 Mi 4.9 -> 4.5, 4.7; the layer's read-modify-write at W = 8 209 -> 199, 210; at W = 64 218 -> 204.5,
// 218; 525 M elements 516 -> 489, 517. (Pairs of vectors, 16 bytes per lane, in the old shapes: 213 and
// 178 for the layer at W = 8, 524 and 341 for 525 M.)
constexpr int kNarrowRmwThreads = 512;
constexpr int kNarrowRmwUnroll = (int)kTileVecs / kNarrowRmwThreads;
// Shape for short tiles: two vectors per lane, and few enough threads that a segment of a few hundred
// elements does not hold the wave slots of a CU for nothing (300 slices at W = 16, gather + accumulate:
// 31.9 us; 256 threads x 1: 40.1; 128 x 1 on eighths: 35.2; 128 x 4 on halves: 33.1; whole tiles: 46.6).
constexpr int kShortThreads = 128;
constexpr int kShortUnroll = (int)kShortTileVecs / kShortThreads;

// The same tiles where most of them are not full: one wavefront each (tile_form in odc_host.cpp).
constexpr int kTinyThreads = 64;
constexpr int kTinyUnroll = (int)kShortTileVecs / kTinyThreads;

// The workgroup sizes of the launches, as the pick_* functions of odc_kernels.hip take them.
inline uint32_t copy_threads(TileForm form) {
  return form == kWholeTiles ? kCopyThreads : form == kTinyTiles ? kTinyThreads : kShortThreads;
}
inline uint32_t publish_threads(TileForm form) { return form != kWholeTiles ? kShortThreads : kThreads; }
inline uint32_t accum_threads(int grad_dtype, int acc_dtype, bool store, AccumPolicy policy, TileForm form) {
  if (form == kTinyTiles) return kTinyThreads;
  if (form != kWholeTiles) return kShortThreads;
  if (grad_dtype != ODC_DTYPE_F32 && acc_dtype != ODC_DTYPE_F32)
    return store || policy.read ? kThreads : kNarrowRmwThreads;
  return store ? kStoreThreads : kThreads;
}

// A dispatch counts its work-items in 32 bits. Launches of more tiles than that leaves workgroups for
// (2^25 of 128 threads, 2^23 of 512) get the largest grid there is, which walks them.
constexpr uint32_t most_workgroups(uint32_t threads) { return 0xffffffffu / threads; }

// A launch carries up to kMaxItems items. One of a single item, a flat parameter on its own, goes out
// in a form without the tables: 64 to 88 bytes of arguments instead of 2.3 to 4 KB, which the host
// hands over in 2.6 us instead of 4.0 (512 bytes: 3.4), and all of it is read at once instead of
// along the item search (SingleWalk in odc_kernels.hip).
template <class D>
struct SingleLaunch {
  typedef D Desc;
  odc_tiles::TileHead tt;
  uint8_t* base;  // arena base (rank 0 region)
  uint64_t rank_stride;
  D item[1];
};

// One of 2 to kFewItems items, as the parameters of a layer are, goes out with tables of that size: 368 to
// 624 bytes of arguments (about 0.6 us less of host time than 4 KB), and the whole prefix table in one
// scalar load (ItemsWalk in odc_kernels.hip). Both short forms are for launches of one workgroup per tile.
// Long streams of up to kSomeItems have such tables too.
template <class D, uint32_t kItems>
struct ItemsLaunch {
  typedef D Desc;
  odc_tiles::ItemsTable<kItems> tt;
  uint8_t* base;  // arena base (rank 0 region)
  uint64_t rank_stride;
  D item[kItems];
};

// One record per item, read with scalar loads by the workgroup that works on the item.
struct GatherDesc {
  uint8_t* dst;
  uint64_t src_off;
  uint64_t seg_bytes;
  ODC_HD uint64_t units() const { return seg_bytes; }
};
struct GatherLaunch {
  typedef GatherDesc Desc;
  TileTable tt;
  uint8_t* base;  // arena base (rank 0 region)
  uint64_t rank_stride;
  CachePolicy policy;    // these three pick the kernel
  OutputForm output = kStream;
  TileForm form = kWholeTiles;
  GatherDesc item[kMaxItems];
};

struct CastGatherDesc {
  uint8_t* dst;         // where rank 0's converted segment goes
  uint64_t dst_stride;  // bytes from one rank's converted segment to the next rank's
  uint64_t src_off;
  uint64_t seg_elems;
  ODC_HD uint64_t units() const { return seg_elems; }
};
struct CastGatherLaunch {
  typedef CastGatherDesc Desc;
  TileTable tt;
  uint8_t* base;
  uint64_t rank_stride;
  CachePolicy policy;    // these three pick the kernel
  OutputForm output = kStream;
  TileForm form = kWholeTiles;
  CastGatherDesc item[kMaxItems];
};

struct AccumDesc {
  const uint8_t* grad;
  uint64_t grad_elems;
  uint64_t acc_off;
  uint64_t seg_elems;
  ODC_HD uint64_t units() const { return seg_elems; }
};
struct AccumLaunch {
  typedef AccumDesc Desc;
  TileTable tt;
  uint8_t* base;
  uint64_t rank_stride;
  AccumPolicy policy;    // these two pick the kernel
  TileForm form = kWholeTiles;
  AccumDesc item[kMaxItems];
};

struct ClearDesc {
  uint64_t off;
  uint64_t seg_bytes;
  ODC_HD uint64_t units() const { return seg_bytes; }
};
struct ClearLaunch {
  typedef ClearDesc Desc;
  TileTable tt;
  uint8_t* base;
  uint64_t rank_stride;
  OutputForm output = kKeep;  // picks the kernel: kKeep or kWriteThrough
  ClearDesc item[kMaxItems];
};

struct PublishDesc {
  uint8_t* out;  // may be null: divide in place only
  uint64_t acc_off;
  uint64_t seg_elems;
  ODC_HD uint64_t units() const { return seg_elems; }
};
struct PublishScale {
  float divisor;
  float reciprocal;     // exact 1 / divisor when divide == 2
  uint32_t divide;      // 0: leave the accumulation untouched, 1: divide, 2: multiply by reciprocal
};
struct PublishLaunch {  // one rank's region only: tt.world == 1
  typedef PublishDesc Desc;
  TileTable tt;
  uint8_t* base;        // of the publishing rank's region
  uint64_t rank_stride; // not used
  PublishScale scale;
  TileForm form = kWholeTiles;  // picks the kernel
  PublishDesc item[kMaxItems];
};
struct PublishSingle : SingleLaunch<PublishDesc> {
  PublishScale scale;
};
struct PublishFewItems : ItemsLaunch<PublishDesc, odc_tiles::kFewItems> {
  PublishScale scale;
};
static_assert(sizeof(SingleLaunch<ClearDesc>) == 64 && sizeof(PublishSingle) == 88, "as SingleLaunch says");
static_assert(sizeof(ItemsLaunch<ClearDesc, odc_tiles::kFewItems>) == 368 &&
                  sizeof(ItemsLaunch<AccumDesc, odc_tiles::kFewItems>) == 624 && sizeof(PublishFewItems) <= 624,
              "as ItemsLaunch says");
static_assert(sizeof(GatherLaunch) <= 4096 && sizeof(AccumLaunch) <= 4096 && sizeof(PublishLaunch) <= 4096 &&
                  sizeof(CastGatherLaunch) <= 4096 && sizeof(ClearLaunch) <= 4096,
              "launch descriptors must fit the kernel-argument segment");

}  // namespace odc_launch

// The device side. Every function returns 0 or a runtime error code that error_string() names;
// dtype arguments are odc_dtype codes.
namespace odc_device {

struct Properties {
  int n_cu;            // compute units
  int lds_per_cu;      // bytes of LDS per compute unit
  int lds_per_wg_max;  // most LDS one workgroup may claim
};

int get_current(int* device);
int set_current(int device);
int properties(int device, Properties* out);
int allocate(void** ptr, uint64_t bytes);  // on the current device
int release(void* ptr);                    // waits for the current device, then frees
bool is_out_of_memory(int code);
const char* error_string(int code);

// Which dtype pairs have a kernel: (gradient, accumulation), (shard, output), (accumulation, output).
bool has_accum(int grad_dtype, int acc_dtype);
bool has_cast_gather(int src_dtype, int dst_dtype);
bool has_publish(int acc_dtype, int out_dtype);

// One launch of `grid` workgroups on `stream`, each claiming `lds_bytes` of LDS it never touches
// (a residency cap; 0 = none). The workgroup size belongs to the kernel.
int launch_gather(const odc_launch::GatherLaunch& launch, uint32_t grid, uint32_t lds_bytes, void* stream);
int launch_cast_gather(int src_dtype, int dst_dtype, const odc_launch::CastGatherLaunch& launch, uint32_t grid,
                       uint32_t lds_bytes, void* stream);
int launch_accum(int grad_dtype, int acc_dtype, bool store, const odc_launch::AccumLaunch& launch, uint32_t grid,
                 uint32_t lds_bytes, void* stream);
int launch_clear(const odc_launch::ClearLaunch& launch, uint32_t grid, void* stream);
int launch_publish(int acc_dtype, int out_dtype, const odc_launch::PublishLaunch& launch, uint32_t grid,
                   uint32_t lds_bytes, void* stream);

}  // namespace odc_device

#endif  // ODC_LAUNCH_H_
