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
using odc_tiles::TileTable;

// Whether a launch leaves what it reads / what it writes in the caches (plain accesses) or streams
// past them (nontemporal ones). For the accumulate "read" is the gradient and "written" the
// accumulation, read and written; for the gathers they are the shards and the output.
struct CachePolicy {
  bool read = false;
  bool written = false;
};

// How a launch is cut, and how its workgroups find their items (wants_short_tiles and tile_form in
// odc_host.cpp).
enum TileForm : uint32_t { kWholeTiles, kShortTiles, kFewShortTiles };

// 16-bit gradients into fp32 accumulations are accumulated and stored in short tiles whatever the
// sizes. What bounds these streams is how reads and writes mix in HBM, and 16 workgroups of 128
// threads with 2 quads per lane in flight (98 KB of loads per CU) mix them better than 8 of 256 with
// 4 (196 KB), the more so the oftener the launch hops between segments. The decoder layer, us,
// 256 x 4 -> 128 x 2: accumulate 344 -> 341 at W = 8, 354 -> 349 at W = 16, 365 -> 352 at W = 32,
// 373 -> 352 at W = 64, 374 -> 370 at W = 128; a 525 M element embedding 863 -> 852; the store
// 206 -> 198 at W = 8, 209 -> 205 at W = 64. (128 x 1: 386, 64 x 2: 371, 64 x 4: 348 and 357 at
// W = 64, 128 x 4: 349 and 372, 256 x 1: 367, 256 x 2: 360.) fp32 gradients move the same bytes per
// lane in both streams and keep 256 x 4 (421; 128 x 2: 429), and so do 16-bit accumulations.
constexpr bool accum_streams_short(int grad_dtype, int acc_dtype) {
  return grad_dtype != ODC_DTYPE_F32 && acc_dtype == ODC_DTYPE_F32;
}

// A launch carries up to kMaxItems items. One of a single item, a flat parameter on its own, goes out
// in a form without the tables: 56 .. 72 bytes of arguments instead of 3 to 4 KB, which the host
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

// One record per item, read with scalar loads by the workgroup that works on the item.
struct GatherDesc {
  uint8_t* dst;
  uint64_t src_off;
  uint64_t seg_bytes;
};
struct GatherLaunch {
  typedef GatherDesc Desc;
  TileTable tt;
  uint8_t* base;  // arena base (rank 0 region)
  uint64_t rank_stride;
  CachePolicy policy;    // these two pick the kernel
  TileForm form = kWholeTiles;
  GatherDesc item[kMaxItems];
};

struct CastGatherDesc {
  uint8_t* dst;         // where rank 0's converted segment goes
  uint64_t dst_stride;  // bytes from one rank's converted segment to the next rank's
  uint64_t src_off;
  uint64_t seg_elems;
};
struct CastGatherLaunch {
  typedef CastGatherDesc Desc;
  TileTable tt;
  uint8_t* base;
  uint64_t rank_stride;
  CachePolicy policy;    // these two pick the kernel
  TileForm form = kWholeTiles;
  CastGatherDesc item[kMaxItems];
};

struct AccumDesc {
  const uint8_t* grad;
  uint64_t grad_elems;
  uint64_t acc_off;
  uint64_t seg_elems;
};
struct AccumLaunch {
  typedef AccumDesc Desc;
  TileTable tt;
  uint8_t* base;
  uint64_t rank_stride;
  CachePolicy policy;    // these two pick the kernel
  TileForm form = kWholeTiles;
  AccumDesc item[kMaxItems];
};

struct ClearDesc {
  uint64_t off;
  uint64_t seg_bytes;
};
struct ClearLaunch {
  typedef ClearDesc Desc;
  TileTable tt;
  uint8_t* base;
  uint64_t rank_stride;
  ClearDesc item[kMaxItems];
};

struct PublishDesc {
  uint8_t* out;  // may be null: divide in place only
  uint64_t acc_off;
  uint64_t seg_elems;
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
