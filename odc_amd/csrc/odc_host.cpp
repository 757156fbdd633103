// odc_host.cpp — the host side of libodc_hip.so: the C ABI of include/odc_hip.h, the symmetric
// arena (one device allocation, W rank regions, one offset valid in all), argument validation and
// launch planning. Plain C++: everything that needs the HIP runtime or a kernel is behind
// namespace odc_device (odc_launch.h), implemented for gfx950 in odc_kernels.hip. Built with g++
// against an odc_device that has no device, this file runs under AddressSanitizer and UBSan on
// bookkeeping-only and dry-run arenas.
//
// Launch model: the work of one launch is cut into tiles of 1024 vectors (16 KiB, odc_tiles.h), or of
// 256 (scatter_in_short_tiles, wants_short_tiles, publish_in_short_tiles, stream_form);
// per-item descriptors (<= ODC_MAX_ITEMS_PER_LAUNCH) travel BY VALUE in the kernel argument
// segment, so a call needs no device-side work list, no host->device copy and no allocation;
// longer item lists are split over several launches.

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "odc_hip.h"
#include "odc_launch.h"
#include "odc_tiles.h"

namespace {

// ------------------------------------------------------------------------------------------------
// errors
// ------------------------------------------------------------------------------------------------
thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

#define ODC_DEVICE_TRY(expr)                                                                   \
  do {                                                                                         \
    const int e_ = (expr);                                                                     \
    if (e_ != 0)                                                                               \
      return fail(ODC_ERR_HIP, "%s failed: %s (%s:%d)", #expr, odc_device::error_string(e_),   \
                  __FILE__, __LINE__);                                                         \
  } while (0)

// ------------------------------------------------------------------------------------------------
// options
// ------------------------------------------------------------------------------------------------
struct Options {
  // measured on MI355X over a Llama-3-8B layer: every kernel peaks with one workgroup per tile
  // and no residency cap
  int64_t gather_blocks_per_cu = 0;
  int64_t gather_resident_cap = 0;  // 512-thread workgroups: 4 per CU without a cap
  int64_t cast_resident_cap = 0;
  int64_t accum_resident_cap = 0;
  int64_t accum_blocks_per_cu = -1;  // -1: by segment length (see scatter_launch)
  int64_t accum_short_segment_tiles = 256;   // segments averaging fewer tiles: rank-outermost tile order
  int64_t accum_persistent_below_tiles = 0;  // segments averaging fewer tiles: persistent launch shape (0: never)
  int64_t accum_small_items_last = 1;  // scatter launches: items of less than one tile per rank go last
  int64_t store_blocks_per_cu = 0;  // the scatter-store (no read of the accumulation)
  int64_t store_resident_cap = 0;
  int64_t clear_blocks_per_cu = 0;
  int64_t publish_blocks_per_cu = 0;
  int64_t publish_resident_cap = 0;
  int64_t rank_major = 1;        // gather: 0 = ranks interleaved, 1 = item-major, 2 = rank outermost
  int64_t accum_tile_order = 3;  // the same for scatter-accumulate / store; 3 = by segment length
  int64_t rank_stagger_bytes = 0;
  int64_t rank_stride_align = 16384;  // rank regions start on multiples of this (read when an arena is created)
  int64_t alloc_align = 16384;        // so do symmetric allocations at least this large
  int64_t cached_arena_bytes = 192ll << 20;   // these and the next two: see cache_policy
  int64_t cached_output_bytes = 64ll << 20;
  int64_t plain_output_bytes = 3ll << 20;    // see output_form
  int64_t cached_gradient_bytes = 128ll << 20;
  int64_t resident_accumulation_bytes = 320ll << 20;  // these and the next two: see resident_below
  int64_t resident_shard_bytes = 80ll << 20;
  int64_t resident_above = 640ll << 20;
  int64_t resident_clear_bytes = 48ll << 20;
  int64_t plain_accumulation_bytes = 3ll << 20;  // see accumulation_form
  int64_t through_store_bytes = 44ll << 20;  // see store_output_form
  int64_t through_clear_bytes = 256ll << 20;  // see clear_form
  int64_t stream_bytes = 8ll << 20;  // see stream_form
  int64_t cast_output_bytes = 32ll << 20;  // see cast_output_form
  int64_t short_tiles_below = 32;             // see wants_short_tiles
  int64_t few_tiles = 32768;                  // see table_form
  int64_t tiny_tiles_from = 2048;             // see tile_form
};
Options g_opt;
std::mutex g_opt_mu;

int64_t* option_slot(const char* name) {
  if (!name) return nullptr;
  if (!strcmp(name, "gather_blocks_per_cu")) return &g_opt.gather_blocks_per_cu;
  if (!strcmp(name, "accum_blocks_per_cu")) return &g_opt.accum_blocks_per_cu;
  if (!strcmp(name, "accum_short_segment_tiles")) return &g_opt.accum_short_segment_tiles;
  if (!strcmp(name, "accum_persistent_below_tiles")) return &g_opt.accum_persistent_below_tiles;
  if (!strcmp(name, "accum_small_items_last")) return &g_opt.accum_small_items_last;
  if (!strcmp(name, "clear_blocks_per_cu")) return &g_opt.clear_blocks_per_cu;
  if (!strcmp(name, "publish_blocks_per_cu")) return &g_opt.publish_blocks_per_cu;
  if (!strcmp(name, "rank_major")) return &g_opt.rank_major;
  if (!strcmp(name, "accum_tile_order")) return &g_opt.accum_tile_order;
  if (!strcmp(name, "rank_stagger_bytes")) return &g_opt.rank_stagger_bytes;
  if (!strcmp(name, "rank_stride_align")) return &g_opt.rank_stride_align;
  if (!strcmp(name, "alloc_align")) return &g_opt.alloc_align;
  if (!strcmp(name, "gather_resident_cap")) return &g_opt.gather_resident_cap;
  if (!strcmp(name, "cast_resident_cap")) return &g_opt.cast_resident_cap;
  if (!strcmp(name, "accum_resident_cap")) return &g_opt.accum_resident_cap;
  if (!strcmp(name, "store_blocks_per_cu")) return &g_opt.store_blocks_per_cu;
  if (!strcmp(name, "store_resident_cap")) return &g_opt.store_resident_cap;
  if (!strcmp(name, "publish_resident_cap")) return &g_opt.publish_resident_cap;
  if (!strcmp(name, "cached_arena_bytes")) return &g_opt.cached_arena_bytes;
  if (!strcmp(name, "cached_output_bytes")) return &g_opt.cached_output_bytes;
  if (!strcmp(name, "plain_output_bytes")) return &g_opt.plain_output_bytes;
  if (!strcmp(name, "cached_gradient_bytes")) return &g_opt.cached_gradient_bytes;
  if (!strcmp(name, "resident_accumulation_bytes")) return &g_opt.resident_accumulation_bytes;
  if (!strcmp(name, "resident_shard_bytes")) return &g_opt.resident_shard_bytes;
  if (!strcmp(name, "resident_above")) return &g_opt.resident_above;
  if (!strcmp(name, "resident_clear_bytes")) return &g_opt.resident_clear_bytes;
  if (!strcmp(name, "plain_accumulation_bytes")) return &g_opt.plain_accumulation_bytes;
  if (!strcmp(name, "through_store_bytes")) return &g_opt.through_store_bytes;
  if (!strcmp(name, "through_clear_bytes")) return &g_opt.through_clear_bytes;
  if (!strcmp(name, "cast_output_bytes")) return &g_opt.cast_output_bytes;
  if (!strcmp(name, "stream_bytes")) return &g_opt.stream_bytes;
  if (!strcmp(name, "short_tiles_below")) return &g_opt.short_tiles_below;
  if (!strcmp(name, "tiny_tiles_from")) return &g_opt.tiny_tiles_from;
  if (!strcmp(name, "few_tiles")) return &g_opt.few_tiles;
  return nullptr;
}

using namespace odc_tiles;
using namespace odc_launch;

// ------------------------------------------------------------------------------------------------
// host side: arena
// ------------------------------------------------------------------------------------------------
constexpr uint64_t kAlign = 256;

inline uint64_t round_up(uint64_t x, uint64_t a) { return (x + a - 1) / a * a; }

}  // namespace

struct odc_arena {
  uint32_t world = 0;
  int device = -1;
  uint32_t flags = 0;
  int n_cu = 256;
  int lds_per_cu = 160 * 1024;
  int lds_per_wg_max = 64 * 1024;
  uint64_t bytes_per_rank = 0;
  uint64_t rank_stride = 0;
  uint64_t alloc_align = 16384;
  void* allocation = nullptr;  // the one device allocation (null without backing)
  uint8_t* base = nullptr;    // rank 0's region: the allocation rounded up to the stride alignment
  uint8_t* origin = nullptr;  // what launches are planned against: base, or a fictitious address on a dry-run arena
  bool dry_run = false;
  std::map<uint64_t, uint64_t> live;  // offset -> size (rounded)
  std::map<uint64_t, uint64_t> free_; // offset -> size, coalesced
  std::atomic<uint64_t> in_use{0};  // changed under mu, read by launches without it
  uint64_t high_water = 0;
  std::mutex mu;
};

namespace {

int check_arena(const odc_arena* a) {
  if (!a) return fail(ODC_ERR_INVALID, "arena is NULL");
  return ODC_OK;
}

// Makes the arena's device current for the scope of one entry point and puts the caller's
// device back afterwards (the caller may be any host thread with any current device).
class DeviceGuard {
 public:
  DeviceGuard() = default;
  DeviceGuard(const DeviceGuard&) = delete;
  DeviceGuard& operator=(const DeviceGuard&) = delete;
  int enter(int device) {
    ODC_DEVICE_TRY(odc_device::get_current(&prev_));
    if (prev_ != device) {
      ODC_DEVICE_TRY(odc_device::set_current(device));
      switched_ = true;
    }
    return ODC_OK;
  }
  ~DeviceGuard() {
    if (switched_) (void)odc_device::set_current(prev_);
  }

 private:
  int prev_ = -1;
  bool switched_ = false;
};

int check_compute(odc_arena* a, DeviceGuard& guard) {
  if (int rc = check_arena(a)) return rc;
  if (a->dry_run) return ODC_OK;  // plans against a fictitious address, launches nothing
  if (!a->base)
    return fail(ODC_ERR_NO_BACKING, "arena has no device memory (created with ODC_ARENA_NO_BACKING)");
  return guard.enter(a->device);
}

// What dry-run arenas have "launched" (process-wide, reset by odc_set_option("dry_run_reset", 0)).
std::atomic<int64_t> g_dry_launches{0}, g_dry_tiles{0}, g_dry_workgroups{0};
std::atomic<int64_t> g_dry_short{0}, g_dry_few{0}, g_dry_tiny{0}, g_dry_stream{0};  // of the launches: those in kShortTiles, ...
std::atomic<int64_t> g_dry_resident{0};  // those that are told of a resident part
std::atomic<int64_t> g_dry_through{0};   // those that write through the L2s

template <class Launch> TileForm form_of(const Launch& L) { return L.form; }
TileForm form_of(const ClearLaunch&) { return kWholeTiles; }
template <class Launch> bool writes_through(const Launch& L) { return L.output == kWriteThrough; }
bool writes_through(const AccumLaunch& L) { return L.policy.read && L.policy.written == kWriteThrough; }
bool writes_through(const PublishLaunch&) { return false; }

// The one place kernels are launched from: `issue` is the odc_device launch of the entry point.
// On a dry-run arena the launch is only counted: the host-side validation, work-list splitting
// and tile tables have all run by then.
template <class Launch, class Issue>
int launch_tiles(const odc_arena* a, const Launch& L, uint32_t grid, Issue issue) {
  if (grid == 0 || grid > L.tt.n_tiles || L.tt.n_tiles != L.tt.tiles_per_rank * L.tt.world)
    return fail(ODC_ERR_INVALID, "internal: launch of %u workgroups over %u tiles", grid, L.tt.n_tiles);
  if (a->dry_run) {
    g_dry_launches += 1;
    g_dry_tiles += L.tt.n_tiles;
    g_dry_workgroups += grid;
    g_dry_short += form_of(L) == kShortTiles;
    g_dry_few += form_of(L) == kFewShortTiles || form_of(L) == kTinyTiles;
    g_dry_tiny += form_of(L) == kTinyTiles;
    g_dry_stream += form_of(L) == kStreamTiles;
    g_dry_resident += L.tt.resident_below != 0;
    g_dry_through += writes_through(L);
    return ODC_OK;
  }
  const int e = issue();
  if (e != 0) return fail(ODC_ERR_HIP, "kernel launch failed: %s", odc_device::error_string(e));
  return ODC_OK;
}

Options options_snapshot() {
  std::lock_guard<std::mutex> lk(g_opt_mu);
  return g_opt;
}

// blocks_per_cu > 0 asks for that many persistent workgroups per CU. Ragged launches (uneven
// shards: unaligned reads, heads and tails) never get them: they hide their extra latency better
// with one workgroup per tile, i.e. full occupancy (measured: +5..10 %). ragged() looks at every item and
// is asked only where persistent workgroups are.
template <class Ragged>
uint32_t grid_for(const odc_arena* a, int64_t blocks_per_cu, uint32_t n_tiles, uint32_t threads, Ragged ragged) {
  const uint32_t most = std::min(n_tiles, most_workgroups(threads));
  if (blocks_per_cu <= 0 || ragged()) return most;
  const uint64_t cu = (uint64_t)a->n_cu, per_cu = (uint64_t)blocks_per_cu;
  return per_cu >= most ? most : (uint32_t)std::min<uint64_t>(cu * per_cu, most);
}
uint32_t grid_for(const odc_arena* a, int64_t blocks_per_cu, uint32_t n_tiles, uint32_t threads) {
  return grid_for(a, blocks_per_cu, n_tiles, threads, [] { return false; });
}

// What a launch leaves in the caches. Nontemporal accesses stream fastest when nothing will be
// found again (a decoder layer's 2.2 GB: +15 % over plain ones), but they also pass by what IS in
// the 256 MB last-level cache and leave nothing there for the kernel that comes next. Measured as
// pairs, in us (16 Mi elements at W = 8, 24 sets of buffers in turn so that nothing else stays
// cached / 3 sets), nontemporal -> plain on the stream named:
//   * the gradient, written by the backward just before: fill + accumulate 35.7 -> 33.3 / 35.5 -> 32.9,
//     fill + store 28.8 -> 24.3 / 28.7 -> 23.8 (nine items), 64 Mi elements 126.8 -> 115.7. Without
//     the fill 64 Mi elements lose 1.5 %, beyond that nothing is left of the gradient when it is
//     read, so the line is 128 MiB of gradient.
//   * the gathers' output, read by the forward or backward just after: gather + read 20.3 -> 18.7 /
//     19.2 -> 17.5, still 64.7 -> 62.3 at 64 Mi elements, but the gather alone is then 42.1 -> 45.8
//     (22.1 -> 19.1 at 32 Mi): the line is 64 MiB of output.
//     What reads it in earnest are products: of a decoder layer's step (gather, forward products, gather,
//     backward products, accumulate) the cached output takes 234 -> 213 at 14 MiB and 512 tokens, 592 ->
//     565 at 35 MiB and 2048, 762 -> 713 at 59 MiB and 2048, 1535 -> 1511 at 8192. It costs where
//     nothing reads it: a gather and accumulate of 17 MiB 21.0 -> 24.0, of 48 MiB 40.4 -> 41.7 (written
//     through, 41.1: output_form).
//   * shards and accumulations come back only in the next microbatch, so what counts is whether ALL
//     symmetric memory in use stays in the cache from one to the next: with 72 MB of it (4 Mi
//     elements, 3 sets) fill + accumulate 12.7 -> 10.8 and accumulate alone 8.9 -> 7.9, with 144 MB
//     accumulate alone 14.6 -> 12.4 and gather alone 7.0 -> 6.2; with 600 MB (24 sets) fill +
//     accumulate 12.8 -> 13.1 and gather + read 7.4 -> 8.0. The line is 192 MiB of the 256.
// How what stays is written: output_form, accumulation_form, a store's accumulations: store_output_form, the converting
// gather's output: cast_output_form.
CachePolicy cache_policy(const odc_arena* a, const Options& opt, uint64_t read_bytes, int64_t read_line,
                         uint64_t written_bytes, int64_t written_line) {
  const bool arena_fits = a->in_use.load(std::memory_order_relaxed) * a->world <= (uint64_t)opt.cached_arena_bytes;
  CachePolicy p;
  p.read = read_line < 0 ? arena_fits : read_bytes <= (uint64_t)read_line;
  p.written = written_line < 0 ? arena_fits : written_bytes <= (uint64_t)written_line;
  return p;
}
constexpr int64_t kSymmetric = -1;  // a line: the stream lies in symmetric memory

// The part of symmetric memory that stays in the last-level cache when all of it does not fit. Streams that
// pass by the cache do not push out what others have left in it (a read-modify-write of 872 MB of which
// 128 MB are read through the caches takes 307 us instead of 346 with 0.9, 1.7 and 3.5 GB of nontemporal
// copies between two of them alike), so a fixed subset of the accumulations, touched twice by every
// accumulate, and of the shards can live there from one kernel to the next (is_resident in odc_tiles.h
// says which bytes, and which launches leave them out: gathers read them, accumulates read and write them, and
// stores and clears write them with plain accesses; everything else of these launches is nontemporal).
// Up to 640 MiB in use there is none, and no accumulation's where the launch's gradient is cached: gradients
// and gathered outputs of such sizes leave no room (bf16 into fp32, three sets of buffers in turn: gather +
// accumulate of 17 Mi elements 41.8 us without, 48.8 with; of 40 M 85 and 99). Otherwise accumulations have
// 320 MiB's share of the memory in use, shards 80 MiB's: with one unit in the arena as much of it as the
// cache takes, with many the parts of all of them together still fit. us without -> with, at W = 8, three
// units in turn: gather + accumulate of 75 M elements 165 -> 158, two microbatches of it 329 -> 313; of a
// decoder layer 473 -> 462; a layer's store, 3 accumulates, 4 gathers and publish 1802 -> 1750; its FSDP2
// minibatch of two microbatches, mixed 1666 -> 1656, bf16 1044 -> 1033, fp32 2061 -> 2039. (384 MiB's share:
// 314, 470, 1742, 1651, 1028; 256: 460, 1751, 1658, 1031. Ten units in turn, each part small and to last for
// 25 GB, at 384: layer 482 -> 481, minibatches 1827 -> 1803, 1685 -> 1688, 1045.5 -> 1044.6. Converting
// gathers gain nothing.) With a layer's forward and backward products between the passes, which read through the
// caches, a step is level: -0.4 to +0.3 % over 94 M and 218 M parameters, 1, 3 and 8 units in turn and 128 to 2048
// tokens (218 M, 3 units, 1024 tokens 2113 -> 2105, its accumulate 339 -> 330; 128 tokens 1479 -> 1483, 344 ->
// 338: the products give back what they no longer find).
uint32_t resident_below(const odc_arena* a, const Options& opt, int64_t most) {
  const double in_use = (double)(a->in_use.load(std::memory_order_relaxed) * a->world);
  if (in_use <= (double)opt.resident_above) return 0;
  return (uint32_t)std::min(4294967295.0, (double)most / in_use * 4294967296.0);
}

// How a gather writes an output that stays in the caches: written through the L2s to the last-level cache
// (store_output in odc_kernels.hip). Plain stores leave up to what the L2s hold (8 x 4 MB) in them as dirty lines,
// whose way out the kernel, or the next one, then waits for; the lines that are written through stay there for the
// next kernel too. Below 3 MiB the two are level or plain stores ahead by up to 0.2 us. Graph-replayed gathers of
// bf16 at W = 8, us, plain -> written through, one item on one set of buffers, nine items on three sets in turn:
//   1 M elements 2.25 -> 2.28, 2.55 -> 2.76; 2.1 M (4 MiB) 2.48 -> 2.38, 3.06 -> 3.07; 4.2 M 3.27 -> 2.84, 4.24 -> 3.61; 8.4 M
//   4.90 -> 4.09, 6.54 -> 6.35; 16.8 M and more level.
// With products of 128 to 1024 tokens that read the output and write the gradient behind the gather, outputs of
// 1 to 25 MiB: level or ahead by up to 2 % (9 MiB, 512 tokens, forward 28.05 -> 27.4, with backward 57.5 -> 57.1).
OutputForm output_form(const Options& opt, bool cached, uint64_t bytes) {
  if (!cached) return kStream;
  return bytes <= (uint64_t)opt.plain_output_bytes ? kKeep : kWriteThrough;
}

// How an accumulate writes accumulations that stay in the caches: likewise from 3 MiB of them on. Where one
// accumulate is repeated over one set of buffers with at most a gather between, accumulations of 8 to 16 MiB never
// leave the L2s and plain stores are ahead; with a clear, other buffers, more items or larger ones between it is the
// other way round, and a minibatch has those. us as above, bf16 into fp32, plain -> written through:
//   accumulate: 1 M elements (4 MiB) 2.86 -> 2.85, 3.35 -> 3.27; 2.1 M 3.45 -> 3.61, 4.60 -> 4.09; 3 M 4.12 -> 4.48, 6.28 -> 5.11;
//     4.2 M (16 MiB) 4.87 -> 5.59, 7.52 -> 6.84; 8.4 M 12.05 -> 9.31, 12.8 -> 12.4; 12.6 M 17.1 -> 15.0, 18.3 -> 18.0; 16.8 M
//     21.9 -> 21.2, 24.0 -> 23.9; into bf16 4.2 M 4.09 -> 3.61, 6.06 -> 5.33, 8.4 M 6.20 -> 5.61, 9.75 -> 8.91;
//   gather, accumulate: 1 M 5.03 -> 4.97, 6.10 -> 5.75; 2.1 M 5.88 -> 6.05, 8.27 -> 7.57; 3 M 6.81 -> 7.11, 9.95 -> 9.40; 4.2 M
//     9.05 -> 8.58, 11.9 -> 11.7; 8.4 M 17.6 -> 16.8, 22.2 -> 22.0; 33.5 M 65.4 -> 66.6, 81.7 -> 81.4;
//   minibatches (clear, four times that, publish): 1 M 24.8 -> 23.4, 29.6 -> 27.2; 2.1 M 30.3 -> 28.2, 36.3 -> 34.9; 4.2 M 47.5 ->
//     39.8, 48.5 -> 48.2 (one item, three sets 43.0 -> 44.2); 8.4 M 84.9 -> 73.1, 89.1 -> 86.7; 12.6 M 113.5 -> 107.8,
//     121.7 -> 121.2; 33.5 M 279 -> 270, 302 -> 302.
OutputForm accumulation_form(const Options& opt, bool cached, uint64_t bytes) {
  if (!cached) return kStream;
  return bytes <= (uint64_t)opt.plain_accumulation_bytes ? kKeep : kWriteThrough;
}

// A store's accumulations, which it does not read: written through from 3 to 44 MiB, nontemporal otherwise. us as
// above, nontemporal -> written through:
//   store of bf16 into fp32: 0.52 M elements 2.19 -> 2.24, 2.66 -> 2.60; 1 M 2.51 -> 2.41, 3.05 -> 3.00; 4.2 M 4.19 -> 4.16, 5.38 ->
//     4.99; 8.4 M 6.46 -> 6.47, 8.40 -> 8.50; 10.5 M (40 MiB) 7.66 -> 7.31, 9.95 -> 9.97; 12.6 M (48 MiB) 9.15 -> 8.44, 11.7 ->
//     13.0; 14.7 M 11.4 -> 9.92, 13.1 -> 16.1; 16.8 M 13.4 -> 12.0, 14.4 -> 14.3, one item over three sets 13.5 -> 16.0;
//   gather, store, gather, accumulate: 4.2 M 17.4 -> 16.0, 20.0 -> 19.2; 8.4 M 29.4 -> 27.8, 35.5 -> 35.9; 10.5 M 35.5 -> 34.5,
//     45.7 -> 43.6; 12.6 M 42.7 -> 42.3, 48.2 -> 48.3; 14.7 M 48.2 -> 47.8, 54.6 -> 54.6; 16.8 M 52.1 -> 51.8, 60.3 -> 60.0;
//   lazy minibatches: 4.2 M 37.0 -> 35.5, 43.3 -> 42.4; 10.5 M 80.5 -> 79.5, 96.5 -> 94.4; 12.6 M 94.7 -> 94.0, 108.4 -> 108.2; 16.8 M
//     115.8 -> 115.3, 134.2 -> 134.0.
// From 48 MiB on what one set gains in passes, 1 %, is less than what the store itself loses over several.
OutputForm store_output_form(const Options& opt, bool cached, uint64_t bytes) {
  const bool through = cached && bytes > (uint64_t)opt.plain_accumulation_bytes && bytes <= (uint64_t)opt.through_store_bytes;
  return through ? kWriteThrough : kStream;
}

// output_form for a gather that converts, and for a conversion of symmetric memory, which are ahead with the output
// written through whoever reads it, as long as it leaves room for the gradients and accumulations of the
// pass: up to 32 MiB, and 64 MiB of copies that the gathers behind find in the cache. Passes, fp32 into bf16 at
// W = 8, us, nontemporal -> written through: gather + accumulate of 9 M elements 27.5 -> 26.9, 13 M 38.2 ->
// 37.3, three microbatches of 9 M 92.7 -> 91.1, FSDP1 minibatches of 9 M 97.1 -> 95.3, 13 M 125.0 -> 122.7,
// 18 M 162.6 -> 156; but gather + accumulate of 24 M 61.2 -> 63.0, 32 M 80.4 -> 86.5. FSDP2 minibatches
// over converted copies of 12 to 57 MB: 185.8 -> 183.7, 245.3 -> 242.2.
// Where all symmetric memory fits they are written through as plain gathers are, us, plain -> written through, one
// item on one set of buffers, nine items on three sets: 1 M elements 2.27 -> 2.13, 2.94 -> 3.00; 2.1 M 2.92 -> 2.66, 3.87 ->
// 3.61; 4.2 M 3.95 -> 3.43, 5.70 -> 5.41; 8.4 M 8.09 -> 5.83, 8.74 -> 8.69; 16.8 M and more level.
OutputForm cast_output_form(const Options& opt, bool cached, uint64_t bytes, int64_t line) {
  return cached ? output_form(opt, true, bytes) : bytes <= (uint64_t)line ? kWriteThrough : kStream;
}

// How a clear without a resident part writes its zeros: through the L2s while the last-level cache holds them
// all, with plain stores beyond. Graph-replayed clears of fp32 accumulations at W = 8, us, plain -> written
// through: one item of 0.26 M elements 1.95 -> 1.82, 1 M 2.36 -> 2.20, 2.1 M 3.06 -> 2.54, 4.2 M 4.53 -> 3.48, 8.4 M
// 6.8 -> 5.5, 16.8 M 10.9 -> 9.7, 33 M 19.1 -> 17.8, 60 M (229 MiB) 32.8 -> 31.1; nine items, three sets in turn,
// 33 M 23.7 -> 22.8, 60 M 41.6 -> 40.0, but 70 M 50.6 -> 53.1, 100 M 68.3 -> 72.7, a decoder layer 142 -> 148.
OutputForm clear_form(const Options& opt, uint64_t bytes) {
  return bytes <= (uint64_t)opt.through_clear_bytes ? kWriteThrough : kKeep;
}

// The items that the next launch over [next, n_items) can take, and their whole tiles and units on one rank.
// also(i) is called for each of them: whatever else a launch's plan sums up over its items is summed on the
// same walk. Passes of six launches, 300 small slices at W = 16, whose host time is level with their kernels',
// took 36.7 -> 39.3 us when plans of long streams had walks of their own; with one walk, no division per
// item and grid_for's look at the items only where it is used, 35.9 -> 36.1, 37.5 -> 36.8 and 36.1 -> 36.8 on three cards.
struct LaunchSize {
  uint32_t items = 0;
  uint64_t tiles = 0;
  uint64_t units = 0;
};
constexpr uint64_t kMostStreamTiles = 1u << 24;  // well below a dispatch's most workgroups
template <uint64_t kTileUnits, class Units, class Also>
LaunchSize launch_size(uint32_t n_items, uint32_t next, Units units, Also also) {
  LaunchSize size;
  for (uint32_t i = next; i < n_items && size.items < (uint32_t)kMaxItems; ++i) {
    const uint64_t n = units(i);
    size.tiles += tiles_for(n, kTileUnits);
    size.units += n;
    size.items += n != 0;
    also(i);
  }
  return size;
}
template <uint64_t kTileUnits, class Units>
LaunchSize launch_size(uint32_t n_items, uint32_t next, Units units) {
  return launch_size<kTileUnits>(n_items, next, units, [](uint32_t) {});
}

// Whether the next launch over items [next, n_items) is cut into short tiles (256 vectors, done by
// 128-thread workgroups): when its segments, one item on one rank, average fewer than `below` = 32
// whole tiles. A workgroup of 256 or 512 threads whose segment holds a few hundred elements keeps the
// wave slots of its CU from others and does nothing with them, and a launch of a few dozen whole tiles
// leaves most CUs idle. Graph-replayed launches, us, whole -> short:
//   300 slices of 64 .. 65 536 elements, gather + accumulate: W = 4 31.7 -> 29.4, W = 16 46.5 -> 31.8,
//     W = 64 122 -> 56;
//   60 items at W = 8, gather: 300 elements per segment 3.6 -> 2.9, 10 000 6.5 -> 5.6, 40 000 14.0 -> 13.8;
//   one item at W = 8, gather: 19 000 elements per segment 2.5 -> 2.2, 300 000 (37 tiles) 3.3 -> 3.2,
//     600 000 (73) 4.55 -> 4.65; converting gather level from there on, store 5.0 -> 5.5 at 600 000.
// Launches of longer segments stream best in whole tiles, with one exception (accum_streams_short).
bool wants_short_tiles(const LaunchSize& size, int64_t below) { return size.tiles < (uint64_t)below * size.items; }

// The same for an accumulate or a store. One that would take short tiles does not where 16-bit
// gradients are stored into 16-bit accumulations and the launch has more than 1536 whole tiles: a short
// tile of theirs moves 4 KB, too little for the cost of a workgroup once there are enough others.
// Graph-replayed stores over 900 MB of buffers in turn, bf16 into bf16, us, short -> whole:
//   W = 8, segments of 31 tiles: 9 items 9.8 -> 9.3, 30 items 24.8 -> 23.1, 60 items 49.7 -> 42.7;
//   of 16 tiles: 30 items 14.6 -> 13.6, 60 items 25.1 -> 23.4; of 8: 30 items (1920 tiles) 8.76 -> 8.45;
//   W = 32: 9 items of 16 tiles 17.1 -> 16.3, 60 of 4 25.3 -> 23.9, nontemporal 16.5 -> 15.2, 24.7 -> 22.8;
//   1152 tiles in all: 6.5 -> 6.25, nontemporal 6.1 -> 6.2; 960: 5.0 -> 4.9 .. 5.3, nontemporal 5.45 ->
//   5.8; 576: 4.1 -> 4.3.
// The read-modify-write of the same types has no such line: nontemporal short tiles are ahead or level
// throughout (60 items of 16 tiles at W = 8 30.1, whole 33.5; 9 of 31 11.3 and 11.0), cached ones are
// behind by up to 7 % at 4 to 17 Mi elements and ahead by as much at 57 Mi.
bool scatter_in_short_tiles(const odc_arena* a, const LaunchSize& size, int64_t below, int grad_dtype, int acc_dtype,
                            bool store) {
  if (accum_streams_short(grad_dtype, acc_dtype)) return true;
  if (!wants_short_tiles(size, below)) return false;
  const bool narrow = grad_dtype != ODC_DTYPE_F32 && acc_dtype != ODC_DTYPE_F32;
  return !(store && narrow) || size.tiles * a->world <= 1536;
}

// Whether a publish of items [next, n_items) is cut into short tiles. It sees a W-th of the elements
// that the other launches see, and a launch of a few hundred whole tiles leaves most of a CU idle;
// two written streams per read one also stream better from 128 x 2 than from 256 x 4. So
// fp32 accumulations always are. 16-bit ones move 4 to 6 KB per short tile, too little for the cost of
// a workgroup, and are only up to 1024 whole tiles (4 workgroups per CU). Graph-replayed
// launches over buffers in turn, us, whole -> short:
//   fp32 into bf16: ten slices of 98 816 elements 3.5 -> 2.9, one of 1 Mi 4.2 -> 3.65, 112 of 3 640
//     5.2 -> 3.65, one of 3.1 M 9.65 -> 7.1, a decoder layer's 27 M at W = 8 45.8 -> 44.0, eight layers
//     369 -> 335, one of 66 M 108.7 -> 103.4;
//   fp32 in place: 3.2 -> 2.65, 3.8 -> 3.35, 4.35 -> 3.3, 7.65 -> 6.1, 35.8 -> 34.5, 284 -> 267,
//     81.2 -> 82.0;
//   bf16 in place: 3.05 -> 2.7, 3.25 -> 3.05, 4.1 -> 3.0, 4.4 -> 4.2, but 19.5 -> 22.6, 134 -> 173,
//     and 42.0 -> 41.4.
bool publish_in_short_tiles(const LaunchSize& size, int acc_bytes) { return acc_bytes == 4 || size.tiles <= 1024; }

// How the workgroups of a launch find their items. Up to eight fills of the chip (4096 workgroups of
// 128 threads each) a launch is mostly the latency from its arguments to its first loads, and the
// whole prefix table read at once pays off; in longer ones the other workgroups of the CU hide that
// latency and the extra loads only cost. Graph-replayed gather + accumulate of one group of slices,
// us, binary search -> table read at once:
//   300 of 64 .. 65 536 elements: W = 4 27.4 -> 23.2, W = 8 28.6 -> 24.3, W = 64 55.6 -> 45.0;
//   112 of 4096: 6.0 -> 5.1, 6.3 -> 5.7, 17.8 -> 13.5;
//   10 of 256 .. 262 144: 6.1 -> 5.9, 6.5 -> 6.2, 7.2 -> 6.9;
//   112 of 160 000 (17 900 tiles): 41.2 -> 39.7, 41.1 -> 40.2; 112 of 640 000 (70 000 tiles): 156 -> 159,
//   159 -> 162; 60 of 900 000 (53 000 tiles): 115 -> 115, 116.5 -> 117.6.
TileForm table_form(TileForm cut, uint32_t n_tiles, int64_t few) {
  return cut == kShortTiles && n_tiles <= (uint64_t)few ? kFewShortTiles : cut;
}

// What is left of their time goes with the number of wavefronts: some 0.55 us per 1000 workgroups of two. Where
// tiles are at most half full on average the second wavefront has little to do, and from 2048 tiles on (8 per CU)
// launches by the full tables have workgroups of one, which moves four vectors per lane in a full tile. us, 100
// ragged items (a factor of 100 between their sizes), two wavefronts -> one, gather / accumulate of bf16 into fp32 /
// converting gather / store:
//   W = 64, 6400 tiles: 0.26 M elements in all 6.27 -> 4.87, 6.77 -> 5.21, 6.59 -> 4.94, 6.71 -> 5.21; 4.2 M 6.78 -> 5.49, 7.80 ->
//     6.68, 7.28 -> 5.76, 7.29 -> 5.81; W = 32, 3200 tiles: 1 M 4.43 -> 3.99, 4.78 -> 4.25, 4.71 -> 4.24, 4.73 -> 4.20;
//   W = 16, 2096 tiles half full: 3.97 -> 3.94, 4.21 -> 4.22, 4.12 -> 3.95, 3.96 -> 3.88; fewer tiles, gather: 784 2.98 -> 3.32,
//     1568 3.58 -> 3.74; 2544 tiles, 94 % full, accumulate 4.61 -> 4.84.
// (Publishes, of one rank, never have so many half-empty tiles, and no kernels for them.)
TileForm tile_form(TileForm cut, const TileTable& tt, uint64_t units, uint64_t whole_tile_units, const Options& opt) {
  const TileForm form = table_form(cut, tt.n_tiles, opt.few_tiles);
  if (form != kFewShortTiles || tt.n_items <= kFewItems || tt.n_tiles < (uint64_t)opt.tiny_tiles_from) return form;
  const bool half_empty = 2 * units * tt.world <= (uint64_t)tt.n_tiles * (whole_tile_units / kShortTileParts);
  return half_empty ? kTinyTiles : form;
}

// Whether a launch that is otherwise cut as `cut` is a long stream: more than 8 MiB written, past the caches,
// by at most 64 items. Long streams go in short tiles, of which 12 workgroups are resident per CU
// (kStreamWaves). They are bound by how HBM mixes reads and writes, which depends on how many loads are in
// flight per CU (with 12 workgroups 72 KiB in the accumulate of 16-bit gradients, 96 KiB in that of fp32 ones, 48
// KiB in the gather and the fp32 store); how many that are had been decided by the time a workgroup took to find
// its item, and by whole tiles. With the items found early (ItemsWalk) it has to be said. One kernel each on real
// data, us, as they were -> long streams (16 and 10 workgroups per CU; 2 quads per lane in each):
//   accumulate bf16 into fp32: a decoder layer at W = 8 354 -> 338 (349, 343), at W = 64 361 -> 350 (357,
//     356), nine items of 11 .. 27 M elements 260 -> 253 (257, 259), 525 M elements 854 -> 826 (850, 814);
//   fp32 into fp32: nine items of 11 .. 13 M 213 -> 207, their store 137 -> 135, the layer level (416 to 425);
//   gather: the layer 137.4 -> 135.0 (136.9, 136.9), at W = 64 143.5 -> 139 (143, 143), 525 M 332 -> 327 (335,
//     333); of fp32 273 -> 266, nine items of 11 .. 13 M 150 -> 144.
// Passes, gather + accumulate: the layer 482 -> 473, at W = 64 496 -> 481, 40 uneven items at W = 12 728 ->
// 704, 525 M elements 1184 -> 1157; fp32 throughout, minibatches of two microbatches, the layer 2096 -> 2067,
// 20 M elements 132.9 -> 131.0, 14 M 97.8 -> 96.0, 9 M (36 MB written) 67.7 -> 66.6, 4.5 M 40.8 -> 39.8, 3 M
// (12 MB) level. Behind: converting gathers (204 -> 225), stores of 16-bit gradients into fp32 (157.6 -> 161)
// and accumulates into 16 bits (205 -> 220), which keep their shapes. Tiles of 128 vectors with 14 workgroups:
// 342 for the layer's accumulate, 831 for 525 M.
TileForm stream_form(const odc_arena* a, const Options& opt, const LaunchSize& size, uint64_t written_bytes, TileForm cut) {
  const bool fits = size.items <= kSomeItems && size.tiles * a->world * tile_parts(kStreamTiles) <= kMostStreamTiles;
  return fits && written_bytes > (uint64_t)opt.stream_bytes ? kStreamTiles : cut;
}

// The same for an accumulate or a store.
TileForm scatter_stream_form(const odc_arena* a, const Options& opt, const LaunchSize& size, int grad_dtype, int acc_dtype,
                             bool store, AccumPolicy policy, TileForm cut) {
  if (acc_dtype != ODC_DTYPE_F32) return cut;
  if (grad_dtype == ODC_DTYPE_F32 ? cut != kWholeTiles : store || policy.read) return cut;
  return stream_form(a, opt, size, size.units * 4 * a->world, cut);
}

// One-workgroup-per-tile launches are dealt out by the hardware dispatcher, which keeps as many
// workgroups resident as fit. Fewer resident workgroups (a smaller window of memory in flight)
// can stream faster; the only lever is to make each workgroup claim a share of the CU's LDS that
// it never touches. Returns the dynamic LDS bytes that leave room for exactly `cap` workgroups.
uint32_t lds_claim_for(const odc_arena* a, int64_t cap, uint32_t grid, uint32_t n_tiles) {
  if (cap <= 0 || grid != n_tiles) return 0;  // persistent grids size themselves
  const uint64_t per_wg = ((uint64_t)a->lds_per_cu / (uint64_t)cap) & ~(uint64_t)1023;
  return (uint32_t)std::min<uint64_t>(per_wg, (uint64_t)a->lds_per_wg_max);
}

}  // namespace

extern "C" {

const char* odc_last_error(void) { return g_err; }

int odc_abi_version(void) { return ODC_HIP_ABI_VERSION; }

int odc_set_option(const char* name, int64_t value) {
  if (name && !strcmp(name, "dry_run_reset")) {
    g_dry_launches = 0; g_dry_tiles = 0; g_dry_workgroups = 0;
    g_dry_short = 0; g_dry_few = 0; g_dry_tiny = 0; g_dry_stream = 0; g_dry_resident = 0; g_dry_through = 0;
    return ODC_OK;
  }
  std::lock_guard<std::mutex> lk(g_opt_mu);
  int64_t* s = option_slot(name);
  if (!s) return fail(ODC_ERR_INVALID, "unknown option '%s'", name ? name : "(null)");
  const bool may_be_auto = s == &g_opt.accum_blocks_per_cu;  // -1: chosen per launch
  if (value < (may_be_auto ? -1 : 0)) return fail(ODC_ERR_INVALID, "option '%s' must be >= 0", name);
  // the arena layout options enter address arithmetic: keep them where it cannot wrap around
  const bool is_layout = s == &g_opt.rank_stagger_bytes || s == &g_opt.rank_stride_align || s == &g_opt.alloc_align;
  if (is_layout && value > (int64_t(1) << 40))
    return fail(ODC_ERR_INVALID, "option '%s' must be <= 2^40", name);
  *s = value;
  return ODC_OK;
}

int odc_get_option(const char* name, int64_t* value) {
  if (name && value) {
    if (!strcmp(name, "dry_run_launches")) { *value = g_dry_launches.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_tiles")) { *value = g_dry_tiles.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_workgroups")) { *value = g_dry_workgroups.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_short_launches")) { *value = g_dry_short.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_few_launches")) { *value = g_dry_few.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_tiny_launches")) { *value = g_dry_tiny.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_stream_launches")) { *value = g_dry_stream.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_resident_launches")) { *value = g_dry_resident.load(); return ODC_OK; }
    if (!strcmp(name, "dry_run_through_launches")) { *value = g_dry_through.load(); return ODC_OK; }
  }
  std::lock_guard<std::mutex> lk(g_opt_mu);
  int64_t* s = option_slot(name);
  if (!s || !value) return fail(ODC_ERR_INVALID, "unknown option '%s'", name ? name : "(null)");
  *value = *s;
  return ODC_OK;
}

int odc_arena_create(uint32_t world_size, uint64_t bytes_per_rank, uint32_t flags,
                     odc_arena** out) {
  if (!out) return fail(ODC_ERR_INVALID, "out is NULL");
  *out = nullptr;
  if (world_size == 0) return fail(ODC_ERR_INVALID, "world_size must be >= 1");
  if (bytes_per_rank == 0) return fail(ODC_ERR_INVALID, "bytes_per_rank must be > 0");
  if (bytes_per_rank > (uint64_t(1) << 60)) return fail(ODC_ERR_INVALID, "bytes_per_rank must be <= 2^60");
  if (flags & ~(uint32_t)(ODC_ARENA_NO_BACKING | ODC_ARENA_DRY_RUN))
    return fail(ODC_ERR_INVALID, "unknown flags 0x%x", flags);
  if (flags & ODC_ARENA_DRY_RUN) flags |= ODC_ARENA_NO_BACKING;  // a dry run never owns device memory
  odc_arena* a = new (std::nothrow) odc_arena();
  if (!a) return fail(ODC_ERR_NOMEM, "host allocation failed");
  a->world = world_size;
  a->flags = flags;
  const Options opt = options_snapshot();
  const uint64_t stride_align = std::max<uint64_t>(round_up((uint64_t)opt.rank_stride_align, kAlign), kAlign);
  a->alloc_align = std::max<uint64_t>(round_up((uint64_t)opt.alloc_align, kAlign), kAlign);
  a->bytes_per_rank = round_up(bytes_per_rank, kAlign);
  a->rank_stride = round_up(a->bytes_per_rank + round_up((uint64_t)opt.rank_stagger_bytes, kAlign), stride_align);
  // the device allocation promises 256 B alignment only; the regions shall start on stride_align
  // boundaries, so the allocation is that much larger: the whole sum must fit 64 bits
  const uint64_t slack = stride_align > kAlign ? stride_align : 0;
  if (a->rank_stride > (~0ull - slack) / world_size) {
    delete a;
    return fail(ODC_ERR_INVALID, "arena size overflows 64 bits");
  }
  if (!(flags & ODC_ARENA_NO_BACKING)) {
    odc_device::Properties prop = {};
    int e = odc_device::get_current(&a->device);
    if (e == 0) e = odc_device::properties(a->device, &prop);
    void* p = nullptr;
    if (e == 0) e = odc_device::allocate(&p, a->rank_stride * world_size + slack);
    if (e != 0) {
      delete a;
      return fail(odc_device::is_out_of_memory(e) ? ODC_ERR_NOMEM : ODC_ERR_HIP,
                  "creating a %u x %llu byte arena failed: %s", world_size,
                  (unsigned long long)bytes_per_rank, odc_device::error_string(e));
    }
    a->n_cu = prop.n_cu;
    a->lds_per_cu = prop.lds_per_cu;
    a->lds_per_wg_max = prop.lds_per_wg_max;
    a->allocation = p;
    a->base = reinterpret_cast<uint8_t*>(round_up((uint64_t)(uintptr_t)p, stride_align));
    a->origin = a->base;
  } else if (flags & ODC_ARENA_DRY_RUN) {
    a->dry_run = true;
    a->origin = reinterpret_cast<uint8_t*>(uintptr_t(1) << 44);  // never dereferenced
  }
  a->free_[0] = a->bytes_per_rank;
  *out = a;
  return ODC_OK;
}

int odc_arena_destroy(odc_arena* a) {
  if (int rc = check_arena(a)) return rc;
  int rc = ODC_OK;
  if (a->base) {
    int cur = -1;
    int e = odc_device::get_current(&cur);
    if (e == 0 && cur != a->device) e = odc_device::set_current(a->device);
    if (e == 0) e = odc_device::release(a->allocation);
    if (e != 0) rc = fail(ODC_ERR_HIP, "releasing the arena failed: %s", odc_device::error_string(e));
  }
  delete a;
  return rc;
}

int odc_arena_alloc(odc_arena* a, uint64_t nbytes, uint64_t* offset) {
  if (int rc = check_arena(a)) return rc;
  if (!offset) return fail(ODC_ERR_INVALID, "offset is NULL");
  std::lock_guard<std::mutex> lk(a->mu);
  const uint64_t need = std::max<uint64_t>(round_up(nbytes, kAlign), kAlign);
  if (need < nbytes) return fail(ODC_ERR_INVALID, "nbytes overflows");
  // a buffer of at least one tile starts on a tile-sized boundary (the read-modify-write of the
  // scatter-accumulate is up to 5.5 % slower on accumulations whose tiles straddle them);
  // smaller ones only need the 256 bytes the vector accesses want
  const uint64_t align = need >= a->alloc_align ? a->alloc_align : kAlign;
  for (auto it = a->free_.begin(); it != a->free_.end(); ++it) {  // first fit
    const uint64_t blk = it->first, blk_sz = it->second;
    const uint64_t off = round_up(blk, align);
    if (off < blk || off - blk > blk_sz || blk_sz - (off - blk) < need) continue;
    a->free_.erase(it);
    if (off > blk) a->free_[blk] = off - blk;  // the gap in front stays free
    if (blk + blk_sz > off + need) a->free_[off + need] = blk + blk_sz - (off + need);
    a->live[off] = need;
    a->in_use += need;
    a->high_water = std::max(a->high_water, off + need);
    *offset = off;
    return ODC_OK;
  }
  uint64_t largest = 0;
  for (const auto& blk : a->free_) largest = std::max(largest, blk.second);
  return fail(ODC_ERR_NOMEM,
              "symmetric arena exhausted: need %llu bytes per rank on a %llu-byte boundary, %llu of %llu "
              "in use, largest free block %llu (raise ODC_SYMMETRIC_SIZE)",
              (unsigned long long)need, (unsigned long long)align, (unsigned long long)a->in_use,
              (unsigned long long)a->bytes_per_rank, (unsigned long long)largest);
}

int odc_arena_free(odc_arena* a, uint64_t offset) {
  if (int rc = check_arena(a)) return rc;
  std::lock_guard<std::mutex> lk(a->mu);
  auto it = a->live.find(offset);
  if (it == a->live.end())
    return fail(ODC_ERR_NOT_FOUND, "offset %llu is not a live allocation", (unsigned long long)offset);
  uint64_t off = it->first, sz = it->second;
  a->live.erase(it);
  a->in_use -= sz;
  auto next = a->free_.lower_bound(off);
  if (next != a->free_.end() && off + sz == next->first) {  // merge with the block after
    sz += next->second;
    next = a->free_.erase(next);
  }
  if (next != a->free_.begin()) {  // merge with the block before
    auto prev = std::prev(next);
    if (prev->first + prev->second == off) {
      prev->second += sz;
      return ODC_OK;
    }
  }
  a->free_[off] = sz;
  return ODC_OK;
}

int odc_arena_reset(odc_arena* a) {
  if (int rc = check_arena(a)) return rc;
  std::lock_guard<std::mutex> lk(a->mu);
  a->live.clear();
  a->free_.clear();
  a->free_[0] = a->bytes_per_rank;
  a->in_use = 0;
  return ODC_OK;
}

int odc_arena_get_info(const odc_arena* a, odc_arena_info* info) {
  if (int rc = check_arena(a)) return rc;
  if (!info) return fail(ODC_ERR_INVALID, "info is NULL");
  odc_arena* m = const_cast<odc_arena*>(a);
  std::lock_guard<std::mutex> lk(m->mu);
  info->world_size = a->world;
  info->device = a->base ? a->device : -1;
  info->flags = a->flags;
  info->n_allocations = (uint32_t)a->live.size();
  info->bytes_per_rank = a->bytes_per_rank;
  info->rank_stride = a->rank_stride;
  info->base = (uint64_t)(uintptr_t)a->base;
  info->bytes_in_use = a->in_use;
  info->high_water = a->high_water;
  return ODC_OK;
}

void* odc_arena_ptr(const odc_arena* a, uint32_t rank, uint64_t offset) {
  if (!a || !a->base || rank >= a->world || offset > a->bytes_per_rank) {
    fail(ODC_ERR_INVALID, "odc_arena_ptr: bad arena, rank %u or offset %llu", rank,
         (unsigned long long)offset);
    return nullptr;
  }
  return a->base + (uint64_t)rank * a->rank_stride + offset;
}

int odc_arena_locate(const odc_arena* a, const void* ptr, uint32_t* rank, uint64_t* alloc_offset,
                     uint64_t* inner) {
  if (int rc = check_arena(a)) return rc;
  if (!a->base) return fail(ODC_ERR_NO_BACKING, "arena has no device memory");
  const uint8_t* p = static_cast<const uint8_t*>(ptr);
  if (p < a->base || p >= a->base + a->rank_stride * a->world)
    return fail(ODC_ERR_NOT_FOUND, "pointer %p is outside the arena", ptr);
  const uint64_t d = (uint64_t)(p - a->base);
  const uint32_t r = (uint32_t)(d / a->rank_stride);
  const uint64_t off = d - (uint64_t)r * a->rank_stride;
  odc_arena* m = const_cast<odc_arena*>(a);
  std::lock_guard<std::mutex> lk(m->mu);
  auto it = a->live.upper_bound(off);
  if (it == a->live.begin()) return fail(ODC_ERR_NOT_FOUND, "pointer %p is not in a live allocation", ptr);
  --it;
  if (off >= it->first + it->second)
    return fail(ODC_ERR_NOT_FOUND, "pointer %p is not in a live allocation", ptr);
  if (rank) *rank = r;
  if (alloc_offset) *alloc_offset = it->first;
  if (inner) *inner = off - it->first;
  return ODC_OK;
}

// ------------------------------------------------------------------------------------------------
// launches
// ------------------------------------------------------------------------------------------------
}  // extern "C"

namespace {

int dtype_bytes(int dt) {
  switch (dt) {
    case ODC_DTYPE_BF16: return 2;
    case ODC_DTYPE_F16: return 2;
    case ODC_DTYPE_F32: return 4;
    default: return 0;
  }
}

// odc_tiles::fill_tile_table with its failure turned into an error message.
// `order`, when given, maps positions of the launch order to the caller's item indices (for the
// message only: units and take already work on positions). The units of a tile are constants of the code, so
// that an item costs a shift and not a division.
template <uint64_t kWhole, class Units, class Take>
int fill_launch(TileTable& tt, uint32_t world, uint32_t n_items, uint32_t* next, TileForm cut, Units units, Take take,
                const uint32_t* order = nullptr) {
  typedef std::integral_constant<uint64_t, kWhole> Whole;
  typedef std::integral_constant<uint64_t, kWhole / kShortTileParts> Short;
  const int n = cut == kWholeTiles ? fill_tile_table(tt, world, n_items, next, Whole{}, units, take)
                                   : fill_tile_table(tt, world, n_items, next, Short{}, units, take);
  if (n < 0) {
    const uint32_t at = (uint32_t)(-1 - n);
    return fail(ODC_ERR_INVALID, "item %u: %llu units per rank is too large for one launch", order ? order[at] : at,
                (unsigned long long)units(at));
  }
  return n;
}

int check_rank_range(const odc_arena* a, const char* what, uint32_t i, uint64_t offset, uint64_t nbytes) {
  if (offset > a->bytes_per_rank || nbytes > a->bytes_per_rank - offset)
    return fail(ODC_ERR_INVALID, "%s %u: [%llu, +%llu) leaves the %llu byte rank region", what, i,
                (unsigned long long)offset, (unsigned long long)nbytes,
                (unsigned long long)a->bytes_per_rank);
  return ODC_OK;
}

// The same for `elems` elements of `elem_bytes` each; an element count whose byte size would wrap
// around is rejected before it is multiplied.
int check_rank_elems(const odc_arena* a, const char* what, uint32_t i, uint64_t offset, uint64_t elems,
                     uint64_t elem_bytes) {
  if (elems > a->bytes_per_rank / elem_bytes)
    return fail(ODC_ERR_INVALID, "%s %u: %llu elements of %llu bytes exceed the %llu byte rank region", what, i,
                (unsigned long long)elems, (unsigned long long)elem_bytes, (unsigned long long)a->bytes_per_rank);
  return check_rank_range(a, what, i, offset, elems * elem_bytes);
}

// dst [d0, d0 + world*seg_bytes) must not overlap any rank's source range at src_offset.
int check_no_overlap(const odc_arena* a, uint32_t i, const void* dst, uint64_t dst_seg_bytes,
                     uint64_t src_offset, uint64_t src_seg_bytes) {
  const uint8_t* d0 = static_cast<const uint8_t*>(dst);
  const uint8_t* d1 = d0 + dst_seg_bytes * a->world;
  if (d1 <= a->origin || d0 >= a->origin + a->rank_stride * a->world) return ODC_OK;
  for (uint32_t r = 0; r < a->world; ++r) {
    const uint8_t* s0 = a->origin + (uint64_t)r * a->rank_stride + src_offset;
    if (d0 < s0 + src_seg_bytes && s0 < d1)
      return fail(ODC_ERR_INVALID, "item %u: dst overlaps rank %u's shard", i, r);
  }
  return ODC_OK;
}

}  // namespace

extern "C" {

int odc_gather(odc_arena* a, const odc_gather_item* items, uint32_t n_items, uint32_t first_rank,
               void* stream) {
  DeviceGuard guard;
  if (int rc = check_compute(a, guard)) return rc;
  if (n_items && !items) return fail(ODC_ERR_INVALID, "items is NULL");
  if (first_rank >= a->world)
    return fail(ODC_ERR_INVALID, "first_rank %u >= world size %u", first_rank, a->world);
  for (uint32_t i = 0; i < n_items; ++i) {
    const odc_gather_item& it = items[i];
    if (it.shard_bytes == 0) continue;
    if (!it.dst) return fail(ODC_ERR_INVALID, "item %u: dst is NULL", i);
    if (int rc = check_rank_range(a, "item", i, it.src_offset, it.shard_bytes)) return rc;
    if (int rc = check_no_overlap(a, i, it.dst, it.shard_bytes, it.src_offset, it.shard_bytes)) return rc;
  }
  const Options opt = options_snapshot();
  uint32_t next = 0;
  while (next < n_items) {
    GatherLaunch L;
    L.base = a->origin;
    L.rank_stride = a->rank_stride;
    L.tt.order = (uint32_t)opt.rank_major;
    L.tt.first_rank = first_rank;
    const auto units = [&](uint32_t i) { return items[i].shard_bytes; };
    const LaunchSize size = launch_size<kTileBytes>(n_items, next, units);
    const uint64_t out_bytes = size.units * a->world;
    L.policy = cache_policy(a, opt, 0, kSymmetric, out_bytes, opt.cached_output_bytes);
    TileForm cut = wants_short_tiles(size, opt.short_tiles_below) ? kShortTiles : kWholeTiles;
    if (cut == kWholeTiles && !L.policy.read && !L.policy.written && opt.gather_blocks_per_cu == 0)
      cut = stream_form(a, opt, size, out_bytes, cut);
    const int n = fill_launch<kTileBytes>(
        L.tt, a->world, n_items, &next, cut, units,
        [&](uint32_t slot, uint32_t i) {
          L.item[slot] = {static_cast<uint8_t*>(items[i].dst), items[i].src_offset, items[i].shard_bytes};
        });
    if (n < 0) return n;
    if (n == 0) continue;
    L.form = tile_form(cut, L.tt, size.units, kTileBytes, opt);
    L.output = output_form(opt, L.policy.written, out_bytes);
    L.tt.resident_below = resident_below(a, opt, opt.resident_shard_bytes);
    const auto ragged = [&] {
      uint64_t bits = 0;
      for (uint32_t k = 0; k < L.tt.n_items; ++k) bits |= (uintptr_t)L.item[k].dst | L.item[k].src_off | L.item[k].seg_bytes;
      return (bits & 15u) != 0;
    };
    const uint32_t grid = grid_for(a, opt.gather_blocks_per_cu, L.tt.n_tiles, copy_threads(L.form), ragged);
    const uint32_t lds = lds_claim_for(a, opt.gather_resident_cap, grid, L.tt.n_tiles);
    if (int rc = launch_tiles(a, L, grid, [&] { return odc_device::launch_gather(L, grid, lds, stream); })) return rc;
  }
  return ODC_OK;
}

int odc_gather_cast(odc_arena* a, const odc_gather_cast_item* items, uint32_t n_items,
                    int src_dtype, int dst_dtype, uint32_t first_rank, void* stream) {
  DeviceGuard guard;
  if (int rc = check_compute(a, guard)) return rc;
  if (n_items && !items) return fail(ODC_ERR_INVALID, "items is NULL");
  if (first_rank >= a->world)
    return fail(ODC_ERR_INVALID, "first_rank %u >= world size %u", first_rank, a->world);
  const int sb = dtype_bytes(src_dtype), db = dtype_bytes(dst_dtype);
  if (!sb || !db) return fail(ODC_ERR_INVALID, "unknown dtype code (src %d, dst %d)", src_dtype, dst_dtype);
  if (!odc_device::has_cast_gather(src_dtype, dst_dtype))
    return fail(ODC_ERR_UNSUPPORTED, "gather from dtype %d into dtype %d is not implemented", src_dtype, dst_dtype);
  for (uint32_t i = 0; i < n_items; ++i) {
    const odc_gather_cast_item& it = items[i];
    if (it.shard_elems == 0) continue;
    if (!it.dst) return fail(ODC_ERR_INVALID, "item %u: dst is NULL", i);
    if (it.shard_elems > a->bytes_per_rank / sb)
      return fail(ODC_ERR_INVALID, "item %u: shard of %llu elements exceeds the rank region", i,
                  (unsigned long long)it.shard_elems);
    if (it.src_offset % sb || (uintptr_t)it.dst % db)
      return fail(ODC_ERR_INVALID, "item %u: src_offset or dst is not aligned to its dtype", i);
    if (int rc = check_rank_elems(a, "item", i, it.src_offset, it.shard_elems, sb)) return rc;
    if (int rc = check_no_overlap(a, i, it.dst, it.shard_elems * db, it.src_offset, it.shard_elems * sb)) return rc;
  }
  const Options opt = options_snapshot();
  uint32_t next = 0;
  while (next < n_items) {
    CastGatherLaunch L;
    L.base = a->origin;
    L.rank_stride = a->rank_stride;
    L.tt.order = (uint32_t)opt.rank_major;
    L.tt.first_rank = first_rank;
    const auto units = [&](uint32_t i) { return items[i].shard_elems; };
    const LaunchSize size = launch_size<kTileElems>(n_items, next, units);
    L.policy = cache_policy(a, opt, 0, kSymmetric, 0, kSymmetric);
    L.output = cast_output_form(opt, L.policy.read, size.units * db * a->world, opt.cast_output_bytes);
    const TileForm cut = wants_short_tiles(size, opt.short_tiles_below) ? kShortTiles : kWholeTiles;
    const int n = fill_launch<kTileElems>(
        L.tt, a->world, n_items, &next, cut, units,
        [&](uint32_t slot, uint32_t i) {
          L.item[slot] = {static_cast<uint8_t*>(items[i].dst), items[i].shard_elems * (uint64_t)db,
                          items[i].src_offset, items[i].shard_elems};
        });
    if (n < 0) return n;
    if (n == 0) continue;
    L.form = tile_form(cut, L.tt, size.units, kTileElems, opt);
    const uint32_t grid = grid_for(a, opt.gather_blocks_per_cu, L.tt.n_tiles, copy_threads(L.form));
    const uint32_t lds = lds_claim_for(a, opt.cast_resident_cap, grid, L.tt.n_tiles);
    if (int rc = launch_tiles(a, L, grid, [&] {
          return odc_device::launch_cast_gather(src_dtype, dst_dtype, L, grid, lds, stream);
        }))
      return rc;
  }
  return ODC_OK;
}

int odc_convert(odc_arena* a, const odc_convert_item* items, uint32_t n_items, int src_dtype,
                int dst_dtype, void* stream) {
  DeviceGuard guard;
  if (int rc = check_compute(a, guard)) return rc;
  if (n_items && !items) return fail(ODC_ERR_INVALID, "items is NULL");
  const int sb = dtype_bytes(src_dtype), db = dtype_bytes(dst_dtype);
  if (!sb || !db) return fail(ODC_ERR_INVALID, "unknown dtype code (src %d, dst %d)", src_dtype, dst_dtype);
  if (!odc_device::has_cast_gather(src_dtype, dst_dtype))
    return fail(ODC_ERR_UNSUPPORTED, "conversion from dtype %d into dtype %d is not implemented", src_dtype, dst_dtype);
  for (uint32_t i = 0; i < n_items; ++i) {
    const odc_convert_item& it = items[i];
    if (it.elems == 0) continue;
    if (it.src_offset % sb || it.dst_offset % db)
      return fail(ODC_ERR_INVALID, "item %u: src_offset or dst_offset is not aligned to its dtype", i);
    if (int rc = check_rank_elems(a, "item (source)", i, it.src_offset, it.elems, sb)) return rc;
    if (int rc = check_rank_elems(a, "item (destination)", i, it.dst_offset, it.elems, db)) return rc;
    // the two ranges lie in the same rank region, in every region: they must not touch
    if (it.dst_offset < it.src_offset + it.elems * sb && it.src_offset < it.dst_offset + it.elems * db)
      return fail(ODC_ERR_INVALID, "item %u: the destination overlaps the source", i);
  }
  const Options opt = options_snapshot();
  uint32_t next = 0;
  while (next < n_items) {
    CastGatherLaunch L;
    L.base = a->origin;
    L.rank_stride = a->rank_stride;
    L.tt.order = (uint32_t)opt.rank_major;
    L.tt.first_rank = 0;
    const auto units = [&](uint32_t i) { return items[i].elems; };
    const LaunchSize size = launch_size<kTileElems>(n_items, next, units);
    L.policy = cache_policy(a, opt, 0, kSymmetric, 0, kSymmetric);
    // (the copies are symmetric memory that every gather of the minibatch reads)
    L.output = cast_output_form(opt, L.policy.read, size.units * db * a->world, opt.cached_output_bytes);
    const TileForm cut = wants_short_tiles(size, opt.short_tiles_below) ? kShortTiles : kWholeTiles;
    const int n = fill_launch<kTileElems>(
        L.tt, a->world, n_items, &next, cut, units,
        [&](uint32_t slot, uint32_t i) {
          // the gather-with-cast kernel with every rank's output in that rank's own region
          L.item[slot] = {a->origin + items[i].dst_offset, a->rank_stride, items[i].src_offset, items[i].elems};
        });
    if (n < 0) return n;
    if (n == 0) continue;
    L.form = tile_form(cut, L.tt, size.units, kTileElems, opt);
    const uint32_t grid = grid_for(a, opt.gather_blocks_per_cu, L.tt.n_tiles, copy_threads(L.form));
    const uint32_t lds = lds_claim_for(a, opt.cast_resident_cap, grid, L.tt.n_tiles);
    if (int rc = launch_tiles(a, L, grid, [&] {
          return odc_device::launch_cast_gather(src_dtype, dst_dtype, L, grid, lds, stream);
        }))
      return rc;
  }
  return ODC_OK;
}

int odc_clear(odc_arena* a, const odc_span* spans, uint32_t n_spans, void* stream) {
  DeviceGuard guard;
  if (int rc = check_compute(a, guard)) return rc;
  if (n_spans && !spans) return fail(ODC_ERR_INVALID, "spans is NULL");
  for (uint32_t i = 0; i < n_spans; ++i)
    if (int rc = check_rank_range(a, "span", i, spans[i].offset, spans[i].nbytes)) return rc;
  const Options opt = options_snapshot();
  uint32_t next = 0;
  while (next < n_spans) {
    ClearLaunch L;
    L.base = a->origin;
    L.rank_stride = a->rank_stride;
    // a write-only stream runs fastest with the ranks interleaved (measured after an accumulate, as
    // in a step: 117 us at W=64 against 123 item-major and 127 rank-outermost; level at W=128)
    L.tt.order = kRanksInterleaved;
    L.tt.first_rank = 0;
    const int n = fill_launch<kTileBytes>(
        L.tt, a->world, n_spans, &next, kWholeTiles, [&](uint32_t i) { return spans[i].nbytes; },
        [&](uint32_t slot, uint32_t i) {
          L.item[slot] = {spans[i].offset, spans[i].nbytes};
        });
    if (n < 0) return n;
    if (n == 0) continue;
    // A clear that leaves the resident part in the cache streams the rest past it, which takes longer (a layer's
    // 872 MB 118 -> 134 us) than leaving the last 256 MB behind unwritten, and pays from 48 MiB of resident
    // zeros on: FSDP2 minibatches 1660 -> 1643, 349 -> 339 (three units in turn, 85 MB each), but 352 -> 360
    // and 331 -> 341 (ten, 26 MB each). Accumulations whose gradients are cached have no resident part; the
    // line is that of 16-bit gradients into fp32.
    uint64_t cleared = 0;
    for (uint32_t k = 0; k < L.tt.n_items; ++k) cleared += L.item[k].seg_bytes * a->world;
    const uint32_t below = resident_below(a, opt, opt.resident_accumulation_bytes);
    const double resident = (double)cleared * below / 4294967296.0;
    if (cleared > 2 * (uint64_t)opt.cached_gradient_bytes && resident >= (double)opt.resident_clear_bytes)
      L.tt.resident_below = below;
    else
      L.output = clear_form(opt, cleared);
    const uint32_t grid = grid_for(a, opt.clear_blocks_per_cu, L.tt.n_tiles, kThreads);
    if (int rc = launch_tiles(a, L, grid, [&] { return odc_device::launch_clear(L, grid, stream); })) return rc;
  }
  return ODC_OK;
}

}  // extern "C"
namespace {

// odc_scatter_accumulate (store == false) and odc_scatter_store (store == true)
int scatter_launch(odc_arena* a, const odc_accum_item* items, uint32_t n_items, int grad_dtype,
                   int acc_dtype, void* stream, bool store) {
  DeviceGuard guard;
  if (int rc = check_compute(a, guard)) return rc;
  if (n_items && !items) return fail(ODC_ERR_INVALID, "items is NULL");
  const int gb = dtype_bytes(grad_dtype), ab = dtype_bytes(acc_dtype);
  if (!gb || !ab) return fail(ODC_ERR_INVALID, "unknown dtype code (grad %d, acc %d)", grad_dtype, acc_dtype);
  if (!odc_device::has_accum(grad_dtype, acc_dtype))
    return fail(ODC_ERR_UNSUPPORTED, "scatter-accumulate of grad dtype %d into acc dtype %d is not implemented",
                grad_dtype, acc_dtype);
  for (uint32_t i = 0; i < n_items; ++i) {
    const odc_accum_item& it = items[i];
    if (it.shard_elems == 0) {
      if (it.grad_elems) return fail(ODC_ERR_INVALID, "item %u: grad_elems > 0 with shard_elems == 0", i);
      continue;
    }
    if (it.shard_elems > a->bytes_per_rank / ab)
      return fail(ODC_ERR_INVALID, "item %u: shard of %llu elements exceeds the rank region", i,
                  (unsigned long long)it.shard_elems);
    if (it.acc_offset % ab)
      return fail(ODC_ERR_INVALID, "item %u: acc_offset %llu is not aligned to the accumulation dtype", i,
                  (unsigned long long)it.acc_offset);
    if (int rc = check_rank_elems(a, "item", i, it.acc_offset, it.shard_elems, ab)) return rc;
    if (it.grad_elems > it.shard_elems * a->world)
      return fail(ODC_ERR_INVALID, "item %u: grad_elems %llu > world_size * shard_elems = %llu", i,
                  (unsigned long long)it.grad_elems, (unsigned long long)(it.shard_elems * a->world));
    if (it.grad_elems && !it.grad) return fail(ODC_ERR_INVALID, "item %u: grad is NULL", i);
    if ((uintptr_t)it.grad % gb)
      return fail(ODC_ERR_INVALID, "item %u: grad pointer is not aligned to the gradient dtype", i);
  }
  const Options opt = options_snapshot();
  // Launch order of the items: those of less than one tile per rank go last. A tiny segment
  // between two long ones (a norm vector's 64-element slice between two projection matrices)
  // slows the read-modify-write stream around it out of all proportion to its size; at the end
  // of the list it costs nothing (measured on the 8B layer, 9 items: -0.6 % of the launch time at
  // W=64, -1.2 % at W=32, -5 % at W=128, nothing at W=8, where there are 16 such tiles instead of
  // 128 or more; the gathers, the clear and the store form do not care). Items of one call are
  // disjoint, so their order never changes the result.
  uint32_t order_inline[256];
  std::vector<uint32_t> order_heap;
  uint32_t* order = order_inline;
  if (n_items > 256) {
    order_heap.resize(n_items);
    order = order_heap.data();
  }
  {
    uint32_t k = 0;
    for (int small = 0; small < 2; ++small)
      for (uint32_t i = 0; i < n_items; ++i)
        if ((opt.accum_small_items_last != 0 && items[i].shard_elems < kTileElems) == (small != 0)) order[k++] = i;
  }
  uint32_t next = 0;
  while (next < n_items) {
    AccumLaunch L;
    L.base = a->origin;
    L.rank_stride = a->rank_stride;
    L.tt.order = (uint32_t)opt.rank_major;
    L.tt.first_rank = 0;
    const auto units = [&](uint32_t i) { return items[order[i]].shard_elems; };
    uint64_t grad_elems = 0;
    const LaunchSize size = launch_size<kTileElems>(n_items, next, units,
                                                    [&](uint32_t i) { grad_elems += items[order[i]].grad_elems; });
    TileForm cut = scatter_in_short_tiles(a, size, opt.short_tiles_below, grad_dtype, acc_dtype, store) ? kShortTiles
                                                                                                      : kWholeTiles;
    const CachePolicy cached = cache_policy(a, opt, grad_elems * gb, opt.cached_gradient_bytes, 0, kSymmetric);
    L.policy.read = cached.read;
    const uint64_t written_bytes = size.units * ab * a->world;
    L.policy.written = store ? store_output_form(opt, cached.written, written_bytes)
                             : accumulation_form(opt, cached.written, written_bytes);
    const bool one_per_tile = (store ? opt.store_blocks_per_cu : opt.accum_blocks_per_cu) <= 0 &&
                              (store || opt.accum_persistent_below_tiles == 0);
    if (one_per_tile && !(cached.read && cached.written))
      cut = scatter_stream_form(a, opt, size, grad_dtype, acc_dtype, store, L.policy, cut);
    const int n = fill_launch<kTileElems>(
        L.tt, a->world, n_items, &next, cut, units,
        [&](uint32_t slot, uint32_t i) {
          const odc_accum_item& it = items[order[i]];
          L.item[slot] = {static_cast<const uint8_t*>(it.grad), it.grad_elems, it.acc_offset, it.shard_elems};
        },
        order);
    if (n < 0) return n;
    if (n == 0) continue;
    L.form = tile_form(cut, L.tt, size.units, kTileElems, opt);
    // Tile order. Item-major (a rank's segment, then the next rank's, item by item) walks the
    // gradient contiguously and hops between rank regions at every segment; rank-outermost walks
    // one rank region from accumulation to accumulation (they are neighbours when registered
    // together) and hops in the gradient instead. The read-modify-write stream is the one worth
    // keeping contiguous once segments get short. Measured on the 8B layer, item-major against
    // rank-outermost: +1.1 % at W=4, +1.6 % at W=16 (370 tiles per segment on average), -1.9 % at
    // W=32 (185), -6 % at W=64, -10 % at W=128.
    const uint64_t segments = (uint64_t)L.tt.n_items * a->world;
    const uint64_t whole_tiles = L.tt.n_tiles / tile_parts(L.form);
    if (opt.accum_tile_order == 3)
      L.tt.order = whole_tiles < (uint64_t)opt.accum_short_segment_tiles * segments ? kRankOutermost : kItemMajor;
    else
      L.tt.order = (uint32_t)opt.accum_tile_order;
    // Launch shape: one workgroup per tile. A persistent shape (one workgroup per CU,
    // "accum_blocks_per_cu" = 1, or automatically below "accum_persistent_below_tiles" tiles per
    // segment) used to win on very short segments (+1.6 % at W=64) only because it suffered less
    // from tiny segments in the middle of the tile order; with those moved to the end the two
    // shapes are level at W=64 and W=128 and one workgroup per tile is ahead everywhere else
    // (W=16: +1.5 %, W=32: +0.9 %), and it is the shape that co-runs with compute kernels
    // without starving them. A persistent grid is never used for ragged launches (a lone
    // workgroup that straddles lines or meets heads, tails and padding falls behind: -7 % on
    // 16 B aligned uneven shards) nor for other dtype pairs than 16-bit gradients into fp32.
    const auto ragged = [&] {
      bool any = !(gb == 2 && ab == 4);
      for (uint32_t k = 0; k < L.tt.n_items; ++k)
        any |= (L.item[k].acc_off & 127u) != 0 || ((L.item[k].seg_elems * ab) & 127u) != 0 ||
               ((L.item[k].seg_elems * gb) & 127u) != 0 || ((uintptr_t)L.item[k].grad & 127u) != 0 ||
               L.item[k].grad_elems != L.item[k].seg_elems * a->world;
      return any;
    };
    L.tt.resident_below = L.policy.read ? 0 : resident_below(a, opt, opt.resident_accumulation_bytes);
    int64_t blocks_per_cu = store ? opt.store_blocks_per_cu : opt.accum_blocks_per_cu;
    if (blocks_per_cu < 0)
      blocks_per_cu = whole_tiles < (uint64_t)opt.accum_persistent_below_tiles * segments ? 1 : 0;
    const uint32_t threads = accum_threads(grad_dtype, acc_dtype, store, L.policy, L.form);
    const uint32_t grid = grid_for(a, blocks_per_cu, L.tt.n_tiles, threads, ragged);
    const int64_t cap = store ? opt.store_resident_cap : opt.accum_resident_cap;
    const uint32_t lds = lds_claim_for(a, cap, grid, L.tt.n_tiles);
    if (int rc = launch_tiles(a, L, grid, [&] {
          return odc_device::launch_accum(grad_dtype, acc_dtype, store, L, grid, lds, stream);
        }))
      return rc;
  }
  return ODC_OK;
}

}  // namespace

extern "C" {

int odc_scatter_accumulate(odc_arena* a, const odc_accum_item* items, uint32_t n_items,
                           int grad_dtype, int acc_dtype, void* stream) {
  return scatter_launch(a, items, n_items, grad_dtype, acc_dtype, stream, false);
}

int odc_scatter_store(odc_arena* a, const odc_accum_item* items, uint32_t n_items, int grad_dtype,
                      int acc_dtype, void* stream) {
  return scatter_launch(a, items, n_items, grad_dtype, acc_dtype, stream, true);
}

int odc_publish(odc_arena* a, uint32_t rank, const odc_publish_item* items, uint32_t n_items,
                int acc_dtype, int out_dtype, float divisor, void* stream) {
  DeviceGuard guard;
  if (int rc = check_compute(a, guard)) return rc;
  if (n_items && !items) return fail(ODC_ERR_INVALID, "items is NULL");
  if (rank >= a->world) return fail(ODC_ERR_INVALID, "rank %u >= world size %u", rank, a->world);
  const int ab = dtype_bytes(acc_dtype), ob = dtype_bytes(out_dtype);
  if (!ab || !ob) return fail(ODC_ERR_INVALID, "unknown dtype code (acc %d, out %d)", acc_dtype, out_dtype);
  if (!(divisor == divisor) || divisor == 0.0f) return fail(ODC_ERR_INVALID, "divisor must be a non-zero number");
  if (!odc_device::has_publish(acc_dtype, out_dtype))
    return fail(ODC_ERR_UNSUPPORTED, "publish from dtype %d into dtype %d is not implemented", acc_dtype, out_dtype);
  uint8_t* region = a->origin + (uint64_t)rank * a->rank_stride;
  for (uint32_t i = 0; i < n_items; ++i) {
    const odc_publish_item& it = items[i];
    if (it.elems == 0) continue;
    if (it.elems > a->bytes_per_rank / ab)
      return fail(ODC_ERR_INVALID, "item %u: %llu elements exceed the rank region", i, (unsigned long long)it.elems);
    if (it.acc_offset % ab || (uintptr_t)it.out % ob)
      return fail(ODC_ERR_INVALID, "item %u: acc_offset or out is not aligned to its dtype", i);
    if (int rc = check_rank_range(a, "item", i, it.acc_offset, it.elems * ab)) return rc;
    if (it.out) {
      const uint8_t* o0 = static_cast<const uint8_t*>(it.out);
      const uint8_t* s0 = region + it.acc_offset;
      if (o0 < s0 + it.elems * ab && s0 < o0 + it.elems * ob)
        return fail(ODC_ERR_INVALID, "item %u: out overlaps the accumulation it is published from", i);
    }
  }
  const Options opt = options_snapshot();
  uint32_t next = 0;
  while (next < n_items) {
    PublishLaunch L;
    L.base = region;
    L.rank_stride = 0;
    L.scale.divisor = divisor;
    L.scale.divide = divisor != 1.0f;
    L.scale.reciprocal = 1.0f;
    // Dividing by a power of two whose reciprocal is a normal number is the same correctly
    // rounded result as multiplying by that reciprocal (both round one exact real value), and
    // costs one instruction instead of the division sequence.
    int exponent = 0;
    if (L.scale.divide && std::fabs(std::frexp(divisor, &exponent)) == 0.5f && exponent > -120 && exponent < 120) {
      L.scale.reciprocal = 1.0f / divisor;
      L.scale.divide = 2;
    }
    L.tt.order = kItemMajor;
    L.tt.first_rank = 0;
    const auto units = [&](uint32_t i) { return items[i].elems; };
    const LaunchSize size = launch_size<kTileElems>(n_items, next, units);
    const TileForm cut = publish_in_short_tiles(size, ab) ? kShortTiles : kWholeTiles;
    const int n = fill_launch<kTileElems>(
        L.tt, 1u, n_items, &next, cut, units,
        [&](uint32_t slot, uint32_t i) {
          L.item[slot] = {static_cast<uint8_t*>(items[i].out), items[i].acc_offset, items[i].elems};
        });
    if (n < 0) return n;
    if (n == 0) continue;
    L.form = table_form(cut, L.tt.n_tiles, opt.few_tiles);
    // one workgroup per tile: the division sequence wants the occupancy, and the launch is short
    const uint32_t grid = grid_for(a, opt.publish_blocks_per_cu, L.tt.n_tiles, publish_threads(L.form));
    const uint32_t lds = lds_claim_for(a, opt.publish_resident_cap, grid, L.tt.n_tiles);
    if (int rc = launch_tiles(a, L, grid, [&] {
          return odc_device::launch_publish(acc_dtype, out_dtype, L, grid, lds, stream);
        }))
      return rc;
  }
  return ODC_OK;
}

}  // extern "C"
