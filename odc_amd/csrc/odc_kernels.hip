// odc_kernels.hip — the device side of libodc_hip.so for gfx950 (MI355X, CDNA4): the kernels and
// the few HIP runtime calls behind namespace odc_device (odc_launch.h). The C ABI, the symmetric
// arena, validation and launch planning are in odc_host.cpp.
//
// Five streaming kernels, all HBM-bandwidth bound (no MFMA, no LDS):
//   gather_kernel       : W shard regions -> one flat buffer          (read 1 B + write 1 B per byte)
//   cast_gather_kernel  : the same with a dtype conversion on the way (fp32 -> bf16: 6 B per element),
//                         into one buffer or into every rank's own region (the conversion pass)
//   accum_kernel        : acc_r += widen(grad chunk r), in place      (bf16 -> fp32: 10 B per element)
//                         or acc_r = +0 + widen(grad chunk r), acc not read          (6 B per element)
//   clear_kernel        : zero a span in every rank region            (write 1 B per byte)
//   publish_kernel      : one rank's acc /= divisor, plus a cast copy (end of a minibatch)
//
// Launch model shared by the kernels: the work of one launch is cut into tiles of 1024 vectors
// (16 KiB), done by workgroups of 256 threads or 512 (odc_launch.h says which), or into short tiles of 256
// vectors, done by 128 threads (64 where most are part-empty, kTinyTiles): launches of short segments
// (wants_short_tiles in odc_host.cpp) and every accumulate and store of 16-bit gradients into fp32
// (accum_streams_short in odc_launch.h), every publish of fp32 accumulations (publish_in_short_tiles in
// odc_host.cpp), and long streams (stream_form there).
// Workgroups walk the tiles with a grid-stride loop, by default one workgroup per tile, so that,
// at any instant, the whole chip streams one compact window of memory. Per-item
// descriptors (<= ODC_MAX_ITEMS_PER_LAUNCH; launches of one item and of up to 16 have smaller tables) travel
// BY VALUE in the kernel argument segment and are read with scalar loads, so a call needs no device-side
// work list, no host->device copy and no allocation; longer item lists are split over several launches.
//
// Each wavefront issues its 2 or 4 independent 128-bit loads per stream before the first store.
// Streams larger than the 256 MB last-level cache are nontemporal on both sides (worth ~15 % over
// plain accesses there); what fits the cache and was just produced, or is about to be consumed, is
// left in it (cache_policy in odc_host.cpp), written through the L2s from 3 MiB on (output_form and those after it
// there), and so is a part of what does not fit (resident_below there). Deeper unrolling or prefetching the next
// tile measured slower: the memory system prefers a small window to more requests in flight.
// Workgroup i runs on XCD i % 8; binding XCDs to address classes (256 B .. 64 KiB granules)
// changed nothing measurable and giving every XCD one contiguous eighth of the tiles costs the
// read-modify-write 3 %, so tiles are simply dealt out in address order: at any instant all
// eight XCDs work side by side in one window of memory.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <iterator>
#include <type_traits>

#include "odc_hip.h"
#include "odc_launch.h"
#include "odc_tiles.h"

namespace {

// ------------------------------------------------------------------------------------------------
// device side
// ------------------------------------------------------------------------------------------------
using namespace odc_tiles;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));

using namespace odc_launch;

// The read side of a tile takes whatever misalignment the written side's alignment leaves it
// with; these typedefs tell the compiler so.
typedef u32x4 u32x4_u __attribute__((aligned(1)));
typedef u32x2 u32x2_u __attribute__((aligned(1)));

template <class V> struct Unaligned;
template <> struct Unaligned<u32x4> { typedef u32x4_u type; };
template <> struct Unaligned<u32x2> { typedef u32x2_u type; };

// An address in device memory. Of an address that comes as an argument of a function, or as a number,
// the compiler must assume that it may lie in LDS or scratch, and it takes the slower flat accesses.
template <class P>
__device__ __forceinline__ P* as_global(P* p) {
  return (P*)(__attribute__((address_space(1))) P*)(uintptr_t)p;
}

// The same of an address that all lanes agree on, in scalar registers: an access to it plus a 32-bit
// lane offset then needs no vector arithmetic of its own.
template <class P>
__device__ __forceinline__ P* scalar_base(P* p) {
  uintptr_t a = (uintptr_t)p;
  asm("" : "+s"(a));
  return as_global((P*)a);
}

// Calls body(std::true_type) or body(std::false_type). The two differ in the cache policy of some
// accesses and in nothing else, and the compiler would make one of them and drop the policy, so one side
// begins and ends with something that the other has not.
template <class Body>
__device__ __forceinline__ void with_policy(bool resident, Body body) {
  if (resident) {
    asm volatile("" ::: "memory");
    body(std::true_type{});
    asm volatile("" ::: "memory");
  } else {
    body(std::false_type{});
  }
}

// kCached: a plain access, which leaves its line in the caches; otherwise nontemporal. Which one a
// stream of a launch takes is the host's choice (cache_policy in odc_host.cpp).
template <bool kCached, class V>
__device__ __forceinline__ V load_any(const uint8_t* p) {  // any alignment
  const auto* q = reinterpret_cast<const typename Unaligned<V>::type*>(p);
  if constexpr (kCached) return *q; else return __builtin_nontemporal_load(q);
}

template <bool kCached, class V>
__device__ __forceinline__ V load_vec(const V* p) {  // aligned
  if constexpr (kCached) return *p; else return __builtin_nontemporal_load(p);
}

template <bool kCached, class V>
__device__ __forceinline__ void store_vec(V* p, V v) {  // aligned
  if constexpr (kCached) *p = v; else __builtin_nontemporal_store(v, p);
}

// A whole tile of a gather's output, converted or not, of a clear or of accumulations: vector `i` of the kVecs that
// start at `tile`, an address that all lanes agree on. What the next kernel is to find in the last-level cache is
// written through the L2 (output_form, accumulation_form, store_output_form, cast_output_form and clear_form in
// odc_host.cpp say from which size on): left in it by plain stores it goes to memory only at the kernel's end or as
// other lines push it out, between the reads of whatever runs next. us, nontemporal / plain / written through (a
// decoder layer's nine parameters, bf16, W = 8, three sets of buffers in turn):
//   gather alone: 35 MiB of output 14.4 / 15.7 / 13.2, 48 MiB 18.6 / 16.7 / 15.4;
//   an accumulate behind it, nothing reads the output: 32.1 / 31.9 / 29.4, 40.4 / 41.7 / 41.1;
//   the products that read the parameters behind it (1024 tokens): 141 / 129 / 126.5, 184 / 160 / 158.5.
constexpr int kSc1 = 16;  // of a buffer store: write through
template <OutputForm kForm, uint32_t kVecs, class V>
__device__ __forceinline__ void store_output(V* tile, uint32_t i, V v) {
  if constexpr (kForm == kWriteThrough) {
    const auto buffer = __builtin_amdgcn_make_buffer_rsrc(tile, 0, kVecs * sizeof(V), 0x00027000);
    if constexpr (sizeof(V) == 16) __builtin_amdgcn_raw_buffer_store_b128(v, buffer, (int)(i * 16), 0, kSc1);
    else __builtin_amdgcn_raw_buffer_store_b64(v, buffer, (int)(i * 8), 0, kSc1);
  } else {
    store_vec<kForm == kKeep>(tile + i, v);
  }
}

// ---- finding a tile's work ------------------------------------------------------------------
// The walk of a workgroup over the tiles of its launch; all its lanes come along.
template <class Launch>
struct TableWalk {
  typedef typename Launch::Desc Desc;
  static constexpr bool kOneTile = false;
  TileCursor cur;
  Desc it = {};  // the item of the tile located last

  __device__ __forceinline__ explicit TableWalk(const Launch&) {}
  __device__ __forceinline__ uint32_t n_tiles(const Launch& launch) const { return launch.tt.n_tiles; }
  __device__ __forceinline__ uint32_t resident_below(const Launch& launch) const { return launch.tt.resident_below; }
  __device__ __forceinline__ uint8_t* region(const Launch& launch, uint32_t rank) const {
    return launch.base + (uint64_t)rank * launch.rank_stride;
  }
  template <uint32_t>
  __device__ __forceinline__ TileCoord locate(const Launch& launch, uint32_t t) {
    if (!cursor_holds(cur, t)) {
      cursor_seek(launch.tt, t, cur);
      it = launch.item[cur.item];  // issued together with the loads of cursor_enter
      cursor_enter(launch.tt, cur);
    }
    return cursor_coord(launch.tt, cur, t);
  }
};

// A launch of one item: a small one is a chain of memory latencies, a third of which was reading
// the arguments in four dependent steps, from memory that no cache has seen. Here all of them are
// read at once. Kernel times, us: gather and accumulate of a 4096-element vector at W = 8 3.0 -> 2.5
// and 3.4 -> 2.8 (an empty kernel takes 1.4); gather, accumulate and publish of 4 Mi elements at
// W = 4 4.6 -> 3.9, 7.1 -> 6.8, 5.2 -> 4.7. Launches of hundreds of megabytes are level.
template <class D>
struct SingleWalk {
  typedef D Desc;
  static constexpr bool kOneTile = true;
  TileHead tt;
  uint8_t* base;
  uint64_t rank_stride;
  Desc it;

  __device__ __forceinline__ explicit SingleWalk(const SingleLaunch<D>& launch) {
    static_assert(sizeof(D) % 8 == 0 && sizeof(D) >= 16 && sizeof(D) <= 32, "2 to 4 words");
    constexpr int kWords = sizeof(D) / 8;
    tt = launch.tt;
    uint64_t b = (uint64_t)(uintptr_t)launch.base, stride = launch.rank_stride;
    uint64_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < kWords; ++i) w[i] = reinterpret_cast<const uint64_t*>(launch.item)[i];
    // (left alone, the compiler reads each value where it is first used)
    asm volatile("" : "+s"(tt.world), "+s"(tt.order), "+s"(tt.first_rank), "+s"(tt.tiles_per_rank), "+s"(tt.resident_below),
                      "+s"(b), "+s"(stride), "+s"(w[0]), "+s"(w[1]), "+s"(w[2]), "+s"(w[3]));
    base = as_global(reinterpret_cast<uint8_t*>((uintptr_t)b));
    rank_stride = stride;
    __builtin_memcpy(&it, w, sizeof(D));
  }
  __device__ __forceinline__ uint32_t resident_below(const SingleLaunch<D>&) const { return tt.resident_below; }
  __device__ __forceinline__ uint8_t* region(const SingleLaunch<D>&, uint32_t rank) const {
    return base + (uint64_t)rank * rank_stride;
  }
  template <uint32_t>
  __device__ __forceinline__ TileCoord locate(const SingleLaunch<D>&, uint32_t t) const { return single_item_coord(tt, t); }
};
// Few short tiles of several items (table_form in odc_host.cpp): again a chain of latencies, the binary
// search being most of it. The whole prefix table is read together with the header instead, one entry
// per lane (two for its second half), and the item found by counting the entries that are not greater
// than the tile's position:
// two round trips to the item in place of up to nine.
template <class Launch>
struct FewTilesWalk {
  typedef typename Launch::Desc Desc;
  static constexpr bool kOneTile = false;
  TileHead tt;
  uint8_t* base;
  uint64_t rank_stride;
  TileCursor cur;
  Desc it = {};
  uint32_t bound[2];  // lane l: seg_prefix[1 + l] and seg_prefix[65 + l]

  __device__ __forceinline__ explicit FewTilesWalk(const Launch& launch) {
    static_assert(kMaxItems > 64 && kMaxItems <= 128, "two prefix entries per lane of a wavefront");
    const uint32_t lane = threadIdx.x & 63u;
    bound[0] = launch.tt.seg_prefix[1 + lane];
    bound[1] = launch.tt.seg_prefix[65 + lane < kMaxItems ? 65 + lane : kMaxItems];
    tt = launch.tt;
    uint64_t b = (uint64_t)(uintptr_t)launch.base, stride = launch.rank_stride;
    asm volatile("" : "+s"(tt.world), "+s"(tt.n_tiles), "+s"(tt.order), "+s"(tt.first_rank), "+s"(tt.tiles_per_rank), "+s"(b), "+s"(stride),
                      "+v"(bound[0]), "+v"(bound[1]));
    base = as_global(reinterpret_cast<uint8_t*>((uintptr_t)b));
    rank_stride = stride;
  }
  __device__ __forceinline__ uint32_t n_tiles(const Launch&) const { return tt.n_tiles; }
  // No resident part: the second body that it takes costs each of these launches some 0.2 us (two microbatches
  // of 33 items, 5.3 M elements in all, at W = 4 26.1 -> 27.4 us, 300 small slices at W = 16 35.2 -> 36.3).
  __device__ __forceinline__ uint32_t resident_below(const Launch&) const { return 0; }
  __device__ __forceinline__ uint8_t* region(const Launch&, uint32_t rank) const {
    return base + (uint64_t)rank * rank_stride;
  }
  template <uint32_t>
  __device__ __forceinline__ TileCoord locate(const Launch& launch, uint32_t t) {
    if (!cursor_holds(cur, t)) {
      const uint32_t x = cursor_position(tt, t, cur);
      // (entries past the last item, the doubled ones among them, hold tiles_per_rank > x)
      cur.item = (uint32_t)__popcll(__ballot(bound[0] <= x)) + (uint32_t)__popcll(__ballot(bound[1] <= x));
      it = launch.item[cur.item];
      cursor_bounds(tt, launch.tt.seg_prefix[cur.item], launch.tt.seg_prefix[cur.item + 1], cur);
    }
    return cursor_coord(tt, cur, t);
  }
};

// 2 to kFewItems items, one workgroup per tile, tiles of any size. From its arguments to its first load a
// workgroup went through eight dependent round trips (two for the header, the binary search, the item) and
// some 350 scalar instructions, about 1 us of which every short launch is made and which the rest of a
// long one has to hide. Here header and table are read at once, into scalar registers, the item is found
// by counting there, and the tiles of a rank segment follow from its size: two round trips and some 200
// instructions, with one division instead of three and no loop around the tile. Graph-replayed launches of
// nine items at W = 8, us, gather / accumulate / publish of bf16 into fp32 by elements per rank and item:
// 4096 2.49 / 2.72 / 2.55 -> 2.43 / 2.70 / 2.36, 30 000 3.59 / 4.47 / 2.71 -> 3.38 / 4.42 / 2.60, 300 000
// 13.5 / 31.9 / 5.8 -> 13.0 / 30.2 / 5.75, 3 M (HBM bound) level; converting gather 30 000 4.36 -> 4.05.
// Up to kSomeItems items have four such tables behind one of their first entries: one round trip more.
template <class Launch, uint32_t kItems>
struct ItemsWalk {
  typedef typename Launch::Desc Desc;
  static constexpr bool kOneTile = true;
  TileHead tt;
  uint8_t* base;
  uint64_t rank_stride;
  Desc it = {};
  u32x16 before;        // of the only block
  u32x4 block_before;   // of several

  __device__ __forceinline__ explicit ItemsWalk(const Launch& launch) {
    static_assert(kFewItems == 16 && (kItems == kFewItems || kItems == 4 * kFewItems), "one scalar load");
    if constexpr (kItems == kFewItems) __builtin_memcpy(&before, launch.tt.tiles_before, sizeof(before));
    else __builtin_memcpy(&block_before, launch.tt.block_before, sizeof(block_before));
    tt = launch.tt;
    uint64_t b = (uint64_t)(uintptr_t)launch.base, stride = launch.rank_stride;
    asm volatile("" : "+s"(tt.world), "+s"(tt.order), "+s"(tt.first_rank), "+s"(tt.tiles_per_rank), "+s"(tt.resident_below),
                      "+s"(b), "+s"(stride));
    if constexpr (kItems == kFewItems) asm volatile("" : "+s"(before));
    else asm volatile("" : "+s"(block_before));
    base = as_global(reinterpret_cast<uint8_t*>((uintptr_t)b));
    rank_stride = stride;
  }
  __device__ __forceinline__ uint32_t resident_below(const Launch&) const { return tt.resident_below; }
  __device__ __forceinline__ uint8_t* region(const Launch&, uint32_t rank) const {
    return base + (uint64_t)rank * rank_stride;
  }
  template <uint32_t kUnits>
  __device__ __forceinline__ TileCoord locate(const Launch& launch, uint32_t t) {
    ItemsTile f = items_position(tt, t);
    if constexpr (kItems != kFewItems) {
      f.item = kFewItems * count_before<4>(block_before, f.position);
      __builtin_memcpy(&before, launch.tt.tiles_before + f.item, sizeof(before));
    }
    f.item += count_before<kFewItems>(before, f.position);
    it = launch.item[f.item];
    return items_coord(tt, f, launch.tt.tiles_before[f.item], (uint32_t)tiles_for(it.units(), kUnits));
  }
};

// The walk that goes with a launch's kind of table.
template <class Launch, bool kFew, class Table = decltype(Launch::tt)> struct WalkOf;
template <class Launch, bool kFew> struct WalkOf<Launch, kFew, TileHead> { typedef SingleWalk<typename Launch::Desc> type; };
template <class Launch, bool kFew, uint32_t kItems>
struct WalkOf<Launch, kFew, ItemsTable<kItems>> { typedef ItemsWalk<Launch, kItems> type; };
template <class Launch> struct WalkOf<Launch, false, TileTable> { typedef TableWalk<Launch> type; };
template <class Launch> struct WalkOf<Launch, true, TileTable> { typedef FewTilesWalk<Launch> type; };
template <class Launch, bool kFew = false> using TileWalk = typename WalkOf<Launch, kFew>::type;

// Calls body(tile) for the tiles of this workgroup: one of as many as there are tiles has its own.
template <class Walk, class Launch, class Body>
__device__ __forceinline__ void each_tile(const Walk& walk, const Launch& launch, Body body) {
  if constexpr (Walk::kOneTile)
    body(blockIdx.x);
  else
    for (uint32_t t = blockIdx.x; t < walk.n_tiles(launch); t += gridDim.x) body(t);
}

// Keeps a kernel at no more than so many wavefronts per SIMD: the compiler has it claim the registers of the
// others. kStreamWaves: stream_form in odc_host.cpp. kMostWaves asks for nothing: as a lower bound it would
// have the compiler spill.
#define ODC_RESIDENT_WAVES(n) __attribute__((amdgpu_waves_per_eu((n) < kMostWaves ? (n) : 1, n)))
constexpr int kMostWaves = 8, kStreamWaves = 6;

// ---- gather -------------------------------------------------------------------------------
// The bytes of a segment's head that one of T lanes moves.
template <int T> constexpr int kHeadBytes = (ODC_BODY_ALIGN - 2) / T + 1;
static_assert(kHeadBytes<kTinyThreads> * kTinyThreads >= ODC_BODY_ALIGN - 1 &&
                  kHeadBytes<kShortThreads> * kShortThreads >= ODC_BODY_ALIGN - 1,
              "every byte of a head has a lane");

// Everything of a tile that is not a run of T * U whole vectors: the last partial run, the
// head and the tail. Kept out of line so that the streaming loop stays tight (inline, the
// short-segment kernels, which come here for most of their tiles, were 5 % slower too).
template <bool kSrcCached, bool kDstCached, int T, int U>
__device__ __attribute__((noinline)) void gather_edges(uint8_t* d, const uint8_t* s, uint32_t chunk, SegShape g) {
  d = as_global(d);
  s = as_global(s);
  // Every load of the tile is issued before its first store (a lone resident workgroup would
  // otherwise pay one memory round trip per vector).
  const uint32_t tid = threadIdx.x;
  const TileWork w = tile_work<T * U>(chunk, g);
  const uint32_t left = is_whole<T * U>(w) ? 0u : w.nv;
  const uint8_t* sb = s + g.head + w.v0 * 16;
  u32x4* db = reinterpret_cast<u32x4*>(d + g.head) + w.v0;
  const bool do_tail = w.tail && tid < g.tail;
  const uint64_t tail_at = g.head + g.nvec * 16 + tid;
  const uint32_t head = w.head ? g.head : 0u;
  constexpr int kHead = kHeadBytes<T>;
  u32x4 v[U];
  uint8_t head_byte[kHead] = {}, tail_byte = 0;
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u * T + tid < left) v[u] = load_any<kSrcCached, u32x4>(sb + (size_t)(u * T + tid) * 16);
#pragma unroll
  for (int h = 0; h < kHead; ++h)
    if (h * T + tid < head) head_byte[h] = s[h * T + tid];
  if (do_tail) tail_byte = s[tail_at];
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (u * T + tid < left) store_vec<kDstCached>(db + u * T + tid, v[u]);
#pragma unroll
  for (int h = 0; h < kHead; ++h)
    if (h * T + tid < head) d[h * T + tid] = head_byte[h];
  if (do_tail) d[tail_at] = tail_byte;
}

// T threads do a tile of T * U vectors in one step; the copies stream best from 512-thread
// workgroups, of which 4 fit a CU.
template <class Launch, bool kSrcCached, OutputForm kDst, bool kFew, int T, int U, int kWaves = kMostWaves>
__global__ __launch_bounds__(T) ODC_RESIDENT_WAVES(kWaves) void gather_kernel(const Launch launch) {
  constexpr uint32_t kVecs = T * U;
  static_assert(kVecs == kTileVecs || kVecs == kShortTileVecs, "a whole tile or a short one");
  const uint32_t tid = threadIdx.x;
  TileWalk<Launch, kFew> walk(launch);
  each_tile(walk, launch, [&](uint32_t t) {
    const TileCoord c = walk.template locate<kVecs * 16>(launch, t);
    const GatherDesc it = walk.it;
    const uint64_t seg = it.seg_bytes;
    const uint8_t* s = walk.region(launch, c.rank) + it.src_off;
    uint8_t* d = as_global(it.dst) + (uint64_t)c.rank * seg;
    const SegShape g = seg_shape<kVecs>((uintptr_t)d, seg, 1, 16);
    const TileWork w = tile_work<kVecs>(c.chunk, g);
    if (is_whole<kVecs>(w)) {
      const uint8_t* sb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) sb[u] = scalar_base(s + g.head + (w.v0 + u * T) * 16);
      u32x4* db = scalar_base(reinterpret_cast<u32x4*>(d + g.head) + w.v0);
      with_policy(kSrcCached || is_resident((uintptr_t)(s + g.head + w.v0 * 16), walk.resident_below(launch)), [&](auto cached) {
        u32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = load_any<cached, u32x4>(sb[u] + tid * 16);
        // a whole tile that also owns its segment's head or tail (the first and last tile of a
        // ragged segment) reads those bytes with the same round trip as its vectors
        const bool do_tail = w.tail && tid < g.tail;
        const uint64_t tail_at = g.head + g.nvec * 16 + tid;
        const uint32_t head = w.head ? g.head : 0u;
        constexpr int kHead = kHeadBytes<T>;
        uint8_t head_byte[kHead] = {}, tail_byte = 0;
#pragma unroll
        for (int h = 0; h < kHead; ++h)
          if (h * T + tid < head) head_byte[h] = s[h * T + tid];
        if (do_tail) tail_byte = s[tail_at];
#pragma unroll
        for (int u = 0; u < U; ++u) store_output<kDst, kVecs>(db, u * T + tid, v[u]);
#pragma unroll
        for (int h = 0; h < kHead; ++h)
          if (h * T + tid < head) d[h * T + tid] = head_byte[h];
        if (do_tail) d[tail_at] = tail_byte;
      });
    } else if (has_edges<kVecs>(w)) {
      gather_edges<kSrcCached, kDst != kStream, T, U>(d, s, c.chunk, g);
    }
  });
}

// ---- clear --------------------------------------------------------------------------------
// Written through the L2s into the last-level cache, which is where the next accumulate finds the zeros: with
// plain stores the lines that the L2s hold at the end still have to leave them, which the kernel's last
// microsecond went to. Longer clears than that cache holds (clear_form in odc_host.cpp) have plain stores,
// which leave their end in the L2s. Nontemporal ones are behind both.
__device__ __attribute__((noinline)) void clear_edges(uint8_t* d, uint32_t chunk, SegShape g) {
  static_assert(kThreads >= ODC_BODY_ALIGN - 1, "one lane per head byte");
  d = as_global(d);
  const u32x4 zero = {0u, 0u, 0u, 0u};
  const uint32_t tid = threadIdx.x;
  const TileWork w = tile_work(chunk, g);
  if (!is_whole(w)) {
    u32x4* db = reinterpret_cast<u32x4*>(d + g.head) + w.v0;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      if (u * kThreads + tid < w.nv) db[u * kThreads + tid] = zero;
  }
  if (w.head && tid < g.head) d[tid] = 0;
  if (w.tail && tid < g.tail) d[g.head + g.nvec * 16 + tid] = 0;
}

template <class Launch, OutputForm kDst>
__global__ __launch_bounds__(kThreads) void clear_kernel(const Launch launch) {
  const u32x4 zero = {0u, 0u, 0u, 0u};
  const uint32_t tid = threadIdx.x;
  TileWalk<Launch> walk(launch);
  each_tile(walk, launch, [&](uint32_t t) {
    const TileCoord c = walk.template locate<kTileBytes>(launch, t);
    const ClearDesc it = walk.it;
    uint8_t* d = walk.region(launch, c.rank) + it.off;
    const SegShape g = seg_shape((uintptr_t)d, it.seg_bytes, 1, 16);
    const TileWork w = tile_work(c.chunk, g);
    if (is_whole(w)) {
      u32x4* db = scalar_base(reinterpret_cast<u32x4*>(d + g.head) + w.v0);
      if constexpr (kDst == kWriteThrough) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) store_output<kWriteThrough, kTileVecs>(db, u * kThreads + tid, zero);
      } else {
        const uint32_t below = walk.resident_below(launch);
        with_policy(!below || is_resident((uintptr_t)db, below), [&](auto cached) {
#pragma unroll
          for (int u = 0; u < kUnroll; ++u) store_vec<cached>(db + u * kThreads + tid, zero);
        });
      }
    }
    if (has_edges(w)) clear_edges(d, c.chunk, g);
  });
}

// ---- scatter-accumulate -------------------------------------------------------------------
// Element codecs. Widening to fp32 is exact for all three types; narrowing rounds to nearest
// even. The add itself is one v_add_f32 per element: no contraction, no reassociation.
struct bf16_tag {};
struct f16_tag {};
struct f32_tag {};

template <class T> struct Codec;
template <> struct Codec<f32_tag> {
  static constexpr int kBytes = 4;
  typedef uint32_t raw_t;
  static __device__ __forceinline__ float widen(uint32_t r) { return __uint_as_float(r); }
  static __device__ __forceinline__ uint32_t narrow(float f) { return __float_as_uint(f); }
};
template <> struct Codec<bf16_tag> {
  static constexpr int kBytes = 2;
  typedef uint16_t raw_t;
  static __device__ __forceinline__ float widen(uint16_t r) { return __uint_as_float((uint32_t)r << 16); }
  static __device__ __forceinline__ uint16_t narrow(float f) {
    const uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;  // NaN
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
  }
};
template <> struct Codec<f16_tag> {
  static constexpr int kBytes = 2;
  typedef uint16_t raw_t;
  static __device__ __forceinline__ float widen(uint16_t r) {
    return (float)__builtin_bit_cast(_Float16, r);
  }
  static __device__ __forceinline__ uint16_t narrow(float f) {
    return __builtin_bit_cast(uint16_t, (_Float16)f);
  }
};

// Four consecutive elements as raw dwords: 2 dwords for the 16-bit types, 4 for fp32.
template <class T> struct Quad;
template <> struct Quad<f32_tag> {
  typedef u32x4 vec_t;
  static __device__ __forceinline__ void widen(vec_t r, float (&f)[4]) {
    f[0] = __uint_as_float(r.x); f[1] = __uint_as_float(r.y);
    f[2] = __uint_as_float(r.z); f[3] = __uint_as_float(r.w);
  }
  static __device__ __forceinline__ vec_t narrow(const float (&f)[4]) {
    vec_t r = {__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
    return r;
  }
};
template <> struct Quad<bf16_tag> {
  typedef u32x2 vec_t;
  static __device__ __forceinline__ void widen(vec_t r, float (&f)[4]) {
    f[0] = __uint_as_float(r.x << 16); f[1] = __uint_as_float(r.x & 0xffff0000u);
    f[2] = __uint_as_float(r.y << 16); f[3] = __uint_as_float(r.y & 0xffff0000u);
  }
  static __device__ __forceinline__ vec_t narrow(const float (&f)[4]) {
    vec_t r;
    r.x = (uint32_t)Codec<bf16_tag>::narrow(f[0]) | ((uint32_t)Codec<bf16_tag>::narrow(f[1]) << 16);
    r.y = (uint32_t)Codec<bf16_tag>::narrow(f[2]) | ((uint32_t)Codec<bf16_tag>::narrow(f[3]) << 16);
    return r;
  }
};
template <> struct Quad<f16_tag> {
  typedef u32x2 vec_t;
  static __device__ __forceinline__ void widen(vec_t r, float (&f)[4]) {
    f[0] = Codec<f16_tag>::widen((uint16_t)(r.x & 0xffffu)); f[1] = Codec<f16_tag>::widen((uint16_t)(r.x >> 16));
    f[2] = Codec<f16_tag>::widen((uint16_t)(r.y & 0xffffu)); f[3] = Codec<f16_tag>::widen((uint16_t)(r.y >> 16));
  }
  static __device__ __forceinline__ vec_t narrow(const float (&f)[4]) {
    vec_t r;
    r.x = (uint32_t)Codec<f16_tag>::narrow(f[0]) | ((uint32_t)Codec<f16_tag>::narrow(f[1]) << 16);
    r.y = (uint32_t)Codec<f16_tag>::narrow(f[2]) | ((uint32_t)Codec<f16_tag>::narrow(f[3]) << 16);
    return r;
  }
};

// kStore: the accumulation is taken to hold +0 and is not read (acc = +0 + g, the value a clear
// followed by an accumulate leaves: -0 gradients still become +0).
//
// The parts of a tile that are not whole runs of valid quads: a partial last run, a run that
// crosses the end of the valid gradient or lies in the zero padding, the head and the tail.
// Gradient elements at index >= grad_elems read as +0 and are still added (so an accumulation
// holding -0 becomes +0, as F.pad followed by add_ leaves it).
//
// What bounds it is latency: it runs in tiles that are alone in their segment, often with one
// workgroup on its CU. So every load of the tile is issued before the first value is used: raw
// vectors are loaded under the lane mask and widened only afterwards (widening inside the guarded
// block made the compiler wait there, one memory round trip per quad), and the one quad that the
// gradient's end may cut is read as elements by the lane that owns it. Nine items of 3 640
// elements per rank (W = 8, one partial tile each) take 3.8 us instead of 5.4, with gradients that end inside
// the last rank's segment 4.0 instead of 4.8 (13 889 elements per rank).
template <class G, class A, bool kStore, bool kGradCached, OutputForm kAcc, int T, int U>
__device__ __attribute__((noinline)) void accum_edges(uint8_t* acc, const uint8_t* grad, uint64_t g_seg,
                                                      uint64_t grad_elems, uint32_t chunk, SegShape g,
                                                      bool body) {
  constexpr bool kAccCached = kAcc != kStream;
  acc = as_global(acc);
  grad = as_global(grad);
  typedef typename Quad<G>::vec_t gvec_t;
  typedef typename Quad<A>::vec_t avec_t;
  typedef typename Codec<G>::raw_t graw_t;
  typedef typename Codec<A>::raw_t araw_t;
  constexpr uint32_t kAB = Codec<A>::kBytes, kGB = Codec<G>::kBytes;
  const uint32_t tid = threadIdx.x;
  const TileWork w = tile_work<T * U>(chunk, g);
  const uint32_t left = body ? w.nv : 0u;
  const uint64_t e0 = g.head + w.v0 * 4;
  avec_t* ap = reinterpret_cast<avec_t*>(acc + e0 * kAB);
  const graw_t* gs = reinterpret_cast<const graw_t*>(grad);
  araw_t* as = reinterpret_cast<araw_t*>(acc);
  const bool do_head = w.head && tid < g.head;
  const bool do_tail = w.tail && tid < g.tail;
  const uint64_t tail_at = g.head + g.nvec * 4 + tid;
  // valid gradient elements from the tile's first body element on: whole quads, and what is left
  const uint64_t g0 = g_seg + e0;
  const uint64_t valid = grad_elems > g0 ? grad_elems - g0 : 0;
  const uint32_t whole_quads = valid >= 4 * T * U ? T * U : (uint32_t)(valid / 4);
  const uint32_t cut = valid >= 4 * T * U ? 0u : (uint32_t)(valid & 3u);
  const bool has_cut = cut != 0 && whole_quads < left && tid == whole_quads % T;

  gvec_t graw[U] = {};
  avec_t araw[U] = {};
  graw_t cut_raw[3] = {0, 0, 0};
  graw_t head_graw = 0, tail_graw = 0;
  araw_t head_araw = 0, tail_araw = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t q = u * T + tid;
    if (q < left && q < whole_quads) graw[u] = load_any<kGradCached, gvec_t>(grad + (g0 + (uint64_t)q * 4) * kGB);
    if constexpr (!kStore) {
      if (q < left) araw[u] = load_vec<kAccCached>(ap + q);
    }
  }
  if (has_cut) {
#pragma unroll
    for (uint32_t k = 0; k < 3; ++k)
      if (k < cut) cut_raw[k] = gs[g0 + (uint64_t)whole_quads * 4 + k];
  }
  if (do_head) {
    if (g_seg + tid < grad_elems) head_graw = gs[g_seg + tid];
    if constexpr (!kStore) head_araw = as[tid];
  }
  if (do_tail) {
    if (g_seg + tail_at < grad_elems) tail_graw = gs[g_seg + tail_at];
    if constexpr (!kStore) tail_araw = as[tail_at];
  }

#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t q = u * T + tid;
    if (q < left) {
      float gf[4], af[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      Quad<G>::widen(graw[u], gf);
      if (has_cut && q == whole_quads) {
#pragma unroll
        for (int k = 0; k < 3; ++k) gf[k] = Codec<G>::widen(cut_raw[k]);
      }
      if constexpr (!kStore) Quad<A>::widen(araw[u], af);
#pragma unroll
      for (int k = 0; k < 4; ++k) af[k] = af[k] + gf[k];
      store_vec<kAccCached>(ap + q, Quad<A>::narrow(af));
    }
  }
  // (raw zero widens to +0 in every type)
  if (do_head) as[tid] = Codec<A>::narrow(Codec<A>::widen(head_araw) + Codec<G>::widen(head_graw));
  if (do_tail) as[tail_at] = Codec<A>::narrow(Codec<A>::widen(tail_araw) + Codec<G>::widen(tail_graw));
}

// kAcc: how the accumulations are written; read past the caches with kStream, through them otherwise.
template <class Launch, class G, class A, bool kStore, bool kGradCached, OutputForm kAcc, bool kFew, int T, int U,
          int kWaves = kMostWaves>
__global__ __launch_bounds__(T) ODC_RESIDENT_WAVES(kWaves) void accum_kernel(const Launch launch) {
  constexpr uint32_t kVecs = T * U;  // quads
  static_assert(kVecs == kTileVecs || kVecs == kShortTileVecs, "a whole tile or a short one");
  typedef typename Quad<G>::vec_t gvec_t;
  typedef typename Quad<A>::vec_t avec_t;
  constexpr uint32_t kAB = Codec<A>::kBytes, kGB = Codec<G>::kBytes;
  static_assert(T >= ODC_BODY_ALIGN / kAB, "one lane per head element");
  const uint32_t tid = threadIdx.x;
  TileWalk<Launch, kFew> walk(launch);
  each_tile(walk, launch, [&](uint32_t t) {
    const TileCoord c = walk.template locate<kVecs * 4>(launch, t);
    const AccumDesc it = walk.it;
    const uint64_t seg = it.seg_elems;
    uint8_t* acc = walk.region(launch, c.rank) + it.acc_off;
    const uint64_t g_seg = (uint64_t)c.rank * seg;  // gradient index of the segment's first element
    const SegShape g = seg_shape<kVecs>((uintptr_t)acc, seg, kAB, 4);
    const TileWork w = tile_work<kVecs>(c.chunk, g);
    const uint64_t e0 = g.head + w.v0 * 4;  // the tile's first body element within the segment
    // whole: all its quads exist in the accumulation AND in the valid part of the gradient
    const bool whole = is_whole<kVecs>(w) && g_seg + e0 + 4 * kVecs <= it.grad_elems;
    if (whole) {
      const uint8_t* gb[U];
      avec_t* ap[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        gb[u] = scalar_base(it.grad + (g_seg + e0 + u * T * 4) * kGB);
        ap[u] = scalar_base(reinterpret_cast<avec_t*>(acc + e0 * kAB) + u * T);
      }
      with_policy(kAcc != kStream || is_resident((uintptr_t)(acc + e0 * kAB), walk.resident_below(launch)), [&](auto cached) {
        constexpr OutputForm kWritten = kAcc == kStream && cached ? kKeep : kAcc;  // (resident parts: plain stores)
        gvec_t graw[U];
        avec_t araw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) graw[u] = load_any<kGradCached, gvec_t>(gb[u] + tid * (uint32_t)sizeof(gvec_t));
        if constexpr (!kStore) {
#pragma unroll
          for (int u = 0; u < U; ++u) araw[u] = load_vec<cached>(ap[u] + tid);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float gf[4], af[4] = {0.0f, 0.0f, 0.0f, 0.0f};
          Quad<G>::widen(graw[u], gf);
          if constexpr (!kStore) Quad<A>::widen(araw[u], af);
#pragma unroll
          for (int k = 0; k < 4; ++k) af[k] = af[k] + gf[k];
          store_output<kWritten, kVecs>(ap[0], u * T + tid, Quad<A>::narrow(af));
        }
      });
    }
    if (!whole ? (w.nv != 0 || w.head || w.tail) : (w.head || w.tail))
      accum_edges<G, A, kStore, kGradCached, kAcc, T, U>(acc, it.grad, g_seg, it.grad_elems, c.chunk, g, !whole);
  });
}

// ---- gather with cast ---------------------------------------------------------------------
// dst[r*stride + i] = narrow_D(widen_S(region_r[off + i])): the gather of shards kept in one dtype
// (fp32 master copies) into a full parameter of another (bf16), in one pass (stride = the
// segment's size: the converted segments lie back to back), or, with stride = the distance
// between rank regions and dst inside rank 0's region, the conversion of every rank's shard into
// a second symmetric buffer.
template <class S, class D, bool kSrcCached, bool kDstCached, int T, int U>
__device__ __attribute__((noinline)) void cast_edges(uint8_t* d, const uint8_t* s, uint32_t chunk, SegShape g) {
  d = as_global(d);
  s = as_global(s);
  typedef typename Quad<S>::vec_t svec_t;
  typedef typename Quad<D>::vec_t dvec_t;
  typedef typename Codec<S>::raw_t sraw_t;
  typedef typename Codec<D>::raw_t draw_t;
  constexpr uint32_t kSB = Codec<S>::kBytes, kDB = Codec<D>::kBytes;
  const uint32_t tid = threadIdx.x;
  const TileWork w = tile_work<T * U>(chunk, g);
  const uint32_t left = is_whole<T * U>(w) ? 0u : w.nv;
  const uint64_t e0 = g.head + w.v0 * 4;
  const uint8_t* sb = s + e0 * kSB;
  dvec_t* dp = reinterpret_cast<dvec_t*>(d + e0 * kDB);
  const sraw_t* ss = reinterpret_cast<const sraw_t*>(s);
  draw_t* ds = reinterpret_cast<draw_t*>(d);
  const bool do_head = w.head && tid < g.head;
  const bool do_tail = w.tail && tid < g.tail;
  const uint64_t tail_at = g.head + g.nvec * 4 + tid;
  // every load of the tile before its first store
  svec_t raw[U];
  sraw_t head_raw = 0, tail_raw = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t q = u * T + tid;
    if (q < left) raw[u] = load_any<kSrcCached, svec_t>(sb + (size_t)q * sizeof(svec_t));
  }
  if (do_head) head_raw = ss[tid];
  if (do_tail) tail_raw = ss[tail_at];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t q = u * T + tid;
    if (q < left) {
      float f[4];
      Quad<S>::widen(raw[u], f);
      store_vec<kDstCached>(dp + q, Quad<D>::narrow(f));
    }
  }
  if (do_head) ds[tid] = Codec<D>::narrow(Codec<S>::widen(head_raw));
  if (do_tail) ds[tail_at] = Codec<D>::narrow(Codec<S>::widen(tail_raw));
}

template <class Launch, class S, class D, bool kSrcCached, OutputForm kDst, bool kFew, int T, int U>
__global__ __launch_bounds__(T) void cast_gather_kernel(const Launch launch) {
  constexpr uint32_t kVecs = T * U;  // quads
  static_assert(kVecs == kTileVecs || kVecs == kShortTileVecs, "a whole tile or a short one");
  static_assert(T >= ODC_BODY_ALIGN / Codec<D>::kBytes, "one lane per head element");
  typedef typename Quad<S>::vec_t svec_t;
  typedef typename Quad<D>::vec_t dvec_t;
  constexpr uint32_t kSB = Codec<S>::kBytes, kDB = Codec<D>::kBytes;
  const uint32_t tid = threadIdx.x;
  TileWalk<Launch, kFew> walk(launch);
  each_tile(walk, launch, [&](uint32_t t) {
    const TileCoord c = walk.template locate<kVecs * 4>(launch, t);
    const CastGatherDesc it = walk.it;
    const uint64_t seg = it.seg_elems;
    const uint8_t* s = walk.region(launch, c.rank) + it.src_off;
    uint8_t* d = as_global(it.dst) + (uint64_t)c.rank * it.dst_stride;
    const SegShape g = seg_shape<kVecs>((uintptr_t)d, seg, kDB, 4);
    const TileWork w = tile_work<kVecs>(c.chunk, g);
    if (is_whole<kVecs>(w)) {
      const uint64_t e0 = g.head + w.v0 * 4;
      const uint8_t* sb = s + e0 * kSB + (size_t)tid * sizeof(svec_t);
      dvec_t* dp = reinterpret_cast<dvec_t*>(d + e0 * kDB);
      svec_t raw[U];
#pragma unroll
      for (int u = 0; u < U; ++u) raw[u] = load_any<kSrcCached, svec_t>(sb + (size_t)u * T * sizeof(svec_t));
      // the head and the tail of the segment, when this whole tile owns them, in the same round trip
      typedef typename Codec<S>::raw_t sraw_t;
      typedef typename Codec<D>::raw_t draw_t;
      const sraw_t* ss = reinterpret_cast<const sraw_t*>(s);
      draw_t* ds = reinterpret_cast<draw_t*>(d);
      const bool do_head = w.head && tid < g.head;
      const bool do_tail = w.tail && tid < g.tail;
      const uint64_t tail_at = g.head + g.nvec * 4 + tid;
      sraw_t head_raw = 0, tail_raw = 0;
      if (do_head) head_raw = ss[tid];
      if (do_tail) tail_raw = ss[tail_at];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float f[4];
        Quad<S>::widen(raw[u], f);
        store_output<kDst, kVecs>(dp, u * T + tid, Quad<D>::narrow(f));
      }
      if (do_head) ds[tid] = Codec<D>::narrow(Codec<S>::widen(head_raw));
      if (do_tail) ds[tail_at] = Codec<D>::narrow(Codec<S>::widen(tail_raw));
    } else if (has_edges<kVecs>(w)) {
      cast_edges<S, D, kSrcCached, kDst != kStream, T, U>(d, s, c.chunk, g);
    }
  });
}

// ---- publish ------------------------------------------------------------------------------
// One rank's accumulations at the end of a minibatch: acc[i] /= divisor in place (a correctly
// rounded IEEE division, rounded to the accumulation dtype) and out[i] = narrow_O(acc[i]).
template <class A>
__device__ __forceinline__ typename Codec<A>::raw_t publish_scale(typename Codec<A>::raw_t raw,
                                                                  const PublishScale& by) {
  const float x = Codec<A>::widen(raw);
  return Codec<A>::narrow(by.divide == 2 ? x * by.reciprocal : x / by.divisor);
}

// Four elements: scales `raw` in place when the launch divides and returns the cast copy.
template <class A, class O>
__device__ __forceinline__ typename Quad<O>::vec_t publish_quad(typename Quad<A>::vec_t& raw,
                                                                const PublishScale& by) {
  float f[4];
  Quad<A>::widen(raw, f);
  if (by.divide) {
    if (by.divide == 2) {
#pragma unroll
      for (int k = 0; k < 4; ++k) f[k] = f[k] * by.reciprocal;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) f[k] = f[k] / by.divisor;
    }
    raw = Quad<A>::narrow(f);
    Quad<A>::widen(raw, f);  // the copy is a cast of the ROUNDED accumulation
  }
  return Quad<O>::narrow(f);
}

// Bound by HBM in long launches, by latency and idle CUs in short ones; which tiles it takes is
// publish_in_short_tiles in odc_host.cpp. Everything is nontemporal in both forms (plain accesses: 3.1 M
// elements 7.0 -> 10.8 us, 8 Mi 15.5 -> 23.2).
template <class Launch, class A, class O, bool kFew, int T, int U>
__global__ __launch_bounds__(T) void publish_kernel(const Launch launch) {
  constexpr uint32_t kVecs = T * U, kElems = kVecs * 4;
  static_assert(kVecs == kTileVecs || kVecs == kShortTileVecs, "a whole tile or a short one");
  typedef typename Codec<A>::raw_t araw_t;
  typedef typename Codec<O>::raw_t oraw_t;
  typedef typename Quad<A>::vec_t avec_t;
  typedef typename Quad<O>::vec_t ovec_t;
  const uint32_t tid = threadIdx.x;
  TileWalk<Launch, kFew> walk(launch);
  each_tile(walk, launch, [&](uint32_t t) {
    const TileCoord c = walk.template locate<kVecs * 4>(launch, t);
    const PublishDesc it = walk.it;
    const uint64_t seg = it.seg_elems;
    const uint64_t in_seg = (uint64_t)c.chunk * kElems;
    araw_t* acc = reinterpret_cast<araw_t*>(walk.region(launch, 0) + it.acc_off) + in_seg;
    oraw_t* out = it.out ? reinterpret_cast<oraw_t*>(as_global(it.out)) + in_seg : nullptr;
    const uint64_t left = seg - in_seg;
    if (left >= kElems && (((uintptr_t)acc) & (sizeof(avec_t) - 1)) == 0 &&
        (((uintptr_t)out) & (sizeof(ovec_t) - 1)) == 0) {
      avec_t* ap = reinterpret_cast<avec_t*>(acc) + tid;
      ovec_t* op = reinterpret_cast<ovec_t*>(out) + tid;
      avec_t raw[U];
      ovec_t cast[U];
#pragma unroll
      for (int u = 0; u < U; ++u) raw[u] = __builtin_nontemporal_load(ap + u * T);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        cast[u] = publish_quad<A, O>(raw[u], launch.scale);
      }
      // The two written streams go out one after the other, not interleaved vector by vector
      // (measured: +6..12 %; plain instead of nontemporal stores for the copy change nothing then).
      if (launch.scale.divide) {
#pragma unroll
        for (int u = 0; u < U; ++u) __builtin_nontemporal_store(raw[u], ap + u * T);
      }
      if (out) {
#pragma unroll
        for (int u = 0; u < U; ++u) __builtin_nontemporal_store(cast[u], op + u * T);
      }
    } else if ((((uintptr_t)acc) & (sizeof(avec_t) - 1)) == 0 && (((uintptr_t)out) & (sizeof(ovec_t) - 1)) == 0) {
      // A partial tile (every accumulation's last one): the same vectors under a lane mask, and
      // the up to three elements behind the last whole vector. The whole tile is one memory round
      // trip; element by element it was sixteen loads per lane and stores of 2 or 4 bytes
      // (256 x 4, nine accumulations of 3 640 elements: 4.2 us instead of 5.9; of 233 016: 5.9 instead
      // of 7.3).
      const uint32_t quads = (uint32_t)left / 4, rest = (uint32_t)left & 3u;
      avec_t* ap = reinterpret_cast<avec_t*>(acc) + tid;
      ovec_t* op = reinterpret_cast<ovec_t*>(out) + tid;
      avec_t raw[U] = {};
      araw_t rest_raw = 0;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (u * T + tid < quads) raw[u] = __builtin_nontemporal_load(ap + u * T);
      if (tid < rest) rest_raw = acc[quads * 4 + tid];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (u * T + tid < quads) {
          const ovec_t cast = publish_quad<A, O>(raw[u], launch.scale);
          if (launch.scale.divide) __builtin_nontemporal_store(raw[u], ap + u * T);
          if (out) __builtin_nontemporal_store(cast, op + u * T);
        }
      }
      if (tid < rest) {
        if (launch.scale.divide) acc[quads * 4 + tid] = rest_raw = publish_scale<A>(rest_raw, launch.scale);
        if (out) out[quads * 4 + tid] = Codec<O>::narrow(Codec<A>::widen(rest_raw));
      }
    } else {
      // accumulations or outputs that are not aligned to their vectors: element by element, all
      // loads before the first store
      constexpr int kPerLane = kElems / T;
      const uint32_t n = left < kElems ? (uint32_t)left : kElems;
      araw_t raw[kPerLane];
#pragma unroll
      for (int j = 0; j < kPerLane; ++j)
        if (j * T + tid < n) raw[j] = acc[j * T + tid];
#pragma unroll
      for (int j = 0; j < kPerLane; ++j) {
        const uint32_t i = j * T + tid;
        if (i < n) {
          if (launch.scale.divide) acc[i] = raw[j] = publish_scale<A>(raw[j], launch.scale);
          if (out) out[i] = Codec<O>::narrow(Codec<A>::widen(raw[j]));
        }
      }
    }
  });
}

// ------------------------------------------------------------------------------------------------
// dtype dispatch
// ------------------------------------------------------------------------------------------------
template <class Launch> using kernel_fn = void (*)(const Launch);
// Launches of one item or of few have one way to find it: one kernel serves both short forms.
template <class Launch> constexpr bool kSearches = std::is_same_v<decltype(Launch::tt), TileTable>;
// Which launches long streams come in, and which are for nothing else.
template <class Launch> constexpr bool kStreams = !kSearches<Launch>;
template <class Launch> constexpr bool kStreamsOnly = std::is_same_v<decltype(Launch::tt), ItemsTable<kSomeItems>>;
// Gathers of whole tiles are bound by HBM and stream better from workgroups that come to their loads one
// after the other along the item search: a layer's 872 MB from bf16 134.1 us by the full tables, 136.4 by the
// small ones, from fp32 196 and 199 (fewer resident workgroups: 224). The other kernels are level there. So
// plain and converting gathers have no kernel for whole tiles by the small table.
template <class Launch>
constexpr bool kGathersWholeTiles = !std::is_same_v<decltype(Launch::tt), ItemsTable<kFewItems>>;

#define ODC_FOR_EACH_DTYPE_PAIR(X)                    \
  X(ODC_DTYPE_BF16, bf16_tag, ODC_DTYPE_BF16, bf16_tag) \
  X(ODC_DTYPE_BF16, bf16_tag, ODC_DTYPE_F16, f16_tag)   \
  X(ODC_DTYPE_BF16, bf16_tag, ODC_DTYPE_F32, f32_tag)   \
  X(ODC_DTYPE_F16, f16_tag, ODC_DTYPE_BF16, bf16_tag)   \
  X(ODC_DTYPE_F16, f16_tag, ODC_DTYPE_F16, f16_tag)     \
  X(ODC_DTYPE_F16, f16_tag, ODC_DTYPE_F32, f32_tag)     \
  X(ODC_DTYPE_F32, f32_tag, ODC_DTYPE_BF16, bf16_tag)   \
  X(ODC_DTYPE_F32, f32_tag, ODC_DTYPE_F16, f16_tag)     \
  X(ODC_DTYPE_F32, f32_tag, ODC_DTYPE_F32, f32_tag)

// (gradient dtype, accumulation dtype). Accumulations are cached only together with the gradient; by a store,
// which does not read them, only written through (store_output_form in odc_host.cpp).
template <class L, class G, class A, bool kFew, int T, int U>
kernel_fn<L> pick_rmw(AccumPolicy policy) {
  if (policy.read && policy.written == kKeep) return accum_kernel<L, G, A, false, true, kKeep, kFew, T, U>;
  if (policy.read && policy.written == kWriteThrough) return accum_kernel<L, G, A, false, true, kWriteThrough, kFew, T, U>;
  return policy.read ? accum_kernel<L, G, A, false, true, kStream, kFew, T, U>
                     : accum_kernel<L, G, A, false, false, kStream, kFew, T, U>;
}

template <class L, class G, class A, bool kFew, int T, int U, int kWaves = kMostWaves>
kernel_fn<L> pick_store(AccumPolicy policy) {
  if (policy.read && policy.written == kWriteThrough)
    return accum_kernel<L, G, A, true, true, kWriteThrough, kFew, T, U, kWaves>;
  return policy.read ? accum_kernel<L, G, A, true, true, kStream, kFew, T, U, kWaves>
                     : accum_kernel<L, G, A, true, false, kStream, kFew, T, U, kWaves>;
}

// kShortOnly: accum_streams_short says so, there is no kernel of whole tiles.
template <class L, class G, class A, bool kShortOnly>
kernel_fn<L> pick_accum_tiles(bool store, AccumPolicy policy, TileForm form);

template <class L, class G, class A, bool kShortOnly>
kernel_fn<L> pick_accum_form(bool store, AccumPolicy policy, TileForm form) {
  if (form == kStreamTiles) {  // into fp32: what scatter_stream_form in odc_host.cpp sends here
    if constexpr (kStreams<L> && Codec<A>::kBytes == 4) {
      if constexpr (Codec<G>::kBytes == 4) {
        if (store) return pick_store<L, G, A, false, kShortThreads, kShortUnroll, kStreamWaves>(policy);
        if (policy.read) return accum_kernel<L, G, A, false, true, kStream, false, kShortThreads, kShortUnroll, kStreamWaves>;
      }
      if (!store && !policy.read)
        return accum_kernel<L, G, A, false, false, kStream, false, kShortThreads, kShortUnroll, kStreamWaves>;
    }
    return nullptr;
  }
  if constexpr (kStreamsOnly<L>) return nullptr;
  else return pick_accum_tiles<L, G, A, kShortOnly>(store, policy, form);
}

template <class L, class G, class A, bool kShortOnly>
kernel_fn<L> pick_accum_tiles(bool store, AccumPolicy policy, TileForm form) {
  if constexpr (kSearches<L>)
    if (form == kTinyTiles)
      return store ? pick_store<L, G, A, true, kTinyThreads, kTinyUnroll>(policy)
                   : pick_rmw<L, G, A, true, kTinyThreads, kTinyUnroll>(policy);
  if (form == kFewShortTiles)
    return store ? pick_store<L, G, A, kSearches<L>, kShortThreads, kShortUnroll>(policy)
                 : pick_rmw<L, G, A, kSearches<L>, kShortThreads, kShortUnroll>(policy);
  if (form == kShortTiles)
    return store ? pick_store<L, G, A, false, kShortThreads, kShortUnroll>(policy)
                 : pick_rmw<L, G, A, false, kShortThreads, kShortUnroll>(policy);
  if constexpr (kShortOnly) return nullptr;
  else if constexpr (Codec<G>::kBytes == 2 && Codec<A>::kBytes == 2) {
    if (store) return pick_store<L, G, A, false, kThreads, kUnroll>(policy);
    return policy.read ? pick_rmw<L, G, A, false, kThreads, kUnroll>(policy)
                       : accum_kernel<L, G, A, false, false, kStream, false, kNarrowRmwThreads, kNarrowRmwUnroll>;
  } else
    return store ? pick_store<L, G, A, false, kStoreThreads, kStoreUnroll>(policy)
                 : pick_rmw<L, G, A, false, kThreads, kUnroll>(policy);
}

template <class L>
kernel_fn<L> pick_accum(int g, int a, bool store, AccumPolicy policy, TileForm form) {
#define X(E1, T1, E2, T2) \
  if (g == E1 && a == E2) return pick_accum_form<L, T1, T2, accum_streams_short(E1, E2)>(store, policy, form);
  ODC_FOR_EACH_DTYPE_PAIR(X)
#undef X
  return nullptr;
}

template <class L, bool kSrcCached, OutputForm kDst>
kernel_fn<L> pick_gather_form(TileForm form) {
  if constexpr (kStreams<L> && kDst == kStream && !kSrcCached)
    if (form == kStreamTiles) return gather_kernel<L, false, kStream, false, kShortThreads, kShortUnroll, kStreamWaves>;
  if constexpr (!kStreamsOnly<L>) {
    if constexpr (kSearches<L>)
      if (form == kTinyTiles) return gather_kernel<L, kSrcCached, kDst, true, kTinyThreads, kTinyUnroll>;
    if (form == kFewShortTiles) return gather_kernel<L, kSrcCached, kDst, kSearches<L>, kShortThreads, kShortUnroll>;
    if (form == kShortTiles) return gather_kernel<L, kSrcCached, kDst, false, kShortThreads, kShortUnroll>;
    if constexpr (kGathersWholeTiles<L>)
      if (form == kWholeTiles) return gather_kernel<L, kSrcCached, kDst, false, kCopyThreads, kCopyUnroll>;
  }
  return nullptr;
}

template <class L, bool kSrcCached>
kernel_fn<L> pick_gather_output(OutputForm output, TileForm form) {
  if (output == kStream) return pick_gather_form<L, kSrcCached, kStream>(form);
  if (output == kKeep) return pick_gather_form<L, kSrcCached, kKeep>(form);
  return pick_gather_form<L, kSrcCached, kWriteThrough>(form);
}

template <class L>
kernel_fn<L> pick_gather(bool shards_cached, OutputForm output, TileForm form) {
  return shards_cached ? pick_gather_output<L, true>(output, form) : pick_gather_output<L, false>(output, form);
}

template <class L, class S, class D, bool kSrcCached, OutputForm kDst>
kernel_fn<L> pick_cast_gather_form(TileForm form) {
  if constexpr (kSearches<L>)
    if (form == kTinyTiles) return cast_gather_kernel<L, S, D, kSrcCached, kDst, true, kTinyThreads, kTinyUnroll>;
  if (form == kFewShortTiles) return cast_gather_kernel<L, S, D, kSrcCached, kDst, kSearches<L>, kShortThreads, kShortUnroll>;
  if (form == kShortTiles) return cast_gather_kernel<L, S, D, kSrcCached, kDst, false, kShortThreads, kShortUnroll>;
  if constexpr (kGathersWholeTiles<L>)
    if (form == kWholeTiles) return cast_gather_kernel<L, S, D, kSrcCached, kDst, false, kCopyThreads, kCopyUnroll>;
  return nullptr;
}

// Shards are cached only together with the output.
template <class L, class S, class D>
kernel_fn<L> pick_cast_gather_output(CachePolicy policy, OutputForm output, TileForm form) {
  if (policy.read)
    return output == kKeep ? pick_cast_gather_form<L, S, D, true, kKeep>(form)
                           : pick_cast_gather_form<L, S, D, true, kWriteThrough>(form);
  return output == kStream ? pick_cast_gather_form<L, S, D, false, kStream>(form)
                           : pick_cast_gather_form<L, S, D, false, kWriteThrough>(form);
}

template <class L>
kernel_fn<L> pick_cast_gather(int s, int d, CachePolicy policy, OutputForm output, TileForm form) {  // (shard dtype, output dtype)
#define X(E1, T1, E2, T2) \
  if (s == E1 && d == E2) return pick_cast_gather_output<L, T1, T2>(policy, output, form);
  ODC_FOR_EACH_DTYPE_PAIR(X)
#undef X
  return nullptr;
}

// publish_in_short_tiles: fp32 accumulations have no kernel of whole tiles. (table_form: nor are there any of one
// wavefront.)
template <class L, class A, class O>
kernel_fn<L> pick_publish_form(TileForm form) {
  if (form == kFewShortTiles) return publish_kernel<L, A, O, kSearches<L>, kShortThreads, kShortUnroll>;
  if (form == kShortTiles) return publish_kernel<L, A, O, false, kShortThreads, kShortUnroll>;
  if constexpr (Codec<A>::kBytes == 4) return nullptr;
  else return publish_kernel<L, A, O, false, kThreads, kUnroll>;
}

template <class L>
kernel_fn<L> pick_publish(int a, int o, TileForm form) {  // (accumulation dtype, output dtype)
#define X(E1, T1, E2, T2) \
  if (a == E1 && o == E2) \
    return pick_publish_form<L, T1, T2>(form);
  ODC_FOR_EACH_DTYPE_PAIR(X)
#undef X
  return nullptr;
}

// A launch of one item, or of up to kFewItems, in its own form.
template <class Form, class Launch>
Form short_form(const Launch& L) {
  Form s;
  if constexpr (std::is_same_v<decltype(s.tt), TileHead>) s.tt = L.tt;
  else s.tt = items_table<std::size(decltype(s.tt.tiles_before){})>(L.tt);
  s.base = L.base;
  s.rank_stride = L.rank_stride;
  std::copy_n(L.item, std::min<size_t>(L.tt.n_items, std::size(s.item)), s.item);
  if constexpr (std::is_same_v<Launch, PublishLaunch>) s.scale = L.scale;
  return s;
}

// The launch's own status, not hipGetLastError(): that one also reports what an earlier,
// unrelated HIP call of the same host thread left behind.
template <class Launch>
int launch(void (*kernel)(const Launch), const Launch& L, uint32_t grid, uint32_t threads, uint32_t lds_bytes,
           void* stream) {
  if (!kernel) return (int)hipErrorInvalidDeviceFunction;
  void* args[] = {const_cast<Launch*>(&L)};
  return (int)hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(grid), dim3(threads), args, lds_bytes,
                              static_cast<hipStream_t>(stream));
}

template <class L> struct Form { typedef L type; };

// The short forms of a launch.
template <class Launch> struct ShortForms {
  typedef SingleLaunch<typename Launch::Desc> Single;
  typedef ItemsLaunch<typename Launch::Desc, kFewItems> FewItems;
  typedef ItemsLaunch<typename Launch::Desc, kSomeItems> SomeItems;
};
template <> struct ShortForms<PublishLaunch> {
  typedef PublishSingle Single;
  typedef PublishFewItems FewItems;
};

// pick(Form<L>) names the kernel for launches of type L. by_table: several items take the full tables,
// however few they are.
template <class Launch, class Pick>
int launch_form(const Launch& L, uint32_t grid, uint32_t threads, uint32_t lds_bytes, void* stream, Pick pick,
                bool by_table = false) {
  const auto issue = [&](const auto& form) {
    typedef std::remove_cv_t<std::remove_reference_t<decltype(form)>> F;
    return launch<F>(pick(Form<F>{}), form, grid, threads, lds_bytes, stream);
  };
  if (grid != L.tt.n_tiles) return issue(L);  // workgroups of more than one tile walk the full tables
  if (L.tt.n_items == 1) return issue(short_form<typename ShortForms<Launch>::Single>(L));
  if (L.tt.n_items <= kFewItems && !by_table) return issue(short_form<typename ShortForms<Launch>::FewItems>(L));
  if constexpr (std::is_same_v<Launch, GatherLaunch> || std::is_same_v<Launch, AccumLaunch>)
    if (L.form == kStreamTiles) return issue(short_form<typename ShortForms<Launch>::SomeItems>(L));
  return issue(L);
}

}  // namespace

// ------------------------------------------------------------------------------------------------
// namespace odc_device (odc_launch.h)
// ------------------------------------------------------------------------------------------------
namespace odc_device {

int get_current(int* device) { return (int)hipGetDevice(device); }

int set_current(int device) { return (int)hipSetDevice(device); }

int properties(int device, Properties* out) {
  hipError_t e = hipDeviceGetAttribute(&out->n_cu, hipDeviceAttributeMultiprocessorCount, device);
  if (e != hipSuccess) return (int)e;
  if (out->n_cu <= 0) out->n_cu = 256;
  // the two LDS sizes only matter for residency caps: keep the gfx950 values when a query fails
  out->lds_per_cu = 160 * 1024;
  out->lds_per_wg_max = 64 * 1024;
  int v = 0;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, device) == hipSuccess && v > 0)
    out->lds_per_cu = v;
  if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, device) == hipSuccess && v > 0)
    out->lds_per_wg_max = v;
  (void)hipGetLastError();
  return 0;
}

int allocate(void** ptr, uint64_t bytes) { return (int)hipMalloc(ptr, bytes); }

int release(void* ptr) {
  hipError_t e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipFree(ptr);
  return (int)e;
}

bool is_out_of_memory(int code) { return code == (int)hipErrorOutOfMemory; }

const char* error_string(int code) { return hipGetErrorString(static_cast<hipError_t>(code)); }

bool has_accum(int g, int a) { return pick_accum<AccumLaunch>(g, a, false, {}, kShortTiles) != nullptr; }
bool has_cast_gather(int s, int d) { return pick_cast_gather<CastGatherLaunch>(s, d, {}, kStream, kWholeTiles) != nullptr; }
bool has_publish(int a, int o) { return pick_publish<PublishLaunch>(a, o, kShortTiles) != nullptr; }

// by_table for whole tiles: kGathersWholeTiles
int launch_gather(const GatherLaunch& L, uint32_t grid, uint32_t lds_bytes, void* stream) {
  return launch_form(L, grid, copy_threads(L.form), lds_bytes, stream, [&](auto form) {
    return pick_gather<typename decltype(form)::type>(L.policy.read, L.output, L.form);
  }, L.form == kWholeTiles);
}

int launch_cast_gather(int s, int d, const CastGatherLaunch& L, uint32_t grid, uint32_t lds_bytes, void* stream) {
  return launch_form(L, grid, copy_threads(L.form), lds_bytes, stream, [&](auto form) {
    return pick_cast_gather<typename decltype(form)::type>(s, d, L.policy, L.output, L.form);
  }, L.form == kWholeTiles);
}

int launch_accum(int g, int a, bool store, const AccumLaunch& L, uint32_t grid, uint32_t lds_bytes, void* stream) {
  return launch_form(L, grid, accum_threads(g, a, store, L.policy, L.form), lds_bytes, stream, [&](auto form) {
    return pick_accum<typename decltype(form)::type>(g, a, store, L.policy, L.form);
  });
}

int launch_clear(const ClearLaunch& L, uint32_t grid, void* stream) {
  return launch_form(L, grid, kThreads, 0u, stream, [&](auto form) {
    typedef typename decltype(form)::type F;
    return L.output == kWriteThrough ? &clear_kernel<F, kWriteThrough> : &clear_kernel<F, kKeep>;
  });
}

int launch_publish(int a, int o, const PublishLaunch& L, uint32_t grid, uint32_t lds_bytes, void* stream) {
  return launch_form(L, grid, publish_threads(L.form), lds_bytes, stream,
                     [&](auto form) { return pick_publish<typename decltype(form)::type>(a, o, L.form); });
}

}  // namespace odc_device
