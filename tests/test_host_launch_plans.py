"""The host side of every compute entry point, exercised WITHOUT a GPU on a dry-run arena
(ODC_ARENA_DRY_RUN): argument validation, the split of long item lists over launches, tile counts
and launch shapes. Nothing is launched; the library counts what it would have launched.

A host-side bug here (an item list cut wrongly, a table that does not add up, a recursion) would
otherwise show only on the GPU box."""

import ctypes
import math

import pytest

from odc_amd import _native

TILE_BYTES = 16 * 1024
TILE_ELEMS = 4096
SHORT_TILE_BYTES = TILE_BYTES // 4
SHORT_TILE_ELEMS = TILE_ELEMS // 4
N_CU = 256  # what a dry-run arena assumes
MOST_WORK_ITEMS = (1 << 32) - 1  # of one dispatch


class DryArena:
    def __init__(self, world, bytes_per_rank):
        self.lib = _native.load()
        self.handle = ctypes.c_void_p()
        _native.check(self.lib.odc_arena_create(world, bytes_per_rank, _native.ODC_ARENA_DRY_RUN, ctypes.byref(self.handle)))
        self.world = world
        info = _native.ArenaInfo()
        _native.check(self.lib.odc_arena_get_info(self.handle, ctypes.byref(info)))
        self.info = info
        _native.set_option("dry_run_reset", 0)

    def counters(self):
        return tuple(_native.get_option(n) for n in ("dry_run_launches", "dry_run_tiles", "dry_run_workgroups"))

    def forms(self):
        """Launches in whole tiles, in short tiles, in few short tiles."""
        launches, short, few = (_native.get_option(f"dry_run_{n}") for n in ("launches", "short_launches", "few_launches"))
        return launches - short - few, short, few

    def close(self):
        _native.check(self.lib.odc_arena_destroy(self.handle))


@pytest.fixture
def arena():
    made = []

    def _make(world, bytes_per_rank=1 << 30):
        a = DryArena(world, bytes_per_rank)
        made.append(a)
        return a

    yield _make
    for a in made:
        a.close()


OUTSIDE = 1 << 33  # a "device address" far from the dry-run arena's fictitious base (1 << 44)
FAR_OUTSIDE = 1 << 50  # the same, above the arena: room for outputs of 2^46 bytes


def test_dry_run_arena_has_no_memory_but_plans(arena):
    a = arena(8)
    assert a.info.device == -1 and a.info.base == 0 and a.info.flags & _native.ODC_ARENA_NO_BACKING
    assert not a.lib.odc_arena_ptr(a.handle, 0, 0)  # no memory to point at
    off = ctypes.c_uint64()
    _native.check(a.lib.odc_arena_alloc(a.handle, 1 << 20, ctypes.byref(off)))
    items = (_native.GatherItem * 1)(_native.GatherItem(OUTSIDE, off.value, 1 << 20))
    _native.check(a.lib.odc_gather(a.handle, items, 1, 0, None))
    assert a.counters() == (1, 8 * 64, 8 * 64)  # one launch, one workgroup per 16 KiB tile per rank


def test_a_plain_no_backing_arena_still_refuses_compute():
    lib = _native.load()
    handle = ctypes.c_void_p()
    _native.check(lib.odc_arena_create(4, 1 << 20, _native.ODC_ARENA_NO_BACKING, ctypes.byref(handle)))
    items = (_native.GatherItem * 1)(_native.GatherItem(OUTSIDE, 0, 4096))
    assert lib.odc_gather(handle, items, 1, 0, None) == _native.ODC_ERR_NO_BACKING
    _native.check(lib.odc_arena_destroy(handle))


@pytest.mark.parametrize("n_items", [1, 9, 63, 64, 65, 128, 129, 300])
def test_long_item_lists_are_split_over_launches(arena, n_items):
    W = 4
    a = arena(W)
    sizes = [(7 * i) % 5 * 10_000 + (i % 3) * 17 for i in range(n_items)]  # some are empty
    items = (_native.GatherItem * n_items)()
    off = 0
    for it, sz in zip(items, sizes):
        it.dst, it.src_offset, it.shard_bytes = OUTSIDE + 64 * off, off, sz
        off += sz
    _native.check(a.lib.odc_gather(a.handle, items, n_items, W - 1, None))
    nonempty = [s for s in sizes if s]
    launches, tiles, workgroups = a.counters()
    assert launches == math.ceil(len(nonempty) / _native.MAX_ITEMS_PER_LAUNCH)
    assert tiles == W * sum(math.ceil(s / SHORT_TILE_BYTES) for s in nonempty)  # segments of 3 whole tiles at most
    assert workgroups == tiles  # the gather runs one workgroup per tile


def test_accumulate_launch_shapes(arena):
    W = 8
    a = arena(W)
    # line-aligned whole shards in short segments: one workgroup per tile by default; the persistent
    # shape, one workgroup per CU, only when asked for through the threshold
    shard = 1 << 18
    items = (_native.AccumItem * 2)(
        _native.AccumItem(OUTSIDE, W * shard, 0, shard), _native.AccumItem(OUTSIDE + (1 << 30), W * shard, 4 * shard, shard)
    )
    _native.check(a.lib.odc_scatter_accumulate(a.handle, items, 2, _native.DTYPE_BF16, _native.DTYPE_F32, None))
    launches, tiles, workgroups = a.counters()
    # (16-bit gradients into fp32 go in short tiles whatever the sizes)
    assert (launches, tiles, workgroups) == (1, 2 * W * shard // SHORT_TILE_ELEMS, 2 * W * shard // SHORT_TILE_ELEMS)
    _native.set_option("dry_run_reset", 0)
    _native.set_option("accum_persistent_below_tiles", 128)  # segments of 64 whole tiles are below it
    try:
        _native.check(a.lib.odc_scatter_accumulate(a.handle, items, 2, _native.DTYPE_BF16, _native.DTYPE_F32, None))
        assert a.counters() == (1, tiles, N_CU)
        # the same as a store, or with a gradient that ends early (padding): one workgroup per tile
        _native.set_option("dry_run_reset", 0)
        _native.check(a.lib.odc_scatter_store(a.handle, items, 2, _native.DTYPE_BF16, _native.DTYPE_F32, None))
        assert a.counters() == (1, tiles, tiles)
        _native.set_option("dry_run_reset", 0)
        items[1].grad_elems -= 5
        _native.check(a.lib.odc_scatter_accumulate(a.handle, items, 2, _native.DTYPE_BF16, _native.DTYPE_F32, None))
        assert a.counters() == (1, tiles, tiles)
    finally:
        _native.set_option("accum_persistent_below_tiles", 0)
    # long segments (128 tiles and more): one workgroup per tile, unless the knob says otherwise
    _native.set_option("dry_run_reset", 0)
    shard = 1 << 20
    long_items = (_native.AccumItem * 2)(
        _native.AccumItem(OUTSIDE, W * shard, 0, shard), _native.AccumItem(OUTSIDE + (1 << 30), W * shard, 4 * shard, shard)
    )
    _native.check(a.lib.odc_scatter_accumulate(a.handle, long_items, 2, _native.DTYPE_BF16, _native.DTYPE_F32, None))
    long_tiles = 2 * W * shard // SHORT_TILE_ELEMS
    assert a.counters() == (1, long_tiles, long_tiles)
    _native.set_option("dry_run_reset", 0)
    _native.set_option("accum_blocks_per_cu", 2)
    try:
        _native.check(a.lib.odc_scatter_accumulate(a.handle, long_items, 2, _native.DTYPE_BF16, _native.DTYPE_F32, None))
    finally:
        _native.set_option("accum_blocks_per_cu", -1)
    assert a.counters() == (1, long_tiles, 2 * N_CU)
    # fewer tiles than CUs: the persistent grid shrinks to the tiles
    _native.set_option("dry_run_reset", 0)
    small = (_native.AccumItem * 1)(_native.AccumItem(OUTSIDE, W * 4096, 0, 4096))
    _native.check(a.lib.odc_scatter_accumulate(a.handle, small, 1, _native.DTYPE_BF16, _native.DTYPE_F32, None))
    assert a.counters() == (1, 4 * W, 4 * W)


def test_clear_cast_gather_and_publish_plan(arena):
    W = 4
    a = arena(W)
    spans = (_native.Span * 3)(_native.Span(0, 100_000), _native.Span(1 << 20, 0), _native.Span(2 << 20, 16_384))
    _native.check(a.lib.odc_clear(a.handle, spans, 3, None))
    assert a.counters() == (1, W * (7 + 1), W * 8)
    _native.set_option("dry_run_reset", 0)
    cast = (_native.GatherCastItem * 1)(_native.GatherCastItem(OUTSIDE, 0, 10_000))
    _native.check(a.lib.odc_gather_cast(a.handle, cast, 1, _native.DTYPE_F32, _native.DTYPE_BF16, 2, None))
    assert a.counters() == (1, W * 10, W * 10)  # 3 whole tiles per segment: cut into short ones
    _native.set_option("dry_run_reset", 0)
    pub = (_native.PublishItem * 2)(_native.PublishItem(0, 10_000, OUTSIDE), _native.PublishItem(1 << 20, 4096, None))
    _native.check(a.lib.odc_publish(a.handle, 1, pub, 2, _native.DTYPE_F32, _native.DTYPE_BF16, ctypes.c_float(8.0), None))
    assert a.counters() == (1, 10 + 4, 14)  # one rank only; fp32 accumulations go in short tiles


def _error(lib, status):
    assert status != 0
    return status, lib.odc_last_error().decode()


def test_validation_errors_come_back_as_codes_and_messages(arena):
    W = 4
    a = arena(W, 1 << 20)
    lib = a.lib
    G, A = _native.GatherItem, _native.AccumItem
    inside = a.info.bytes_per_rank  # an offset just past the region
    fake_base = 1 << 44

    def gather(*items, first_rank=0):
        arr = (G * len(items))(*items)
        return lib.odc_gather(a.handle, arr, len(items), first_rank, None)

    def accum(*items, g=_native.DTYPE_BF16, acc=_native.DTYPE_F32):
        arr = (A * len(items))(*items)
        return lib.odc_scatter_accumulate(a.handle, arr, len(items), g, acc, None)

    assert _error(lib, gather(G(None, 0, 64)))[0] == _native.ODC_ERR_INVALID  # dst NULL
    code, msg = _error(lib, gather(G(OUTSIDE, inside - 32, 64)))
    assert code == _native.ODC_ERR_INVALID and "rank region" in msg
    assert _error(lib, gather(G(OUTSIDE, 0, 64), first_rank=W))[0] == _native.ODC_ERR_INVALID
    code, msg = _error(lib, gather(G(fake_base + 128, 0, 4096)))  # dst inside the arena range it reads
    assert code == _native.ODC_ERR_INVALID and "overlaps" in msg
    assert gather(G(None, 0, 0)) == 0  # an empty item needs no destination
    assert lib.odc_gather(a.handle, None, 1, 0, None) == _native.ODC_ERR_INVALID
    assert lib.odc_gather(None, None, 0, 0, None) == _native.ODC_ERR_INVALID

    code, msg = _error(lib, accum(A(OUTSIDE, W * 64 + 1, 0, 64)))
    assert code == _native.ODC_ERR_INVALID and "grad_elems" in msg
    assert _error(lib, accum(A(OUTSIDE, 64, 2, 64)))[0] == _native.ODC_ERR_INVALID  # acc_offset not fp32 aligned
    assert _error(lib, accum(A(OUTSIDE + 1, 64, 0, 64)))[0] == _native.ODC_ERR_INVALID  # grad not bf16 aligned
    assert _error(lib, accum(A(None, 64, 0, 64)))[0] == _native.ODC_ERR_INVALID
    assert _error(lib, accum(A(OUTSIDE, 64, 0, 64), g=7))[0] == _native.ODC_ERR_INVALID  # unknown dtype code
    assert _error(lib, accum(A(OUTSIDE, 1, 0, 0)))[0] == _native.ODC_ERR_INVALID  # data for an empty shard
    assert accum(A(OUTSIDE, 0, 0, 64)) == 0  # an all-padding gradient is fine
    pub = (_native.PublishItem * 1)(_native.PublishItem(0, 64, OUTSIDE))
    for bad in (0.0, float("nan")):
        assert lib.odc_publish(a.handle, 0, pub, 1, _native.DTYPE_F32, _native.DTYPE_BF16, ctypes.c_float(bad), None) \
            == _native.ODC_ERR_INVALID
    assert lib.odc_publish(a.handle, W, pub, 1, _native.DTYPE_F32, _native.DTYPE_BF16, ctypes.c_float(2.0), None) \
        == _native.ODC_ERR_INVALID
    assert a.counters() == (1, W, W)  # the one valid, non-empty call above: the padding-only accumulate


def test_an_item_too_large_for_one_launch_is_refused_not_truncated(arena):
    a = arena(1, 1 << 46)
    items = (_native.GatherItem * 1)(_native.GatherItem(FAR_OUTSIDE, 0, 1 << 46))  # 2^32 tiles
    status = a.lib.odc_gather(a.handle, items, 1, 0, None)
    assert status == _native.ODC_ERR_INVALID and "too large for one launch" in a.lib.odc_last_error().decode()
    assert a.counters() == (0, 0, 0)
    # just under the limit it is one launch
    _native.set_option("dry_run_reset", 0)
    items[0].shard_bytes = ((1 << 31) - 1) * TILE_BYTES
    _native.check(a.lib.odc_gather(a.handle, items, 1, 0, None))
    assert a.counters() == (1, (1 << 31) - 1, MOST_WORK_ITEMS // 512)


def test_many_large_items_split_when_the_tile_count_would_overflow(arena):
    a = arena(2, 1 << 46)
    per_item = (1 << 29) * TILE_BYTES  # 2^29 tiles per rank, 2^30 per item
    items = (_native.GatherItem * 3)()
    for i, it in enumerate(items):
        it.dst, it.src_offset, it.shard_bytes = FAR_OUTSIDE, i * per_item, per_item
    _native.check(a.lib.odc_gather(a.handle, items, 3, 0, None))
    launches, tiles, _ = a.counters()
    assert (launches, tiles) == (3, 3 << 30)  # 2^30 + 2^30 would reach 2^31: one item per launch


def test_convert_plans_one_launch_over_all_ranks(arena):
    W = 8
    a = arena(W)
    C = _native.ConvertItem
    items = (C * 3)(C(0, 1 << 24, 1_000_000), C(0, 0, 0), C(1 << 25, 1 << 26, 4096))
    _native.check(a.lib.odc_convert(a.handle, items, 3, _native.DTYPE_F32, _native.DTYPE_BF16, None))
    tiles = W * (math.ceil(1_000_000 / TILE_ELEMS) + 1)
    assert a.counters() == (1, tiles, tiles)  # the empty item takes no part
    lib = a.lib

    def status(src, dst, elems, sd=_native.DTYPE_F32, dd=_native.DTYPE_BF16):
        arr = (C * 1)(C(src, dst, elems))
        return lib.odc_convert(a.handle, arr, 1, sd, dd, None)

    assert _error(lib, status(2, 1 << 24, 64))[0] == _native.ODC_ERR_INVALID  # source not fp32 aligned
    assert _error(lib, status(0, (1 << 24) + 1, 64))[0] == _native.ODC_ERR_INVALID  # destination not bf16 aligned
    code, msg = _error(lib, status(0, 128, 64))  # [0, 256) read, [128, 256) written
    assert code == _native.ODC_ERR_INVALID and "overlaps" in msg
    assert status(0, 256, 64) == 0  # touching ranges are fine
    code, msg = _error(lib, status(0, 1 << 24, 1 << 62))  # elems * 4 would wrap around
    assert code == _native.ODC_ERR_INVALID and "exceed" in msg
    assert _error(lib, status(0, a.info.bytes_per_rank - 64, 64))[0] == _native.ODC_ERR_INVALID  # destination leaves the region
    assert _error(lib, status(0, 1 << 24, 64, sd=9))[0] == _native.ODC_ERR_INVALID
    assert lib.odc_convert(a.handle, None, 2, _native.DTYPE_F32, _native.DTYPE_BF16, None) == _native.ODC_ERR_INVALID
    # equal dtypes: a symmetric copy
    assert status(0, 1 << 24, 4096, sd=_native.DTYPE_BF16, dd=_native.DTYPE_BF16) == 0


def test_arena_size_plus_alignment_slack_cannot_wrap():
    """world * rank_stride can fit 64 bits while the allocation, which is one stride alignment
    larger so that rank 0 can start on a multiple of it, does not: 17 regions of 986 895 * 2^40
    bytes are 2^64 - 2^40 bytes. Such an arena is refused, with or without backing."""
    lib = _native.load()
    handle = ctypes.c_void_p()
    _native.set_option("rank_stride_align", 1 << 40)
    try:
        stride = 986_895 << 40
        assert 17 * stride == (1 << 64) - (1 << 40)
        for flags in (_native.ODC_ARENA_DRY_RUN, _native.ODC_ARENA_NO_BACKING):
            assert lib.odc_arena_create(17, stride, flags, ctypes.byref(handle)) == _native.ODC_ERR_INVALID
            assert "overflows" in lib.odc_last_error().decode() and not handle.value
        # one region fewer fits
        _native.check(lib.odc_arena_create(16, stride, _native.ODC_ARENA_NO_BACKING, ctypes.byref(handle)))
        _native.check(lib.odc_arena_destroy(handle))
    finally:
        _native.set_option("rank_stride_align", 16384)


@pytest.mark.parametrize("n_items", [5, 256, 257, 700])
def test_accumulate_item_lists_with_tiny_items_keep_every_item(arena, n_items):
    """Items of less than one tile per rank are launched after the others (also through the
    heap-allocated order of lists longer than 256): launches and tiles still add up, and an item
    that is too large is still reported under the caller's index."""
    W = 4
    a = arena(W, 1 << 46)
    sizes = [(100 if i % 3 == 0 else 0 if i % 7 == 0 else 5000 + i) for i in range(n_items)]
    items = (_native.AccumItem * n_items)()
    off = 0
    for it, sz in zip(items, sizes):
        it.grad, it.grad_elems, it.acc_offset, it.shard_elems = OUTSIDE, W * sz, off, sz
        off += -(-4 * sz // 256) * 256
    _native.check(a.lib.odc_scatter_accumulate(a.handle, items, n_items, _native.DTYPE_BF16, _native.DTYPE_F32, None))
    nonempty = [s for s in sizes if s]
    launches, tiles, _ = a.counters()
    assert launches == math.ceil(len(nonempty) / _native.MAX_ITEMS_PER_LAUNCH)
    assert tiles == W * sum(math.ceil(s / SHORT_TILE_ELEMS) for s in nonempty)
    bad = n_items - 2  # position in the caller's list; in launch order it sits elsewhere
    items[bad].shard_elems = (1 << 31) * TILE_ELEMS // W  # 2^31 tiles in all: one too many for a launch
    items[bad].grad_elems, items[bad].acc_offset = 0, 0
    status = a.lib.odc_scatter_accumulate(a.handle, items, n_items, _native.DTYPE_BF16, _native.DTYPE_F32, None)
    message = a.lib.odc_last_error().decode()
    assert status == _native.ODC_ERR_INVALID and f"item {bad}:" in message and "too large for one launch" in message


BF16, F16, F32 = _native.DTYPE_BF16, _native.DTYPE_F16, _native.DTYPE_F32
# entry point -> (item type, an item of n units at symmetric offset off, the call, elements (or bytes) of a whole tile)
PLANNED = {
    "gather": (_native.GatherItem, lambda W, off, n: (OUTSIDE, off, n),
               lambda lib, a, items, n: lib.odc_gather(a, items, n, 0, None), TILE_BYTES),
    "gather_cast": (_native.GatherCastItem, lambda W, off, n: (OUTSIDE, off, n),
                    lambda lib, a, items, n: lib.odc_gather_cast(a, items, n, F32, BF16, 0, None), TILE_ELEMS),
    "convert": (_native.ConvertItem, lambda W, off, n: (off, (1 << 34) + off, n),
                lambda lib, a, items, n: lib.odc_convert(a, items, n, F32, BF16, None), TILE_ELEMS),
    "accumulate": (_native.AccumItem, lambda W, off, n: (OUTSIDE, W * n, off, n),
                   lambda lib, a, items, n: lib.odc_scatter_accumulate(a, items, n, F32, F32, None), TILE_ELEMS),
    "store": (_native.AccumItem, lambda W, off, n: (OUTSIDE, W * n, off, n),
              lambda lib, a, items, n: lib.odc_scatter_store(a, items, n, F32, F32, None), TILE_ELEMS),
}


def _plan(a, what, sizes):
    kind, item, call, _tile = PLANNED[what]
    items, off = (kind * len(sizes))(), 0
    for k, n in enumerate(sizes):
        items[k] = kind(*item(a.world, off, n))
        off += -(-4 * n // 256) * 256
    _native.set_option("dry_run_reset", 0)
    _native.check(call(a.lib, a.handle, items, len(sizes)))
    return a.counters(), a.forms()


@pytest.mark.parametrize("what", PLANNED)
def test_launches_are_cut_as_on_a_device(arena, what):
    """Short segments go in short tiles, long ones in whole tiles, launch by launch; up to 32768
    short tiles in a launch are 'few'."""
    W, tile = 4, PLANNED[what][3]
    a = arena(W, 1 << 36)
    long, edge = 32 * tile, 31 * tile  # segments that average 32 whole tiles and more are long
    assert _plan(a, what, [1]) == ((1, W, W), (0, 0, 1))
    assert _plan(a, what, [edge]) == ((1, W * 4 * 31, W * 4 * 31), (0, 0, 1))
    assert _plan(a, what, [long]) == ((1, W * 32, W * 32), (1, 0, 0))
    assert _plan(a, what, [long, 0, edge])[1] == (0, 0, 1)  # 31.5 on average
    assert _plan(a, what, [long + tile, 0, edge])[1] == (1, 0, 0)
    many = [edge] * 67  # 67 * 4 * 124 short tiles: more than 32768
    assert _plan(a, what, many) == ((1, W * 4 * 31 * 67, W * 4 * 31 * 67), (0, 1, 0))
    assert _plan(a, what, many[1:])[1] == (0, 0, 1)
    # every launch of a longer list is cut by its own items: 112 long ones, 112 of one whole tile
    # each, 70 shorter ones that 42 longer ones outweigh, and three long ones
    mixed = [long] * 112 + [tile] * 112 + [edge] * 70 + [8 * long] * 42 + [2 * long] * 3
    tiles = W * (32 * 112 + 4 * 112 + (31 * 70 + 8 * 32 * 42) + 64 * 3)
    assert _plan(a, what, mixed) == ((4, tiles, tiles), (3, 0, 1))


def test_publish_is_cut_as_on_a_device(arena):
    a = arena(2, 1 << 36)

    def plan(sizes, acc, out):
        items, off = (_native.PublishItem * len(sizes))(), 0
        for k, n in enumerate(sizes):
            items[k] = _native.PublishItem(off, n, OUTSIDE)
            off += -(-4 * n // 256) * 256
        _native.set_option("dry_run_reset", 0)
        _native.check(a.lib.odc_publish(a.handle, 1, items, len(items), acc, out, ctypes.c_float(2.0), None))
        return a.counters(), a.forms()

    # fp32 accumulations always in short tiles, few of them up to 32768
    assert plan([1, 4096], F32, BF16) == ((1, 5, 5), (0, 0, 1))
    assert plan([32768 * 1024], F32, F16) == ((1, 32768, 32768), (0, 0, 1))
    assert plan([32768 * 1024 + 1], F32, F32) == ((1, 32769, 32769), (0, 1, 0))
    # 16-bit ones up to 1024 whole tiles per launch
    assert plan([1000 * 4096, 24 * 4096], BF16, BF16) == ((1, 4096, 4096), (0, 0, 1))
    assert plan([1000 * 4096, 24 * 4096 + 1], BF16, BF16) == ((1, 1025, 1025), (1, 0, 0))
    # launch by launch: 112 items of 10 whole tiles, then 5 of one
    assert plan([10 * 4096] * 112 + [0, 0] + [4096] * 5, F16, F32) == ((2, 1120 + 20, 1140), (1, 0, 1))


@pytest.mark.parametrize("grad", [BF16, F16])
def test_16_bit_gradients_into_fp32_always_go_in_short_tiles(arena, grad):
    W = 4
    a = arena(W, 1 << 36)
    for call in (a.lib.odc_scatter_accumulate, a.lib.odc_scatter_store):
        for n, form in ((1, (0, 0, 1)), (8192 * 1024, (0, 0, 1)), (8192 * 1024 + 1, (0, 1, 0))):
            _native.set_option("dry_run_reset", 0)
            items = (_native.AccumItem * 1)(_native.AccumItem(OUTSIDE, W * n, 0, n))
            _native.check(call(a.handle, items, 1, grad, F32, None))
            tiles = W * math.ceil(n / SHORT_TILE_ELEMS)
            assert (a.counters(), a.forms()) == ((1, tiles, tiles), form)


@pytest.mark.parametrize("call,grad,acc,tile,threads", [
    ("odc_scatter_accumulate", BF16, F32, SHORT_TILE_ELEMS, 128), ("odc_scatter_store", F16, F32, SHORT_TILE_ELEMS, 128),
    ("odc_scatter_accumulate", BF16, BF16, TILE_ELEMS, 512), ("odc_scatter_store", BF16, BF16, TILE_ELEMS, 256),
    ("odc_scatter_accumulate", F32, F32, TILE_ELEMS, 256), ("odc_scatter_store", F32, F32, TILE_ELEMS, 512),
])
def test_a_grid_never_exceeds_the_work_items_of_a_dispatch(arena, call, grad, acc, tile, threads):
    """Launches of more tiles than a dispatch has workgroups for are walked by the largest grid."""
    W = 2
    a = arena(W, 1 << 46)
    most = MOST_WORK_ITEMS // threads
    for tiles_per_rank in (most // W, most // W + 1, 1 << 28):
        n, tiles = tiles_per_rank * tile, W * tiles_per_rank
        for items in ([(0, n)], [(0, n - tile), (1 << 45, tile)]):  # one item, the same work in two
            arr = (_native.AccumItem * len(items))(*[_native.AccumItem(FAR_OUTSIDE, W * m, off, m) for off, m in items])
            _native.set_option("dry_run_reset", 0)
            _native.check(getattr(a.lib, call)(a.handle, arr, len(arr), grad, acc, None))
            assert a.counters() == (1, tiles, min(tiles, most))


def test_grids_of_the_other_entry_points_are_bounded_too(arena):
    a = arena(1, 1 << 46)
    n = 1 << 28  # whole tiles
    span = (_native.Span * 1)(_native.Span(0, n * TILE_BYTES))
    _native.check(a.lib.odc_clear(a.handle, span, 1, None))
    assert a.counters() == (1, n, MOST_WORK_ITEMS // 256)
    for out, acc, tiles, threads in ((F32, F32, 4 * n, 128), (BF16, BF16, n, 256)):
        pub = (_native.PublishItem * 1)(_native.PublishItem(0, n * TILE_ELEMS, FAR_OUTSIDE))
        _native.set_option("dry_run_reset", 0)
        _native.check(a.lib.odc_publish(a.handle, 0, pub, 1, acc, out, ctypes.c_float(3.0), None))
        assert a.counters() == (1, tiles, MOST_WORK_ITEMS // threads)
    cast = (_native.GatherCastItem * 1)(_native.GatherCastItem(FAR_OUTSIDE, 0, n * TILE_ELEMS))
    _native.set_option("dry_run_reset", 0)
    _native.check(a.lib.odc_gather_cast(a.handle, cast, 1, F32, BF16, 0, None))
    assert a.counters() == (1, n, MOST_WORK_ITEMS // 512)
    _native.set_option("gather_blocks_per_cu", 1 << 62)  # more workgroups than there are
    try:
        _native.set_option("dry_run_reset", 0)
        _native.check(a.lib.odc_gather_cast(a.handle, cast, 1, F32, BF16, 0, None))
        assert a.counters() == (1, n, MOST_WORK_ITEMS // 512)
    finally:
        _native.set_option("gather_blocks_per_cu", 0)


@pytest.mark.parametrize("grad,acc", [(BF16, BF16), (F16, BF16), (F16, F16)])
def test_long_stores_of_16_bit_types_stay_in_whole_tiles(arena, grad, acc):
    """Up to 1536 whole tiles in the launch a store of short segments goes in short tiles; the
    read-modify-write always does."""
    W = 4
    a = arena(W, 1 << 36)
    for sizes, store_form in (([24 * 4096] * 16, (0, 0, 1)), ([24 * 4096] * 15 + [24 * 4096 + 1], (1, 0, 0)), ([4096] * 112, (0, 0, 1))):
        items, off = (_native.AccumItem * len(sizes))(), 0
        for k, n in enumerate(sizes):
            items[k] = _native.AccumItem(OUTSIDE, W * n, off, n)
            off += 4 * n + 256
        for call, form in ((a.lib.odc_scatter_store, store_form), (a.lib.odc_scatter_accumulate, (0, 0, 1))):
            _native.set_option("dry_run_reset", 0)
            _native.check(call(a.handle, items, len(items), grad, acc, None))
            assert a.forms() == form
