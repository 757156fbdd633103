"""Long streams: which launches are cut as such, on a dry-run arena, and their kernels against the oracle
at the edges of a tile and of the item tables."""

import ctypes

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

BF16, F16, F32 = _native.DTYPE_BF16, _native.DTYPE_F16, _native.DTYPE_F32
OUTSIDE = 1 << 50
MB = 1 << 20


def _with_options(options):
    saved = {name: _native.get_option(name) for name in options}
    for name, value in options.items():
        _native.set_option(name, value)
    return saved


@pytest.mark.parametrize("what,elem,min_bytes", [  # bytes written per element, line of a cached input
    (("gather",), 1, 64 * MB), (("odc_scatter_accumulate", BF16, F32), 4, 256 * MB), (("odc_scatter_accumulate", F32, F32), 4, 8 * MB),
    (("odc_scatter_store", F32, F32), 4, 8 * MB), (("odc_scatter_store", BF16, F32), 4, None),
    (("odc_scatter_accumulate", BF16, BF16), 2, None), (("odc_scatter_accumulate", F32, BF16), 2, None),
], ids=str)
def test_which_launches_are_long_streams(what, elem, min_bytes):
    W, lib, handle, at = 4, _native.load(), ctypes.c_void_p(), ctypes.c_uint64()
    saved = _with_options({"cached_arena_bytes": 0})
    _native.check(lib.odc_arena_create(W, 1 << 36, _native.ODC_ARENA_DRY_RUN, ctypes.byref(handle)))
    _native.check(lib.odc_arena_alloc(handle, 1 << 20, ctypes.byref(at)))  # memory in use does not fit the cache
    try:
        def streams(sizes):  # bytes written per rank and item
            _native.set_option("dry_run_reset", 0)
            n, off = len(sizes), 0
            items = ((_native.GatherItem if what[0] == "gather" else _native.AccumItem) * n)()
            for it, size in zip(items, sizes):
                if what[0] == "gather":
                    it.dst, it.src_offset, it.shard_bytes = OUTSIDE, off, size
                else:
                    it.grad, it.grad_elems, it.acc_offset, it.shard_elems = OUTSIDE, W * (size // elem), off, size // elem
                off += size
            if what[0] == "gather":
                _native.check(lib.odc_gather(handle, items, n, 0, None))
            else:
                _native.check(getattr(lib, what[0])(handle, items, n, what[1], what[2], None))
            assert _native.get_option("dry_run_tiles") == _native.get_option("dry_run_workgroups")
            return _native.get_option("dry_run_stream_launches")

        far = [16 * MB] * 64
        assert streams(far) == (min_bytes is not None)
        assert streams(far + [16 * MB]) == 0  # one item more than the table holds
        assert streams([1 << 33]) == (min_bytes is not None)
        if min_bytes:
            assert streams([min_bytes // W]) == 0 and streams([min_bytes // W + 4096]) == 1
    finally:
        _native.check(lib.odc_arena_destroy(handle))
        for name, value in saved.items():
            _native.set_option(name, value)


# workgroups that walk many tiles, beside everything that would make a launch a long stream
WALKED = [
    {"gather_blocks_per_cu": 1, "accum_blocks_per_cu": 1, "store_blocks_per_cu": 1},
    {"accum_persistent_below_tiles": 1 << 30},
    {"accum_blocks_per_cu": 0, "accum_persistent_below_tiles": 1 << 30, "store_blocks_per_cu": 2},
    {"accum_resident_cap": 2, "gather_resident_cap": 1, "store_resident_cap": 4},
]
FAR_STREAMS = {"stream_bytes": 0, "cached_output_bytes": 0, "cached_gradient_bytes": 0, "cached_arena_bytes": 0, "short_tiles_below": 0}
SHARDS = {1: [96 * 4096], 3: [64 * 4096, 4096, 31 * 4096]}  # whole tiles, more of them than a GPU has CUs


@pytest.mark.parametrize("sizes", SHARDS.values(), ids=len)
@pytest.mark.parametrize("knobs", WALKED, ids=str)
def test_a_long_stream_has_a_workgroup_per_tile(knobs, sizes):
    """There are no kernels that walk a long stream's tiles: whatever asks for fewer workgroups than tiles
    keeps a launch from being one."""
    W, lib, handle, at = 4, _native.load(), ctypes.c_void_p(), ctypes.c_uint64()
    saved = _with_options({**FAR_STREAMS, **knobs})
    _native.check(lib.odc_arena_create(W, 1 << 30, _native.ODC_ARENA_DRY_RUN, ctypes.byref(handle)))
    _native.check(lib.odc_arena_alloc(handle, 1 << 20, ctypes.byref(at)))
    try:
        for name, *codes in [("odc_gather", 0)] + [(call, g, a) for call in ("odc_scatter_accumulate", "odc_scatter_store")
                                                   for g in (BF16, F16, F32) for a in (BF16, F16, F32)]:
            is_gather = name == "odc_gather"
            items, off = ((_native.GatherItem if is_gather else _native.AccumItem) * len(sizes))(), 0
            for k, n in enumerate(sizes):
                items[k] = _native.GatherItem(OUTSIDE, off, 4 * n) if is_gather else _native.AccumItem(OUTSIDE, W * n, off, n)
                off += 4 * n
            _native.set_option("dry_run_reset", 0)
            _native.check(getattr(lib, name)(handle, items, len(sizes), *codes, None))
            tiles, workgroups, streams = (_native.get_option(f"dry_run_{n}") for n in ("tiles", "workgroups", "stream_launches"))
            assert tiles == workgroups or not streams, (name, codes)
            if is_gather:
                walked = "gather_blocks_per_cu" in knobs
                assert (workgroups < tiles, streams) == (walked, not walked)
    finally:
        _native.check(lib.odc_arena_destroy(handle))
        for name, value in saved.items():
            _native.set_option(name, value)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", SHARDS.values(), ids=len)
@pytest.mark.parametrize("knobs", WALKED, ids=str)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=str)
def test_walked_tiles_beside_long_streams(make_world, dtype, knobs, sizes):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    saved = _with_options({**FAR_STREAMS, **knobs})
    try:
        W = 4
        group = make_world(W, 16 * MB)
        registry = SymmBufferRegistry.get_instance()
        gather, red = GatherService(), ReductionService(accumulation_dtype=torch.float32, lazy_clear=True)
        gen = torch.Generator().manual_seed(29)
        shards = [[torch.randn(n, generator=gen).to(dtype) for _ in range(W)] for n in sizes]
        sources = [put_shards(registry, ("p", i), s) for i, s in enumerate(shards)]
        outs = [torch.full((W * n,), float("nan"), dtype=dtype, device="cuda") for n in sizes]
        gather.gather_into_tensors(outs, sources, group)
        for out, s in zip(outs, shards):
            assert_bit_equal(out, oracle.gather(s))
        keys = list(range(len(sizes)))
        for key, n in zip(keys, sizes):
            red.register(key, (n,), dtype, torch.float32, group)
        want = [[torch.zeros(n) for _ in range(W)] for n in sizes]
        red.clear_accumulations()
        for _ in range(2):  # the store form, then read-modify-write
            grads = [torch.randn(W * n, generator=gen).to(dtype) for n in sizes]
            red.scatter_accumulate_multi(keys, [g.cuda() for g in grads], group)
            for accs, g in zip(want, grads):
                oracle.scatter_accumulate(accs, g)
        for key, accs in zip(keys, want):
            for r, got in enumerate(red.get_peer_accumulations(key)):
                assert_bit_equal(got, accs[r], f"size {sizes[key]} rank {r}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)


@pytest.mark.gpu
@pytest.mark.parametrize("order", [0, 1, 2])  # of the tiles: interleaved ranks, item major, rank outermost
@pytest.mark.parametrize("share", [0, 1 << 19])  # of the memory in use that stays in the cache
@pytest.mark.parametrize("n_items", [1, 2, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("grad_dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
def test_long_streams(make_world, grad_dtype, n_items, share, order):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    saved = _with_options({
        "stream_bytes": 0, "cached_output_bytes": 0, "cached_gradient_bytes": 0, "cached_arena_bytes": 0, "short_tiles_below": 0,
        "rank_major": order, "accum_tile_order": order, "resident_above": 0, "resident_accumulation_bytes": share,
        "resident_shard_bytes": share, "resident_clear_bytes": 0,
    })
    try:
        W = 3
        group = make_world(W, 8 * MB)
        registry = SymmBufferRegistry.get_instance()
        gather, red = GatherService(), ReductionService(accumulation_dtype=torch.float32, lazy_clear=True)
        gen = torch.Generator().manual_seed(23)
        # around the edges of a short tile, of a line, and a dozen tiles; only the last items of a list are long
        sizes = [(1024, 1, 1025, 1023, 63, 2049, 4096, 3)[i % 8] + (i // 8) for i in range(n_items - 1)] + [12_801]
        shards = [[torch.randn(n, generator=gen).to(grad_dtype) for _ in range(W)] for n in sizes]
        sources = [put_shards(registry, ("p", i), s) for i, s in enumerate(shards)]
        outs = [torch.full((W * n,), float("nan"), dtype=grad_dtype, device="cuda") for n in sizes]
        gather.gather_into_tensors(outs, sources, group)
        for out, s in zip(outs, shards):
            assert_bit_equal(out, oracle.gather(s))
        keys = list(range(n_items))
        for key, n in zip(keys, sizes):
            red.register(key, (n,), grad_dtype, torch.float32, group)
        want = [[torch.zeros(n) for _ in range(W)] for n in sizes]
        red.clear_accumulations()
        for m in range(3):  # the store form, then read-modify-write; gradients that end early
            valid = [max(0, W * n - 5 * m) for n in sizes]
            grads = [torch.randn(v, generator=gen).to(grad_dtype) for v in valid]
            red.scatter_accumulate_multi(keys, [g.cuda() for g in grads], group, valid_numels=valid)
            for accs, g, n in zip(want, grads, sizes):
                oracle.scatter_accumulate(accs, torch.nn.functional.pad(g, [0, W * n - g.numel()]))
        for key, accs in zip(keys, want):
            for r, got in enumerate(red.get_peer_accumulations(key)):
                assert_bit_equal(got, accs[r], f"size {sizes[key]} rank {r}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
