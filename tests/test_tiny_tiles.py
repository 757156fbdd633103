"""Launches of many tiles that are mostly part-empty have workgroups of one wavefront: which launches those are, on
dry-run arenas, and their bits at the edges of segments and tiles."""

import ctypes

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _tiny(world, sizes):
    """(launches, tiny launches) of a gather of bf16 and of an accumulate into fp32 of items of `sizes` elements."""
    got = _plan(world, sizes, BF16, BF16, F32)
    return [got["gather"], got["accumulate"]]


def _plan(world, sizes, shard_dtype, compute_dtype, acc_dtype):
    """(launches, tiny launches) of the gather, accumulate and store of items of `sizes` elements."""
    lib, handle, got = _native.load(), ctypes.c_void_p(), {}
    code = {BF16: _native.DTYPE_BF16, F16: _native.DTYPE_F16, F32: _native.DTYPE_F32}
    _native.check(lib.odc_arena_create(world, 1 << 30, _native.ODC_ARENA_DRY_RUN, ctypes.byref(handle)))
    try:
        n, out, off = len(sizes), 1 << 33, 0
        gathered, cast, added = (_native.GatherItem * n)(), (_native.GatherCastItem * n)(), (_native.AccumItem * n)()
        for k, m in enumerate(sizes):
            gathered[k] = _native.GatherItem(out, off, m * shard_dtype.itemsize)
            cast[k] = _native.GatherCastItem(out, off, m)
            added[k] = _native.AccumItem(out, world * m, off, m)
            off += 4 * m
            out += 4 * world * m
        pair = code[compute_dtype], code[acc_dtype]
        calls = {
            "gather": (lambda: lib.odc_gather(handle, gathered, n, 0, None)) if shard_dtype == compute_dtype else
                      (lambda: lib.odc_gather_cast(handle, cast, n, code[shard_dtype], code[compute_dtype], 0, None)),
            "accumulate": lambda: lib.odc_scatter_accumulate(handle, added, n, *pair, None),
            "store": lambda: lib.odc_scatter_store(handle, added, n, *pair, None),
        }
        for name, call in calls.items():
            _native.set_option("dry_run_reset", 0)
            _native.check(call())
            got[name] = tuple(_native.get_option(f"dry_run_{c}") for c in ("launches", "tiny_launches"))
    finally:
        _native.check(lib.odc_arena_destroy(handle))
    return got


def test_which_launches():
    # 2048 tiles in all, at most half full (2048 elements of a gather in bf16, 1024 of an accumulate)
    assert _tiny(64, [100] * 32) == [(1, 1), (1, 1)]
    assert _tiny(64, [100] * 31) == [(1, 0), (1, 0)]
    assert _tiny(64, [512] * 32) == [(1, 1), (1, 1)]
    assert _tiny(64, [512] * 31 + [528]) == [(1, 1), (1, 0)]
    assert _tiny(64, [1024] * 32) == [(1, 1), (1, 0)]
    assert _tiny(64, [1032] * 32) == [(1, 0), (1, 0)]  # (two tiles per segment of the accumulate, half full)
    assert _tiny(256, [100] * 16) == [(1, 0), (1, 0)]  # up to 16 items have tables of their own
    assert _tiny(256, [100] * 17) == [(1, 1), (1, 1)]
    assert _tiny(64, [100] * 112 + [100] * 20) == [(2, 1), (2, 1)]  # launch by launch


def test_where_they_begin_is_an_option():
    saved = _native.get_option("tiny_tiles_from")
    try:
        assert saved == 2048
        _native.set_option("tiny_tiles_from", 0)
        assert _tiny(2, [100] * 17) == [(1, 1), (1, 1)] and _tiny(2, [100] * 16) == [(1, 0), (1, 0)]
        assert _tiny(2, [1032] * 17) == [(1, 0), (1, 0)]
        _native.set_option("tiny_tiles_from", 1 << 40)
        assert _tiny(64, [100] * 112) == [(1, 0), (1, 0)]
    finally:
        _native.set_option("tiny_tiles_from", saved)


@pytest.mark.gpu
@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("shard_dtype,compute_dtype,acc_dtype", [(BF16, BF16, F32), (F32, BF16, BF16), (F32, F32, F32), (F16, F16, F16)])
@pytest.mark.parametrize("sizes", [
    [(37 * i) % 130 for i in range(65)],  # less than a line, odd starts, empty ones
    [255, 256, 257, 511, 512, 513, 1, 3, 1024, 1025, 127, 129] * 3,
], ids=["small", "edges"])
def test_bits(make_world, sizes, shard_dtype, compute_dtype, acc_dtype, order):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    options = {"rank_major": order, "accum_tile_order": order}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        W, n = 64, len(sizes)
        plan = _plan(W, sizes, shard_dtype, compute_dtype, acc_dtype)
        assert plan["gather"] == plan["accumulate"] == (1, 1)
        offsets = [sum(sizes[:i]) for i in range(n)]
        group = make_world(W, 1 << 20)
        gather, red = GatherService(), ReductionService(accumulation_dtype=acc_dtype, lazy_clear=True)
        gen = torch.Generator().manual_seed(n)
        shards = [torch.randn(sum(sizes), generator=gen).to(shard_dtype) for _ in range(W)]
        source = put_shards(SymmBufferRegistry.get_instance(), "p", shards)
        around = [torch.full((W * m + 128,), 7.0, dtype=compute_dtype, device="cuda") for m in sizes]
        outs = [t[63 : 63 + W * m] for t, m in zip(around, sizes)]
        gather.gather_slices(outs, source, offsets, sizes, group)
        for t, off, m in zip(around, offsets, sizes):
            want = torch.full((W * m + 128,), 7.0, dtype=compute_dtype)
            pieces = [s[off : off + m] for s in shards]
            want[63 : 63 + W * m] = oracle.gather(pieces) if shard_dtype == compute_dtype else oracle.gather_cast(pieces, compute_dtype)
            assert_bit_equal(t, want, f"size {m}")
        want = [torch.zeros(sum(sizes), dtype=acc_dtype) for _ in range(W)]
        for m in range(3):  # adds, then (after a clear) the store form, then adds; gradients that end early
            grads = [torch.randn(max(0, W * s - m), generator=gen).to(compute_dtype) for s in sizes]
            red.scatter_accumulate_slices("g", [g.cuda() for g in grads], offsets, sizes, group)
            for g, off, s in zip(grads, offsets, sizes):
                padded = torch.nn.functional.pad(g, [0, W * s - g.numel()])
                oracle.scatter_accumulate([w[off : off + s] for w in want], padded)
            for r, got in enumerate(red.get_peer_accumulations("g")):
                assert_bit_equal(got, want[r], f"rank {r} pass {m}")
            if m == 0:
                red.clear_accumulations()
                for w in want:
                    w.zero_()
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)


LARGE = 1 << 40
FORMS = {
    "plain": {"plain_output_bytes": LARGE, "plain_accumulation_bytes": LARGE, "cached_arena_bytes": LARGE},
    "written through": {"plain_output_bytes": 0, "plain_accumulation_bytes": 0, "cached_arena_bytes": LARGE,
                        "through_store_bytes": LARGE, "cast_output_bytes": LARGE},
    "past the caches": {"cached_output_bytes": 0, "cached_gradient_bytes": 0, "cached_arena_bytes": 0, "cast_output_bytes": 0},
    "outputs written through": {"plain_output_bytes": 0, "cached_output_bytes": LARGE, "cached_arena_bytes": 0,
                                "cast_output_bytes": LARGE},  # shards and accumulations past the caches
}


def _reach(start, segment_bytes, vec_units_bytes, tile_bytes):
    """Of a segment written at `start`: the head of its first tile if that is whole, and its whole tiles behind it."""
    head = min(-start % 128, segment_bytes)
    whole = (segment_bytes - head) // vec_units_bytes * vec_units_bytes // tile_bytes
    return head if whole else 0, max(0, whole - 1)


@pytest.mark.gpu
@pytest.mark.parametrize("apart", [1, 64], ids=["packed", "on lines"])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shard_dtype,compute_dtype,acc_dtype", [
    (BF16, BF16, F32), (F32, BF16, BF16), (F32, F32, F32), (F16, F16, F16), (F16, F32, F32), (BF16, BF16, BF16)])
def test_whole_tiles_among_them(make_world, shard_dtype, compute_dtype, acc_dtype, form, apart):
    """Long lists of tiny items with a few longer ones: tiles that are whole, heads of more bytes than a wavefront has
    lanes, later tiles of their segments, part-filled last ones, in each of the ways that tiles are written."""
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    sizes = [(7 * i) % 41 for i in range(64)] + [1024 + 127, 2048 + 32, 3 * 1024, 5000, 9001]
    saved = {name: _native.get_option(name) for name in FORMS[form]}
    try:
        for name, value in FORMS[form].items():
            _native.set_option(name, value)
        W, n = 64, len(sizes)
        plan = _plan(W, sizes, shard_dtype, compute_dtype, acc_dtype)
        stores = (1, 0) if compute_dtype.itemsize == acc_dtype.itemsize == 2 else (1, 1)  # (those go in whole tiles)
        assert plan == {"gather": (1, 1), "accumulate": (1, 1), "store": stores}
        offsets, total = [], 0
        for m in sizes:
            offsets.append(total)
            total = -(-(total + m) // apart) * apart
        group = make_world(W, 2 << 20)
        gather, red = GatherService(), ReductionService(accumulation_dtype=acc_dtype, lazy_clear=True)
        gen = torch.Generator().manual_seed(n)
        shards = [torch.randn(total, generator=gen).to(shard_dtype) for _ in range(W)]
        source = put_shards(SymmBufferRegistry.get_instance(), "p", shards)
        around = [torch.full((W * m + 128,), 7.0, dtype=compute_dtype, device="cuda") for m in sizes]
        outs = [t[63 : 63 + W * m] for t, m in zip(around, sizes)]
        cast, size = shard_dtype != compute_dtype, compute_dtype.itemsize
        reach = [_reach(t.data_ptr() + r * m * size, m * size, 4 * size if cast else 16, 1024 * size if cast else 4096)
                 for t, m in zip(outs, sizes) for r in range(W)]
        assert max(head for head, _ in reach) > 64 and max(later for _, later in reach) > 1
        gather.gather_slices(outs, source, offsets, sizes, group)
        for t, off, m in zip(around, offsets, sizes):
            want = torch.full((W * m + 128,), 7.0, dtype=compute_dtype)
            pieces = [s[off : off + m] for s in shards]
            want[63 : 63 + W * m] = oracle.gather_cast(pieces, compute_dtype) if cast else oracle.gather(pieces)
            assert_bit_equal(t, want, f"size {m}")
        want = [torch.zeros(total, dtype=acc_dtype) for _ in range(W)]
        for m in range(3):  # adds, then (after a clear) the store form, then adds; gradients that end early
            grads = [torch.randn(max(0, W * s - m), generator=gen).to(compute_dtype) for s in sizes]
            red.scatter_accumulate_slices("g", [g.cuda() for g in grads], offsets, sizes, group, accumulation_numel=total)
            for g, off, s in zip(grads, offsets, sizes):
                padded = torch.nn.functional.pad(g, [0, W * s - g.numel()])
                oracle.scatter_accumulate([w[off : off + s] for w in want], padded)
            peers = red.get_peer_accumulations("g")
            for r, got in enumerate(peers):
                assert_bit_equal(got, want[r], f"rank {r} pass {m}")
            if m == 0:
                size = acc_dtype.itemsize
                reach = [_reach(p.data_ptr() + off * size, s * size, 4 * size, 1024 * size)
                         for p in peers for off, s in zip(offsets, sizes)]
                assert max(later for _, later in reach) > 1 and (max(head for head, _ in reach) > 0) == (apart == 1)
                red.clear_accumulations()
                for w in want:
                    w.zero_()
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
