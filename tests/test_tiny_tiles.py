"""Launches of many tiles that are mostly part-empty have workgroups of one wavefront: which launches those are, on
dry-run arenas, and their bits at the edges of segments and tiles."""

import ctypes

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _tiny(world, sizes, store=False):
    """(launches, tiny launches) of a gather of bf16 and of an accumulate into fp32 of items of `sizes` elements."""
    lib, handle, got = _native.load(), ctypes.c_void_p(), []
    _native.check(lib.odc_arena_create(world, 1 << 30, _native.ODC_ARENA_DRY_RUN, ctypes.byref(handle)))
    try:
        gathered, added, off = (_native.GatherItem * len(sizes))(), (_native.AccumItem * len(sizes))(), 0
        for k, n in enumerate(sizes):
            gathered[k] = _native.GatherItem(1 << 33, off, 2 * n)
            added[k] = _native.AccumItem(1 << 33, world * n, off, n)
            off += 4 * n
        bf16, f32 = _native.DTYPE_BF16, _native.DTYPE_F32
        for call in (lambda: lib.odc_gather(handle, gathered, len(sizes), 0, None),
                     lambda: lib.odc_scatter_accumulate(handle, added, len(sizes), bf16, f32, None)):
            _native.set_option("dry_run_reset", 0)
            _native.check(call())
            got.append(tuple(_native.get_option(f"dry_run_{n}") for n in ("launches", "tiny_launches")))
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
