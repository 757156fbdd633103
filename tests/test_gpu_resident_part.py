"""A part of symmetric memory is read, and where nothing is read written, through the caches
(resident_below in odc_host.cpp): which launches are told of it, on a dry-run arena, and that the bits do
not depend on which tiles those are."""

import contextlib
import ctypes

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from odc_amd.primitives.utils import native_dtype
from oracle import odc_oracle as oracle

# elements per rank: less than a tile, a tile, ragged tails, many 16 KiB granules
SIZES = [63, 4096, 4099, 70_001, 200_000]
LISTS = [SIZES, [n - i for i, n in enumerate(4 * SIZES)]]  # small tables, and the full ones
W = 3

FORMS = [pytest.mark.parametrize("share", [0.0, 0.4, 2.0]),  # of what is in use; 2: all of it
         pytest.mark.parametrize("below", [0, 32, 1 << 30]),  # whole tiles where there is a choice, the default, short tiles
         pytest.mark.parametrize("stream", [0, 1 << 40], ids=["long streams", "no streams"]),
         pytest.mark.parametrize("grad_dtype,acc_dtype", [(torch.bfloat16, torch.float32), (torch.float32, torch.float32),
                                                          (torch.float16, torch.bfloat16)])]


def every_form(test):
    for mark in FORMS:
        test = mark(test)
    return test


@contextlib.contextmanager
def resident_options(sizes, share, below, stream, grad_dtype, acc_dtype):
    """Nothing else decides: no gradient, output or arena is small enough to be cached, any clear is long
    enough, and no launch is short enough for the table that ignores the part."""
    in_use = sum(n * (grad_dtype.itemsize + acc_dtype.itemsize) for n in sizes) * W
    part = int(share * in_use)
    options = {"resident_above": 0, "resident_accumulation_bytes": part, "resident_shard_bytes": part,
               "resident_clear_bytes": 0, "cached_arena_bytes": 0, "cached_gradient_bytes": 0, "cached_output_bytes": 0,
               "short_tiles_below": below, "stream_bytes": stream, "few_tiles": 0}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        yield
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)


@pytest.mark.parametrize("sizes", LISTS, ids=len)
@every_form
def test_the_launches_have_it(sizes, grad_dtype, acc_dtype, stream, below, share):
    lib, handle = _native.load(), ctypes.c_void_p()
    outside, grad, acc = 1 << 50, native_dtype(grad_dtype), native_dtype(acc_dtype)
    _native.check(lib.odc_arena_create(W, 64 << 20, _native.ODC_ARENA_DRY_RUN, ctypes.byref(handle)))
    try:
        def allocated(nbytes):
            at = ctypes.c_uint64()
            _native.check(lib.odc_arena_alloc(handle, nbytes, ctypes.byref(at)))
            return at.value

        gathers, accums, spans = ((kind * len(sizes))() for kind in (_native.GatherItem, _native.AccumItem, _native.Span))
        for k, n in enumerate(sizes):
            gathers[k] = _native.GatherItem(outside, allocated(n * grad_dtype.itemsize), n * grad_dtype.itemsize)
            at = allocated(n * acc_dtype.itemsize)
            accums[k] = _native.AccumItem(outside, W * n, at, n)
            spans[k] = _native.Span(at, n * acc_dtype.itemsize)
        count = len(sizes)
        with resident_options(sizes, share, below, stream, grad_dtype, acc_dtype):
            for call in (lambda: lib.odc_gather(handle, gathers, count, 0, None),
                         lambda: lib.odc_scatter_store(handle, accums, count, grad, acc, None),
                         lambda: lib.odc_scatter_accumulate(handle, accums, count, grad, acc, None),
                         lambda: lib.odc_clear(handle, spans, count, None)):
                _native.set_option("dry_run_reset", 0)
                _native.check(call())
                assert _native.get_option("dry_run_launches") == 1 and _native.get_option("dry_run_few_launches") == 0
                assert _native.get_option("dry_run_resident_launches") == (share > 0)
            if not below and acc_dtype == torch.float32:  # the last accumulate and the gather can be long streams
                _native.set_option("dry_run_reset", 0)
                _native.check(lib.odc_gather(handle, gathers, count, 0, None))
                _native.check(lib.odc_scatter_accumulate(handle, accums, count, grad, acc, None))
                assert _native.get_option("dry_run_stream_launches") == (0 if stream else 2)
    finally:
        _native.check(lib.odc_arena_destroy(handle))


@pytest.mark.gpu
@every_form
def test_every_form(make_world, grad_dtype, acc_dtype, stream, below, share):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    group = make_world(W, 32 << 20)
    registry = SymmBufferRegistry.get_instance()
    gen = torch.Generator().manual_seed(17)
    for sizes in LISTS:
        with resident_options(sizes, share, below, stream, grad_dtype, acc_dtype):
            gather, red = GatherService(), ReductionService(accumulation_dtype=acc_dtype)
            shards = [[torch.randn(n, generator=gen).to(grad_dtype) for _ in range(W)] for n in sizes]
            sources = [put_shards(registry, ("p", len(sizes), i), s) for i, s in enumerate(shards)]
            outs = [torch.full((W * n,), float("nan"), dtype=grad_dtype, device="cuda") for n in sizes]
            keys = [(len(sizes), i) for i in range(len(sizes))]
            for key, n in zip(keys, sizes):
                red.register(key, (n,), grad_dtype, acc_dtype, group)
            for first in range(len(sizes)):  # lists of all items, down to one
                gather.gather_into_tensors(outs[first:], sources[first:], group)
            for out, s in zip(outs, shards):
                assert_bit_equal(out, oracle.gather(s))
            for lazy in (False, True):  # a clear kernel, then the store form
                red.lazy_clear = lazy
                red.clear_accumulations()
                want = [[torch.zeros(n, dtype=acc_dtype) for _ in range(W)] for n in sizes]
                for _ in range(3):
                    grads = [torch.randn(W * n, generator=gen).to(grad_dtype) for n in sizes]
                    red.scatter_accumulate_multi(keys, [g.cuda() for g in grads], group)
                    for accs, g in zip(want, grads):
                        oracle.scatter_accumulate(accs, g)
                for key, accs in zip(keys, want):
                    for r, got in enumerate(red.get_peer_accumulations(key)):
                        assert_bit_equal(got, accs[r], f"lazy {lazy} key {key} rank {r}")
            red.lazy_clear = False
            red.clear_accumulations()
            for key in keys:
                assert not any(acc.any() for acc in red.get_peer_accumulations(key))
