"""A part of symmetric memory is read, and where nothing is read written, through the caches
(resident_below in odc_host.cpp): the bits do not depend on which tiles those are."""

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu

# elements per rank: less than a tile, a tile, ragged tails, many 16 KiB granules
SIZES = [63, 4096, 4099, 70_001, 200_000]


@pytest.mark.parametrize("share", [0.0, 0.3, 0.9])
@pytest.mark.parametrize("below", [0, 32, 1 << 30])  # whole tiles where there is a choice, the default, short tiles
@pytest.mark.parametrize("grad_dtype,acc_dtype", [
    (torch.bfloat16, torch.float32), (torch.float32, torch.float32), (torch.float16, torch.bfloat16),
])
def test_every_form(make_world, grad_dtype, acc_dtype, below, share):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry, _native

    W = 3
    in_use = sum(n * (grad_dtype.itemsize + acc_dtype.itemsize) for n in SIZES) * W
    part = int(share * in_use)
    options = {"resident_above": 0, "resident_accumulation_bytes": part, "resident_shard_bytes": part,
               "resident_clear_bytes": 0, "cached_arena_bytes": 0, "short_tiles_below": below}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        group = make_world(W, 8 << 20)
        registry = SymmBufferRegistry.get_instance()
        gather, red = GatherService(), ReductionService(accumulation_dtype=acc_dtype)
        gen = torch.Generator().manual_seed(17)
        shards = [[torch.randn(n, generator=gen).to(grad_dtype) for _ in range(W)] for n in SIZES]
        sources = [put_shards(registry, ("p", i), s) for i, s in enumerate(shards)]
        outs = [torch.full((W * n,), float("nan"), dtype=grad_dtype, device="cuda") for n in SIZES]
        keys = list(range(len(SIZES)))
        for key, n in zip(keys, SIZES):
            red.register(key, (n,), grad_dtype, acc_dtype, group)
        for first in range(len(SIZES)):  # lists of five items, down to one
            gather.gather_into_tensors(outs[first:], sources[first:], group)
        for out, s in zip(outs, shards):
            assert_bit_equal(out, oracle.gather(s))
        for lazy in (False, True):  # a clear kernel, then the store form
            red.lazy_clear = lazy
            red.clear_accumulations()
            want = [[torch.zeros(n, dtype=acc_dtype) for _ in range(W)] for n in SIZES]
            for _ in range(3):
                grads = [torch.randn(W * n, generator=gen).to(grad_dtype) for n in SIZES]
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
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
