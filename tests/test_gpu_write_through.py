"""Gathers whose output is written through the L2: whole and short tiles, aligned and ragged segments, and
nothing written outside the output."""

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shards_cached", [0, 1 << 40])
@pytest.mark.parametrize("below", [0, 1 << 30], ids=["whole tiles", "short tiles"])
@pytest.mark.parametrize("sizes", [[16 * 4096], [8191, 8192, 8193, 2 * 8192 + 7], [1, 2047, 2048, 2049, 0, 65 * 1024]], ids=str)
def test_bits_and_bounds(make_world, sizes, below, shards_cached):
    from odc_amd import GatherService, SymmBufferRegistry

    options = {"plain_output_bytes": 0, "cached_output_bytes": 1 << 40, "cached_arena_bytes": shards_cached, "short_tiles_below": below}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        W, pad = 3, 64
        group = make_world(W, 4 << 20)
        gen = torch.Generator().manual_seed(9)
        shards = [[torch.randn(n, generator=gen).bfloat16() for _ in range(W)] for n in sizes]
        sources = [put_shards(SymmBufferRegistry.get_instance(), ("p", i), s) for i, s in enumerate(shards)]
        for start in (0, 1, 37):  # elements: outputs on a line, and not even on 4 bytes
            around = [torch.full((pad + start + W * n + pad,), 7.0, dtype=torch.bfloat16, device="cuda") for n in sizes]
            outs = [t[pad + start : pad + start + W * n] for t, n in zip(around, sizes)]
            GatherService().gather_into_tensors(outs, sources, group)
            for t, s, n in zip(around, shards, sizes):
                want = torch.full_like(t, 7.0, device="cpu")
                want[pad + start : pad + start + W * n] = oracle.gather(s)
                assert_bit_equal(t, want, f"size {n} start {start}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
