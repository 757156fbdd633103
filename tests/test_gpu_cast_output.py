"""Converted outputs written through the L2: whole and short tiles, aligned and ragged segments, every pair of
dtypes, into one output and into every rank's own region, and nothing written outside them."""

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


@pytest.mark.parametrize("line", [0, 1 << 40], ids=["nontemporal", "written through"])
@pytest.mark.parametrize("below", [0, 1 << 30], ids=["whole tiles", "short tiles"])
@pytest.mark.parametrize("sizes", [[16 * 4096], [4095, 4096, 4097, 2 * 4096 + 7], [1, 1023, 1024, 1025, 0, 33 * 1024]], ids=str)
@pytest.mark.parametrize("pair", [(a, b) for a in DTYPES for b in DTYPES if a != b], ids=str)
def test_bits_and_bounds(make_world, pair, sizes, below, line):
    from odc_amd import GatherService, SymmBufferRegistry

    src, dst = pair
    options = {"cast_output_bytes": line, "cached_output_bytes": line, "cached_arena_bytes": 0, "short_tiles_below": below}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        W, pad = 3, 64
        group = make_world(W, 4 << 20)
        registry, gather = SymmBufferRegistry.get_instance(), GatherService()
        gen = torch.Generator().manual_seed(9)
        shards = [[torch.randn(n, generator=gen).to(src) for _ in range(W)] for n in sizes]
        sources = [put_shards(registry, ("p", i), s) for i, s in enumerate(shards)]
        for start in (0, 1, 37):  # elements: outputs on a line, and not even on 4 bytes
            around = [torch.full((pad + start + W * n + pad,), 7.0, dtype=dst, device="cuda") for n in sizes]
            outs = [t[pad + start : pad + start + W * n] for t, n in zip(around, sizes)]
            gather.gather_into_tensors(outs, sources, group)
            for t, s, n in zip(around, shards, sizes):
                want = torch.full_like(t, 7.0, device="cpu")
                want[pad + start : pad + start + W * n] = oracle.gather_cast(s, dst)
                assert_bit_equal(t, want, f"size {n} start {start}")
        for i, (n, parts) in enumerate(zip(sizes, shards)):
            if n:
                registry.allocate_symm_buffer(("c", i), (n,), dst)
                gather.convert_symm_buffer(("c", i), ("p", i))
                for got, s in zip(registry.peer_tensors[("c", i)], parts):
                    assert_bit_equal(got, s.to(dst))
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
