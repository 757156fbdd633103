"""Launches of one item have kernels of their own, without the item search: where a tile lies, by
brute force on the CPU, and every one of those kernels against the oracle."""

import subprocess
from pathlib import Path

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

ROOT = Path(__file__).resolve().parent.parent
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def test_where_a_tile_lies(tmp_path):
    exe = tmp_path / "single_item_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-Wno-unknown-pragmas", f"-I{ROOT / 'odc_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpu" / "single_item_check.cpp"), "-o", str(exe)], check=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0 and "single items ok" in proc.stdout, proc.stdout + proc.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("order", [0, 1, 2])  # of the tiles: interleaved ranks, item major, rank outermost
@pytest.mark.parametrize("below", [0, 1 << 30])  # whole tiles where there is a choice, short tiles everywhere
@pytest.mark.parametrize("a", DTYPES, ids=str)
@pytest.mark.parametrize("b", DTYPES, ids=str)
def test_one_item(make_world, a, b, order, below):
    """Shards of ``a`` gathered into ``b``, gradients of ``a`` into accumulations of ``b`` (stored, then
    added), published as ``a``, with and without a divisor."""
    import odc_amd
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    options = {"short_tiles_below": below, "rank_major": order, "accum_tile_order": order}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        W = 3
        group = make_world(W, 8 << 20)
        registry = SymmBufferRegistry.get_instance()
        gather, red = GatherService(), ReductionService(accumulation_dtype=b, lazy_clear=True)
        gen = torch.Generator().manual_seed(7)
        for n in (1, 1025, 4096, 20_483):
            shards = [torch.randn(n, generator=gen).to(a) for _ in range(W)]
            source = put_shards(registry, ("p", n), shards)
            out = torch.full((W * n,), float("nan"), dtype=b, device="cuda")
            with odc_amd.virtual_rank(2):  # the walk starts at another rank
                gather.gather_into_tensor(out, registry.get_symm_buffer(("p", n)), group)
            assert_bit_equal(out, oracle.gather(shards) if a == b else oracle.gather_cast(shards, b))

            red.register(n, (n,), a, b, group)
            want = [torch.zeros(n, dtype=b) for _ in range(W)]
            red.clear_accumulations()
            for _ in range(2):
                grad = torch.randn(W * n, generator=gen).to(a)
                red.scatter_accumulate(n, grad.cuda(), group)
                oracle.scatter_accumulate(want, grad)
            for r, got in enumerate(red.get_peer_accumulations(n)):
                assert_bit_equal(got, want[r], f"size {n} rank {r}")
            for divisor in (1.0, 3.0, 4.0):
                (published,) = red.publish([n], out_dtype=a, divisor=divisor)
                want[0] = (want[0].float() / divisor).to(b)
                assert_bit_equal(published, want[0].to(a), f"size {n} divisor {divisor}")
            assert_bit_equal(red.get_accumulation(n), want[0])
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
