"""Launches of 2 to 16 items have tables of their own and kernels that read them at once: where a tile
lies, by brute force on the CPU, and every one of those kernels against the oracle, with the next larger
list beside them."""

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
    exe = tmp_path / "few_items_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-Wno-unknown-pragmas", f"-I{ROOT / 'odc_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpu" / "few_items_check.cpp"), "-o", str(exe)], check=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0 and "few items ok" in proc.stdout, proc.stdout + proc.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("order", [0, 1, 2])  # of the tiles: interleaved ranks, item major, rank outermost
@pytest.mark.parametrize("below", [0, 1 << 30])  # whole tiles where there is a choice, short tiles everywhere
@pytest.mark.parametrize("n_items", [2, 16, 17])
@pytest.mark.parametrize("pair", [(a, b) for a in DTYPES for b in DTYPES], ids=str)
def test_a_few_items(make_world, pair, n_items, order, below):
    """Shards of ``a`` gathered into ``b``, gradients of ``a`` into accumulations of ``b`` (stored, then
    added), published as ``a``; one tile, one element more, one less, and several."""
    import odc_amd
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    a, b = pair
    options = {"short_tiles_below": below, "rank_major": order, "accum_tile_order": order}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        W = 3
        group = make_world(W, 16 << 20)
        registry = SymmBufferRegistry.get_instance()
        gather, red = GatherService(), ReductionService(accumulation_dtype=b, lazy_clear=True)
        gen = torch.Generator().manual_seed(7)
        sizes = [(4096, 1, 4097, 1023, 20_483)[i % 5] + i // 5 for i in range(n_items)]
        shards = [[torch.randn(n, generator=gen).to(a) for _ in range(W)] for n in sizes]
        sources = []
        for i, parts in enumerate(shards):
            put_shards(registry, ("p", i), parts)
            sources.append(registry.get_symm_buffer(("p", i)))
        outs = [torch.full((W * n,), float("nan"), dtype=b, device="cuda") for n in sizes]
        with odc_amd.virtual_rank(2):  # the walk starts at another rank
            gather.gather_into_tensors(outs, sources, group)
        for out, parts in zip(outs, shards):
            assert_bit_equal(out, oracle.gather(parts) if a == b else oracle.gather_cast(parts, b))

        for i, n in enumerate(sizes):
            red.register(i, (n,), a, b, group)
        want = [[torch.zeros(n, dtype=b) for _ in range(W)] for n in sizes]
        red.clear_accumulations()
        for _ in range(2):
            grads = [torch.randn(W * n, generator=gen).to(a) for n in sizes]
            red.scatter_accumulate_multi(list(range(n_items)), [g.cuda() for g in grads], group)
            for accs, grad in zip(want, grads):
                oracle.scatter_accumulate(accs, grad)
        for i, accs in enumerate(want):
            for r, got in enumerate(red.get_peer_accumulations(i)):
                assert_bit_equal(got, accs[r], f"item {i} rank {r}")
        for out, accs in zip(red.publish(list(range(n_items)), out_dtype=a, divisor=4.0), want):
            assert_bit_equal(out, (accs[0].float() / 4.0).to(b).to(a))
        red.lazy_clear = False
        red.clear_accumulations()
        for i in range(n_items):
            assert not any(acc.any() for acc in red.get_peer_accumulations(i))
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
