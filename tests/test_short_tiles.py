"""Short tiles: their geometry by brute force on the CPU, how launches are planned in them on a
dry-run arena, and the kernels at the edges of a short tile against the oracle."""

import ctypes
import subprocess
from pathlib import Path

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

ROOT = Path(__file__).resolve().parent.parent


def test_short_tile_geometry(tmp_path):
    exe = tmp_path / "short_tile_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-Wno-unknown-pragmas", f"-I{ROOT / 'odc_amd' / 'csrc'}",
                    str(ROOT / "tests" / "cpu" / "short_tile_check.cpp"), "-o", str(exe)], check=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0 and "short tiles ok" in proc.stdout, proc.stdout + proc.stderr


@pytest.mark.parametrize("shard,acc_dtype,tiles", [
    (1024, _native.DTYPE_F32, 1), (1025, _native.DTYPE_F32, 2), (200_000, _native.DTYPE_F32, 196),  # always short
    (4096, _native.DTYPE_BF16, 4), (40 * 4096, _native.DTYPE_BF16, 40),  # short below 32 whole tiles per segment
])
def test_plans_in_short_tiles(shard, acc_dtype, tiles):
    W, lib, handle = 4, _native.load(), ctypes.c_void_p()
    _native.check(lib.odc_arena_create(W, 1 << 30, _native.ODC_ARENA_DRY_RUN, ctypes.byref(handle)))
    _native.set_option("dry_run_reset", 0)
    item = (_native.AccumItem * 1)(_native.AccumItem(1 << 33, W * shard, 0, shard))
    _native.check(lib.odc_scatter_accumulate(handle, item, 1, _native.DTYPE_BF16, acc_dtype, None))
    assert _native.get_option("dry_run_tiles") == _native.get_option("dry_run_workgroups") == W * tiles
    _native.check(lib.odc_arena_destroy(handle))


@pytest.mark.gpu
@pytest.mark.parametrize("below,few", [(0, 0), (1 << 30, 0), (1 << 30, 1 << 30)])  # whole tiles, short ones, few short ones
@pytest.mark.parametrize("dtypes", [
    (torch.bfloat16, torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16, torch.bfloat16),
    (torch.float32, torch.float32, torch.float32), (torch.float16, torch.float32, torch.float16),
], ids=lambda d: "-".join(str(x).rsplit(".", 1)[-1] for x in d))
def test_kernels_at_the_edges_of_a_short_tile(make_world, below, few, dtypes):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    shard_dtype, compute_dtype, acc_dtype = dtypes
    saved = {name: _native.get_option(name) for name in ("short_tiles_below", "few_tiles")}
    _native.set_option("short_tiles_below", below)
    _native.set_option("few_tiles", few)
    try:
        W, sizes = 3, [1, 63, 1023, 1024, 1025, 2047, 2049, 4095, 4097, 20_481]
        group = make_world(W, 4 << 20)
        registry = SymmBufferRegistry.get_instance()
        gather, red = GatherService(), ReductionService(accumulation_dtype=acc_dtype, lazy_clear=True)
        gen = torch.Generator().manual_seed(11)
        shards = [[torch.randn(n, generator=gen).to(shard_dtype) for _ in range(W)] for n in sizes]
        sources = [put_shards(registry, ("p", i), s) for i, s in enumerate(shards)]
        outs = [torch.full((W * n,), float("nan"), dtype=compute_dtype, device="cuda") for n in sizes]
        gather.gather_into_tensors(outs, sources, group)
        for out, s in zip(outs, shards):
            assert_bit_equal(out, oracle.gather(s) if shard_dtype == compute_dtype else oracle.gather_cast(s, compute_dtype))

        keys = list(range(len(sizes)))
        for key, n in zip(keys, sizes):
            red.register(key, (n,), compute_dtype, acc_dtype, group)
        want = [[torch.zeros(n, dtype=acc_dtype) for _ in range(W)] for n in sizes]
        red.clear_accumulations()
        for m in range(3):  # the store form, then read-modify-write; gradients that end early
            valid = [max(0, W * n - m) for n in sizes]
            grads = [torch.randn(v, generator=gen).to(compute_dtype) for v in valid]
            red.scatter_accumulate_multi(keys, [g.cuda() for g in grads], group, valid_numels=valid)
            for accs, g, n in zip(want, grads, sizes):
                oracle.scatter_accumulate(accs, torch.nn.functional.pad(g, [0, W * n - g.numel()]))
        red.sync(group)
        for key, accs in zip(keys, want):
            for r, got in enumerate(red.get_peer_accumulations(key)):
                assert_bit_equal(got, accs[r], f"size {sizes[key]} rank {r}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)


@pytest.mark.gpu
@pytest.mark.parametrize("order", [0, 1, 2])  # of the tiles: interleaved ranks, item major, rank outermost
@pytest.mark.parametrize("n", [2, 63, 64, 65, 66, 111, 112, 113])
def test_every_item_is_found_among_few_tiles(make_world, n, order):
    """The search of launches of few tiles reads the prefix table in two halves of one entry per lane:
    item counts around a half and around a whole launch, items of none to three tiles."""
    from odc_amd import GatherService, ReductionService

    options = {"rank_major": order, "accum_tile_order": order, "few_tiles": 1 << 30}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        from odc_amd import SymmBufferRegistry

        W, sizes = 3, [(701 * i + 5) % 2500 for i in range(n)]
        offsets = [sum(sizes[:i]) for i in range(n)]
        group = make_world(W, 4 << 20)
        gather, red = GatherService(), ReductionService(accumulation_dtype=torch.float32)
        gen = torch.Generator().manual_seed(n)
        shards = [torch.randn(sum(sizes), generator=gen).bfloat16() for _ in range(W)]
        source = put_shards(SymmBufferRegistry.get_instance(), "p", shards)
        outs = [torch.full((W * m,), float("nan"), dtype=torch.bfloat16, device="cuda") for m in sizes]
        gather.gather_slices(outs, source, offsets, sizes, group)
        for out, off, m in zip(outs, offsets, sizes):
            assert_bit_equal(out, oracle.gather([s[off : off + m] for s in shards]))
        grads = [torch.randn(W * m, generator=gen).bfloat16() for m in sizes]
        red.scatter_accumulate_slices("g", [g.cuda() for g in grads], offsets, sizes, group)
        for r, got in enumerate(red.get_peer_accumulations("g")):
            assert_bit_equal(got, torch.cat([g.view(W, -1)[r] if g.numel() else g for g in grads]).float(), f"rank {r}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)


@pytest.mark.gpu
@pytest.mark.parametrize("few", [0, 1 << 30])  # the binary search, the table read at once
@pytest.mark.parametrize("acc_dtype,out_dtype", [
    (torch.float32, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.float16),
])
@pytest.mark.parametrize("n", [1, 2, 64, 66, 112, 113])
def test_publish_of_many_items_in_short_tiles(make_world, n, acc_dtype, out_dtype, few):
    """Items of none to a few tiles and around the edges of one, in one launch and in two."""
    from odc_amd import SymmBufferRegistry
    from odc_amd.primitives.utils import get_world, native_dtype

    make_world(2, 8 << 20)
    registry = SymmBufferRegistry.get_instance()
    sizes = [[1023, 1024, 1025, 2049, 4097, 0, 5, 3070][i % 8] for i in range(n)]
    starts = [sum(-(-m // 64) * 64 for m in sizes[:i]) for i in range(n)]
    total = starts[-1] + sizes[-1] + 64
    registry.allocate_symm_buffer("acc", (total,), acc_dtype)
    acc = registry.peer_tensors["acc"][1]
    start = torch.randn(total, generator=torch.Generator().manual_seed(n)).to(acc_dtype)
    saved = _native.get_option("few_tiles")
    _native.set_option("few_tiles", few)
    try:
        for divisor in (8.0, 3.0, 1.0):
            acc.copy_(start)
            outs = [torch.full((m + 8,), 7.0, dtype=out_dtype, device="cuda") for m in sizes]
            items = (_native.PublishItem * n)(*[
                _native.PublishItem(registry.get_offset("acc") + at * acc_dtype.itemsize, m, out.data_ptr())
                for at, m, out in zip(starts, sizes, outs)])
            _native.check(_native.load().odc_publish(
                get_world().arena.handle, 1, items, n, native_dtype(acc_dtype), native_dtype(out_dtype), divisor,
                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
            want = start.clone()
            for at, m, out in zip(starts, sizes, outs):
                copy = torch.full((m + 8,), 7.0, dtype=out_dtype)
                if m:
                    copy[:m] = oracle.fsdp1_publish(want[at : at + m], divisor, out_dtype)
                assert_bit_equal(out, copy, f"output at {at} / {divisor}")
            assert_bit_equal(acc, want, f"accumulations / {divisor}")
    finally:
        _native.set_option("few_tiles", saved)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1024 * 4096, 1024 * 4096 + 1, 1025 * 4096 + 1027])  # the longest in short tiles, then whole ones
def test_publish_of_16_bit_accumulations_around_the_line(make_world, n):
    from odc_amd import ReductionService

    group = make_world(2, 32 << 20)
    red = ReductionService(accumulation_dtype=torch.bfloat16)
    red.register("k", (n,), torch.bfloat16, torch.bfloat16, group)
    start = torch.randn(n, generator=torch.Generator().manual_seed(n)).bfloat16()
    red.get_accumulation("k").copy_(start)
    (out,) = red.publish(["k"], out_dtype=torch.float32, divisor=3.0)
    assert_bit_equal(out, oracle.fsdp1_publish(start, 3.0, torch.float32))
    assert_bit_equal(red.get_accumulation("k"), start)
