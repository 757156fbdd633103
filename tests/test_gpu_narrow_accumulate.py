"""Launches of 16-bit gradients into 16-bit accumulations that are cut into whole tiles: the store, and
the read-modify-write on either side of the line up to which gradients are read through the caches."""

import pytest
import torch

from helpers import assert_bit_equal
from odc_amd import _native
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cached", [0, 1 << 40])  # bytes of gradient up to which it is cached
@pytest.mark.parametrize("grad_dtype,acc_dtype", [
    (torch.bfloat16, torch.bfloat16), (torch.float16, torch.bfloat16), (torch.float16, torch.float16),
], ids=str)
@pytest.mark.parametrize("sizes", [[32 * 4096], [40 * 4096 + 1], [33 * 4096 + 4095, 45 * 4096 - 1, 7, 64 * 4096]], ids=str)
def test_whole_tiles(make_world, sizes, grad_dtype, acc_dtype, cached):
    from odc_amd import ReductionService

    W, saved = 3, {name: _native.get_option(name) for name in ("cached_gradient_bytes", "short_tiles_below")}
    try:
        _native.set_option("cached_gradient_bytes", cached)
        _native.set_option("short_tiles_below", 0)
        group = make_world(W, 4 << 20)
        red = ReductionService(accumulation_dtype=acc_dtype, lazy_clear=True)
        keys = list(range(len(sizes)))
        for key, n in zip(keys, sizes):
            red.register(key, (n,), grad_dtype, acc_dtype, group)
        gen = torch.Generator().manual_seed(5)
        want = [[torch.zeros(n, dtype=acc_dtype) for _ in range(W)] for n in sizes]
        red.clear_accumulations()
        for m in range(3):  # the store form, then read-modify-write; gradients that end early
            valid = [W * n - 3 * m if n > 7 else W * n for n in sizes]
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
