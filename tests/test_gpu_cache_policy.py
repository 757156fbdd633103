"""Every cached / nontemporal form of the kernels gives the oracle's bits, whichever the sizes of a
launch and of the arena would pick."""

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu

OPTIONS = ("cached_arena_bytes", "cached_output_bytes", "cached_gradient_bytes")
SIZES = [1, 63, 4096, 4099, 12_290]  # elements per rank: less than a tile, a tile, ragged tails


@pytest.mark.parametrize("grad_dtype,acc_dtype", [
    (torch.bfloat16, torch.float32), (torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
])
@pytest.mark.parametrize("lines", [(0, 0, 0), (1 << 40, 0, 0), (0, 1 << 40, 0), (0, 0, 1 << 40), (1 << 40,) * 3])
def test_every_policy(make_world, grad_dtype, acc_dtype, lines):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry, _native

    saved = {name: _native.get_option(name) for name in OPTIONS}
    try:
        for name, value in zip(OPTIONS, lines):
            _native.set_option(name, value)
        W = 3
        group = make_world(W, 4 << 20)
        registry = SymmBufferRegistry.get_instance()
        gather = GatherService()
        reduction = ReductionService(accumulation_dtype=acc_dtype, lazy_clear=True)
        gen = torch.Generator().manual_seed(5)
        shards = [[torch.randn(n, generator=gen) for _ in range(W)] for n in SIZES]
        sources = [put_shards(registry, ("p", i), s) for i, s in enumerate(shards)]
        for dtype in (torch.float32, torch.bfloat16):  # plain and converting
            outs = [torch.full((W * n,), float("nan"), dtype=dtype, device="cuda") for n in SIZES]
            gather.gather_into_tensors(outs, sources, group)
            for out, s in zip(outs, shards):
                assert_bit_equal(out, oracle.gather_cast(s, dtype) if dtype != torch.float32 else oracle.gather(s))

        keys = list(range(len(SIZES)))
        for key, n in zip(keys, SIZES):
            reduction.register(key, (n,), grad_dtype, acc_dtype, group)
        want = [[torch.zeros(n, dtype=acc_dtype) for _ in range(W)] for n in SIZES]
        reduction.clear_accumulations()
        for _ in range(3):  # the store form once, then read-modify-write
            grads = [torch.randn(W * n, generator=gen).to(grad_dtype) for n in SIZES]
            reduction.scatter_accumulate_multi(keys, [g.cuda() for g in grads], group)
            for accs, g in zip(want, grads):
                oracle.scatter_accumulate(accs, g)
        reduction.sync(group)
        for key, accs in zip(keys, want):
            for r, got in enumerate(reduction.get_peer_accumulations(key)):
                assert_bit_equal(got, accs[r], f"key {key} rank {r}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
