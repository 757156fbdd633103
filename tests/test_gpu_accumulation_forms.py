"""Accumulations and converted outputs that stay in the caches, written with plain stores and through the L2s:
launches at the edges of their tiles give the oracle's bits, and nothing beside what they write is written."""

import pytest
import torch

from helpers import assert_bit_equal, put_shards
from odc_amd import _native
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("plain", [0, 1 << 40], ids=["written through", "plain"])
@pytest.mark.parametrize("grad_dtype,acc_dtype", [(BF16, F32), (F32, F32), (BF16, BF16), (F16, F32), (F32, F16)])
@pytest.mark.parametrize("sizes", [[8 * 4096], [1023, 1024, 1025, 4096 + 3], [640] * 17, [40 * 4096 + 5] * 2],
                         ids=lambda sizes: f"{len(sizes)}x{max(sizes)}")
def test_bits_and_bounds(make_world, sizes, grad_dtype, acc_dtype, plain):
    from odc_amd import ReductionService, SymmBufferRegistry

    options = {"plain_accumulation_bytes": plain, "through_store_bytes": 1 << 40, "cached_arena_bytes": 1 << 40,
               "cached_gradient_bytes": 1 << 40}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        W, gap = 3, 68  # elements between the slices: what lies there stays as it is
        offsets, total = [], gap
        for n in sizes:
            offsets.append(total)
            total += n + gap
        group = make_world(W, total * 4 + (1 << 20))
        reduction = ReductionService(accumulation_dtype=acc_dtype)
        reduction.register("k", (total,), grad_dtype, acc_dtype, group)
        peers = SymmBufferRegistry.get_instance().peer_tensors["rs_accumulation_k"]
        for peer in peers:
            peer.fill_(7)
        want = [torch.full((total,), 7, dtype=acc_dtype) for _ in range(W)]
        host = _native.load_torch_binding()
        gen = torch.Generator().manual_seed(3)
        for store in (False, True, False):
            grads = [torch.randn(W * n, generator=gen).to(grad_dtype) for n in sizes]
            on_device = [g.cuda() for g in grads]
            items = host.slice_layout(offsets, sizes).batch(reduction._table["k"], W, on_device)
            reduction._launch(("k",), items, len(sizes), items.grad_code, items.acc_code, store)
            for g, o, n in zip(grads, offsets, sizes):
                slices = [w[o : o + n] for w in want]
                if store:
                    for piece in slices:
                        piece.zero_()
                oracle.scatter_accumulate(slices, g)
            reduction.sync(group)
            for r, peer in enumerate(peers):
                assert_bit_equal(peer, want[r], f"rank {r} store {store}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)


@pytest.mark.parametrize("plain", [0, 1 << 40], ids=["written through", "plain"])
@pytest.mark.parametrize("src,dst", [(F32, BF16), (BF16, F32), (F16, BF16)])
@pytest.mark.parametrize("sizes", [[8 * 4096], [1023, 1024, 1025, 4096 + 3], [640] * 17, [40 * 4096 + 5] * 2],
                         ids=lambda sizes: f"{len(sizes)}x{max(sizes)}")
def test_converted_outputs(make_world, sizes, src, dst, plain):
    from odc_amd import GatherService, SymmBufferRegistry

    options = {"plain_output_bytes": plain, "cached_arena_bytes": 1 << 40}
    saved = {name: _native.get_option(name) for name in options}
    try:
        for name, value in options.items():
            _native.set_option(name, value)
        W, pad = 3, 67
        group = make_world(W, sum(sizes) * 4 + (2 << 20))
        gen = torch.Generator().manual_seed(4)
        shards = [[torch.randn(n, generator=gen).to(src) for _ in range(W)] for n in sizes]
        sources = [put_shards(SymmBufferRegistry.get_instance(), ("p", i), s) for i, s in enumerate(shards)]
        around = [torch.full((W * n + 2 * pad,), 7.0, dtype=dst, device="cuda") for n in sizes]
        GatherService().gather_into_tensors([t[pad : pad + W * n] for t, n in zip(around, sizes)], sources, group)
        for t, s, n in zip(around, shards, sizes):
            want = torch.full((W * n + 2 * pad,), 7.0, dtype=dst)
            want[pad : pad + W * n] = oracle.gather_cast(s, dst)
            assert_bit_equal(t, want, f"size {n}")
    finally:
        for name, value in saved.items():
            _native.set_option(name, value)
