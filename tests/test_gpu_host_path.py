"""The extension module that reads the tensors of a call (odc_torch.cpp): what it accepts, what it
refuses and how, and that a service never uses what it noted about buffers that are gone."""

import numpy as np
import pytest
import torch

from helpers import assert_bit_equal, put_shards
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu


def test_sequences_of_any_kind_and_mixed_forms(make_world):
    """Tuples, numpy sizes, duplicate keys, empty slices and a key in both store and add form."""
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    W, sizes = 4, [5, 0, 4097]
    group = make_world(W, 1 << 20)
    gather, red = GatherService(), ReductionService(accumulation_dtype=torch.float32, lazy_clear=True)
    gen = torch.Generator().manual_seed(3)
    shards = [torch.randn(sum(sizes), generator=gen).bfloat16() for _ in range(W)]
    source = put_shards(SymmBufferRegistry.get_instance(), "g", shards)
    offsets = np.cumsum([0] + sizes[:-1])
    outs = tuple(torch.empty(W * n, dtype=torch.bfloat16, device="cuda") for n in sizes)
    gather.gather_slices(outs, source, offsets, tuple(np.array(sizes)), group)
    for out, off, n in zip(outs, offsets, sizes):
        assert_bit_equal(out, oracle.gather([s[off : off + n] for s in shards]))

    grads = [torch.randn(W * 7, generator=gen).bfloat16() for _ in range(3)]
    red.scatter_accumulate("a", grads[0].cuda(), group)
    red.clear_accumulations()  # lazily: the next add of "a" stores
    red.scatter_accumulate_multi(("a", "b", "a"), tuple(g.cuda() for g in grads), group)
    want = {"a": [torch.zeros(7) for _ in range(W)], "b": [torch.zeros(7) for _ in range(W)]}
    for key, g in zip("aba", grads):
        oracle.scatter_accumulate(want[key], g)
    for key, accs in want.items():
        for r, got in enumerate(red.get_peer_accumulations(key)):
            assert_bit_equal(got, accs[r], f"{key} rank {r}")


def test_refusals(make_world):
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    W = 4
    group = make_world(W, 1 << 20)
    registry = SymmBufferRegistry.get_instance()
    shard = registry.allocate_symm_buffer("s", (8,), torch.bfloat16)
    gather, red = GatherService(), ReductionService(accumulation_dtype=torch.float32)
    full = torch.zeros(W * 8, dtype=torch.bfloat16, device="cuda")
    for outs, inputs in (([full[:-1]], [shard]), ([full.view(2, -1).t()], [shard]), ([full.cpu()], [shard]),
                         ([full, full.float()], [shard, shard])):
        with pytest.raises(AssertionError):
            gather.gather_into_tensors(outs, inputs, group)
    with pytest.raises(ValueError, match="symmetric arena"):
        gather.gather_into_tensor(full, torch.zeros(8, dtype=torch.bfloat16, device="cuda"), group)
    with pytest.raises(TypeError):
        gather.gather_into_tensors([None], [shard], group)
    with pytest.raises(TypeError, match="gather supports bf16/fp16/fp32, not Double"):
        gather.gather_into_tensor(full.double(), shard, group)
    red.register("k", (8,), torch.bfloat16, torch.float32, group)
    for grads, valid in (([full.cpu()], None), ([full[:-1]], None), ([full.view(2, -1)], None),
                         ([torch.cat([full, full])], None), ([full], [W * 8 + 1])):
        with pytest.raises(AssertionError):
            red.scatter_accumulate_multi(["k"], grads, group, valid_numels=valid)
    with pytest.raises(AssertionError):
        red.scatter_accumulate_multi(["unknown"], [full], group, valid_numels=[3])
    with pytest.raises(AssertionError):
        red.scatter_accumulate_slices("k", [full, full], [0, 4], [4, 8], group)
    for peer in red.get_peer_accumulations("k"):
        assert not peer.any()


def test_counts_and_their_limits(make_world):
    """Valid sizes go through int() and the list may be longer than the keys; negative sizes and
    offsets are assertions, and nothing is written by a refused call."""
    from odc_amd import GatherService, ReductionService, SymmBufferRegistry

    W = 2
    group = make_world(W, 1 << 20)
    gather, red = GatherService(), ReductionService(accumulation_dtype=torch.float32)
    red.register("k", (4,), torch.bfloat16, torch.float32, group)
    grad = torch.arange(8, dtype=torch.bfloat16, device="cuda")
    for count in (7.0, torch.tensor(7), np.int32(7)):
        red.scatter_accumulate_multi(["k"], [grad], group, valid_numels=[count, 99])
    want = torch.arange(8, dtype=torch.float32) * 3
    want[7] = 0
    for r, got in enumerate(red.get_peer_accumulations("k")):
        assert_bit_equal(got, want.view(W, -1)[r])
    shard = SymmBufferRegistry.get_instance().allocate_symm_buffer("s", (8,), torch.bfloat16)
    for call in (lambda: gather.gather_slices([grad], shard, [-1], [4], group),
                 lambda: gather.gather_slices([grad], shard, [5], [4], group),
                 lambda: red.scatter_accumulate_slices("k", [grad], [-1], [4], group),
                 lambda: red.scatter_accumulate_multi(["k"], [grad], group, valid_numels=[-1]),
                 lambda: red.scatter_accumulate_multi(["k"], [grad], group, valid_numels=[])):
        with pytest.raises(AssertionError):
            call()
    for r, got in enumerate(red.get_peer_accumulations("k")):
        assert_bit_equal(got, want.view(W, -1)[r])


def test_buffers_that_are_gone_are_not_used(make_world):
    """A registry that freed its buffers voids what services noted about them, in the same arena."""
    from odc_amd import ReductionService, SymmBufferRegistry

    W = 2
    group = make_world(W, 1 << 20)
    red = ReductionService(accumulation_dtype=torch.float32)
    grad = torch.ones(W * 64, dtype=torch.bfloat16, device="cuda")
    red.scatter_accumulate("k", grad, group)
    red.scatter_accumulate_slices("s", [grad], [0], [64], group)
    SymmBufferRegistry.get_instance().finalize()
    other = SymmBufferRegistry.get_instance().allocate_symm_buffer("other", (4096,), torch.float32)
    other.zero_()
    for call in (lambda: red.scatter_accumulate("k", grad, group), red.clear_accumulations,
                 lambda: red.scatter_accumulate_slices("s", [grad], [0], [64], group)):
        with pytest.raises(KeyError):
            call()
    assert not other.any()
