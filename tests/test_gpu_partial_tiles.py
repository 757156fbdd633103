"""The tiles of a launch that are not whole: the last one of a segment, gradients that end inside
a vector, accumulations and outputs off their vectors' alignment. Bit-exact against the oracle."""

import ctypes

import pytest
import torch

from helpers import assert_bit_equal
from oracle import odc_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grad_dtype,acc_dtype", [
    (torch.bfloat16, torch.float32), (torch.float32, torch.float32), (torch.float16, torch.float32),
    (torch.bfloat16, torch.bfloat16),
])
@pytest.mark.parametrize("shard", [3, 4, 1023, 4095, 4096, 4097, 8192 + 2050])
def test_gradient_ends_anywhere_in_a_vector(make_world, grad_dtype, acc_dtype, shard):
    """Nine accumulations in one launch whose gradients stop 0..8 elements short of W * shard: the
    cut quad, the quads before it, and the zero padding behind it (which is added as +0)."""
    from odc_amd import ReductionService

    W = 2
    group = make_world(W, 9 * (shard * 4 + 32768) + (1 << 20))
    reduction = ReductionService(accumulation_dtype=acc_dtype)
    gen = torch.Generator().manual_seed(shard)
    keys, valid, want = list(range(9)), [W * shard - min(k, W * shard) for k in range(9)], []
    for key in keys:
        reduction.register(key, (shard,), grad_dtype, acc_dtype, group)
        start = torch.randn(W, shard, generator=gen).to(acc_dtype)
        start[:, -1] = -0.0  # padding turns -0 into +0
        for r, peer in enumerate(reduction.get_peer_accumulations(key)):
            peer.copy_(start[r])
        want.append(list(start.clone()))
    grads = [torch.randn(n, generator=gen).to(grad_dtype) for n in valid]
    reduction.scatter_accumulate_multi(keys, [g.cuda() for g in grads], group, valid_numels=valid)
    reduction.sync(group)
    for key, accs, grad in zip(keys, want, grads):
        oracle.scatter_accumulate(accs, torch.nn.functional.pad(grad, [0, W * shard - grad.numel()]))
        for r, got in enumerate(reduction.get_peer_accumulations(key)):
            assert_bit_equal(got, accs[r], f"{key} elements short, rank {r}")


@pytest.mark.parametrize("acc_dtype,out_dtype", [
    (torch.float32, torch.bfloat16), (torch.float32, torch.float32), (torch.bfloat16, torch.float32),
    (torch.float32, torch.float16),
])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 1027, 4095, 4096, 4097, 12_286])
@pytest.mark.parametrize("acc_lead,out_lead", [(0, 0), (1, 0), (0, 1)])
def test_publish_of_partial_and_misaligned_tiles(make_world, acc_dtype, out_dtype, n, acc_lead, out_lead):
    """odc_publish on [acc_lead, acc_lead + n) into an output that starts out_lead elements into its
    buffer: what lies around either range is left alone."""
    from odc_amd import SymmBufferRegistry, _native
    from odc_amd.primitives.utils import get_world, native_dtype

    make_world(2, 1 << 20)
    registry = SymmBufferRegistry.get_instance()
    registry.allocate_symm_buffer("acc", (n + 8,), acc_dtype)
    acc = registry.peer_tensors["acc"][1]
    gen = torch.Generator().manual_seed(n)
    start = torch.randn(n + 8, generator=gen).to(acc_dtype)
    for divisor in (8.0, 3.0, 1.0):
        acc.copy_(start)
        out = torch.full((n + 8,), 7.0, dtype=out_dtype, device="cuda")
        item = (_native.PublishItem * 1)()
        item[0].acc_offset = registry.get_offset("acc") + acc_lead * acc_dtype.itemsize
        item[0].elems = n
        item[0].out = out.data_ptr() + out_lead * out_dtype.itemsize
        _native.check(_native.load().odc_publish(
            get_world().arena.handle, 1, item, 1, native_dtype(acc_dtype), native_dtype(out_dtype), divisor,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        want_acc, want_out = start.clone(), torch.full((n + 8,), 7.0, dtype=out_dtype)
        piece = want_acc[acc_lead : acc_lead + n]
        want_out[out_lead : out_lead + n] = oracle.fsdp1_publish(piece, divisor, out_dtype)
        assert_bit_equal(acc, want_acc, f"accumulation / {divisor}")
        assert_bit_equal(out, want_out, f"output / {divisor}")
