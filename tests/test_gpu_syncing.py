"""``ReductionService.syncing``: what its block launches comes behind the adds of every stream, and at its end the
host has waited for them."""

import types

import pytest
import torch

from helpers import assert_bit_equal
from oracle import odc_oracle as oracle


@pytest.mark.gpu
@pytest.mark.parametrize("policy", [None, "dedicated"])
def test_publish_behind_adds_of_a_busy_stream(make_world, policy, monkeypatch):
    from odc_amd import ReductionService

    if policy:
        monkeypatch.setenv("ODC_COMM_STREAM", policy)
    W, n = 4, 40_000
    group = make_world(W, 4 << 20)
    service = ReductionService(accumulation_dtype=torch.float32)
    service.register("k", (n,), torch.bfloat16, torch.float32, group)
    gen = torch.Generator().manual_seed(1)
    grads = [torch.randn(W * n, generator=gen).bfloat16() for _ in range(3)]
    on_device = [g.cuda() for g in grads]
    work = [torch.randn(2048, 2048, device="cuda") for _ in grads]
    torch.cuda.synchronize()
    sides = [torch.cuda.Stream() for _ in range(2)]
    for side, g, w in zip((*sides, torch.cuda.current_stream()), on_device, work):
        with torch.cuda.stream(side):
            for _ in range(20):
                torch.mm(w, w).mul_(1e-4)
            service.scatter_accumulate("k", g, group)
    with service.syncing(group):
        (out,) = service.publish(["k"], out_dtype=torch.bfloat16, divisor=float(W))
    assert service.dispatched_tasks == 0
    if not policy:  # (the adds are on the callers' streams)
        assert all(side.query() for side in sides)
    want = torch.zeros(n)
    for g in grads:
        oracle.scatter_accumulate([want] + [torch.zeros(n) for _ in range(W - 1)], g)
    want /= W
    assert_bit_equal(out, want.bfloat16())


@pytest.mark.gpu
def test_a_sync_of_another_thread_during_the_block(make_world):
    """It waits for the adds that the block has yet to wait for, and they are counted until then."""
    import threading

    from odc_amd import ReductionService
    from odc_amd.primitives import utils

    W, n = 4, 40_000
    group = make_world(W, 4 << 20)
    service = ReductionService(accumulation_dtype=torch.float32)
    service.register("k", (n,), torch.bfloat16, torch.float32, group)
    grad = torch.ones(W * n, dtype=torch.bfloat16, device="cuda")
    work, side, seen = torch.randn(2048, 2048, device="cuda"), torch.cuda.Stream(), []
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(40):
            torch.mm(work, work).mul_(1e-4)
        service.scatter_accumulate("k", grad, group)
    with service.syncing(group):
        seen.append(service.dispatched_tasks)
        other = threading.Thread(target=lambda: (service.sync(group), seen.append(side.query())))
        other.start()
        other.join()
    assert seen == [1, True] and service.dispatched_tasks == 0 and not utils._waits
    assert torch.equal(service.get_accumulation("k"), torch.ones(n, device="cuda"))


@pytest.mark.gpu
def test_a_sync_of_the_callers_own_is_called_first(make_world):
    from odc_amd import ReductionService

    calls = []

    class Service(ReductionService):
        def sync(self, pg=None):
            calls.append(("sync", pg))
            super().sync(pg)

    group = make_world(2, 1 << 20)
    with Service().syncing(group):
        calls.append("block")
    assert calls == [("sync", group), "block"]


def test_users_hooks_are_seen():
    from odc_amd.fsdp.fsdp2 import _has_gradient_hooks

    def group(all_reduce_hook=None, hooks=None, reduced=True):
        param = types.SimpleNamespace(sharded_param=types.SimpleNamespace(_post_accumulate_grad_hooks=hooks))
        group = types.SimpleNamespace(fsdp_params=[param])
        if reduced:
            group._odc_reduce_context = {"all_reduce_hook": all_reduce_hook}
        return group

    assert not _has_gradient_hooks(group()) and not _has_gradient_hooks(group(hooks={}, reduced=False))
    assert _has_gradient_hooks(group(all_reduce_hook=print)) and _has_gradient_hooks(group(hooks={0: print}))
