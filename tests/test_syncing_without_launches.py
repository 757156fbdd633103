"""The end of a minibatch with no launch to wait for: ``sync`` touches neither arena nor device then, and neither does
what waits in its place."""

import types

import pytest
import torch

from odc_amd import ReductionService
from odc_amd.fsdp import fsdp1, fsdp2
from odc_amd.primitives import utils


@pytest.fixture
def no_device(monkeypatch, launch_list):
    """No arena, no launches, and every question that needs a device refused (as on a machine without one)."""
    from odc_amd.primitives import scatter_accumulate

    def refuse(*_):
        raise RuntimeError("asked the device")

    monkeypatch.setattr(utils, "_world", None)
    monkeypatch.setattr(scatter_accumulate, "_is_capturing", refuse)
    monkeypatch.setattr(torch.cuda, "current_stream", refuse)


def test_syncing_needs_no_arena(no_device):
    service, ran = ReductionService(), []
    service.sync()
    with service.syncing():
        ran.append(True)
    assert ran and service.dispatched_tasks == 0


@pytest.mark.parametrize("module", [fsdp1, fsdp2])
def test_end_of_a_minibatch_without_units(no_device, monkeypatch, module):
    monkeypatch.setattr(module, "reduction_service", ReductionService())
    module.pre_optimizer_step(types.SimpleNamespace(process_group=None, _all_handles=[], _odc_param_groups=[]))


def test_end_of_a_minibatch_that_reduced_nothing(no_device, monkeypatch):
    """A group of FSDP2, which has nothing to publish."""
    monkeypatch.setattr(fsdp2, "reduction_service", ReductionService())
    group = types.SimpleNamespace(pg=None, name="unit", update_gradients=lambda: None)
    fsdp2.pre_optimizer_step(types.SimpleNamespace(_odc_param_groups=[group]))
