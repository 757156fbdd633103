"""Whoever replaces ``ReductionService.sync`` sees every end of a minibatch, in front of the gradients: a subclass, an
attribute of the service or of the class, and a service that has no ``syncing``."""

import types

import pytest

from odc_amd import ReductionService
from odc_amd.fsdp import fsdp1, fsdp2

pytestmark = pytest.mark.usefixtures("launch_list")


def _minibatch_ends(module, monkeypatch, service, calls):
    monkeypatch.setattr(module, "reduction_service", service)
    group = types.SimpleNamespace(pg="pg", name="unit", update_gradients=lambda: calls.append("publish"))
    if module is fsdp1:
        monkeypatch.setattr(fsdp1, "_publish_gradients", lambda m, s: calls.append("publish"))
    module.pre_optimizer_step(types.SimpleNamespace(process_group="pg", _odc_param_groups=[group]))


@pytest.mark.parametrize("module", [fsdp1, fsdp2])
@pytest.mark.parametrize("how", ["class", "class, by a service that is there already", "subclass", "attribute", "no syncing", "proxy"])
def test_a_replaced_sync_is_called(monkeypatch, module, how):
    calls, service = [], ReductionService()
    original = ReductionService.sync

    def traced(self, pg=None):
        calls.append(("sync", pg))
        return original(self, pg)

    if how.startswith("class"):
        monkeypatch.setattr(ReductionService, "sync", traced)
        if how == "class":
            service = ReductionService()
    elif how == "subclass":
        service = type("Service", (ReductionService,), {"sync": traced})()
    elif how == "attribute":
        service.sync = lambda pg=None: traced(service, pg)
    elif how == "no syncing":
        service = types.SimpleNamespace(sync=lambda pg=None: calls.append(("sync", pg)))
    else:
        class Proxy:
            def __init__(self, inner):
                self.inner = inner

            def __getattr__(self, name):
                return getattr(self.inner, name)

            def sync(self, pg=None):
                calls.append(("sync", pg))
                self.inner.sync(pg)

        service = Proxy(service)
    _minibatch_ends(module, monkeypatch, service, calls)
    assert calls == [("sync", "pg"), "publish"]


@pytest.mark.parametrize("module", [fsdp1, fsdp2])
def test_the_service_as_it_is_publishes_first(monkeypatch, module):
    service, calls = ReductionService(), []
    service.dispatched_tasks = 3
    group = types.SimpleNamespace(pg="pg", name="unit", update_gradients=lambda: calls.append(service.dispatched_tasks))
    monkeypatch.setattr(fsdp1, "_publish_gradients", lambda m, s: group.update_gradients())
    monkeypatch.setattr(module, "reduction_service", service)
    module.pre_optimizer_step(types.SimpleNamespace(process_group="pg", _odc_param_groups=[group]))
    assert calls == [3] and service.dispatched_tasks == 0


def test_a_sync_that_raises_keeps_the_gradients_from_being_handed_out(monkeypatch):
    calls = []

    class Service(ReductionService):
        def sync(self, pg=None):
            raise TimeoutError("a rank is missing")

    with pytest.raises(TimeoutError):
        _minibatch_ends(fsdp2, monkeypatch, Service(), calls)
    assert calls == []
