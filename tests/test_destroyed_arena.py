"""A service call after the arena is gone. (In a file of its own: the extension reports refusals as
C++ exceptions inside, which a preloaded sanitizer runtime does not let through.)"""

import pytest
import torch

from odc_amd import _native
from odc_amd.primitives import utils


def test_calls_after_the_arena_is_destroyed_are_refused(monkeypatch):
    """The services hand the arena's address to the extension; once the arena is gone there is none
    to hand over, whoever still holds the world."""
    from odc_amd.primitives import gather, scatter_accumulate

    world = utils._VirtualWorld(utils.SymmetricArena(4, 1 << 20, backing=False))
    monkeypatch.setattr(utils, "_world", world)
    for module in (gather, scatter_accumulate):
        monkeypatch.setattr(module, "plain_launch_stream", lambda w: 0)
    monkeypatch.setattr(scatter_accumulate, "_is_capturing", lambda: False)
    red = scatter_accumulate.ReductionService()
    red._accumulation_table(world)["k"] = (0, 8, _native.DTYPE_F32)
    red.accumulation_keys.append("k")
    shard, out = torch.zeros(8), torch.zeros(32)
    with pytest.raises(_native.OdcNativeError):  # alive, but without memory
        red.clear_accumulations()
    with pytest.raises(AssertionError, match="GPU"):
        gather.GatherService().gather_into_tensor(out, shard, world.group)
    world.arena.destroy()
    for call in (red.clear_accumulations, lambda: gather.GatherService().gather_into_tensor(out, shard, world.group)):
        with pytest.raises(RuntimeError, match="finalized"):
            call()
