"""Clears written through the L2s and with plain stores: the spans are zero, whatever lies between them is as
it was."""

import pytest
import torch

from odc_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("line", [0, 1 << 40], ids=["plain", "written through"])
@pytest.mark.parametrize("sizes", [
    [16_384], [16_383, 16_384, 16_385], [4, 252, 256, 0, 5 * 16_384 + 12], [1028] * 17, [16_384 + 128] * 113,
], ids=lambda sizes: f"{len(sizes)}x{max(sizes)}")  # bytes: one tile and its neighbours; few, 16+ and 112+ spans
def test_zeros_and_bounds(make_world, sizes, line):
    import ctypes

    from odc_amd import SymmBufferRegistry
    from odc_amd.primitives.utils import get_world

    saved = _native.get_option("through_clear_bytes")
    try:
        _native.set_option("through_clear_bytes", line)
        W, gap = 3, 1024 + 4
        total = sum(sizes) + gap * (len(sizes) + 1)
        make_world(W, total + (1 << 20))
        registry, arena = SymmBufferRegistry.get_instance(), get_world().arena
        registry.allocate_symm_buffer("all", (total,), torch.uint8)
        for peer in registry.peer_tensors["all"]:
            peer.fill_(7)
        start, spans, at = registry.get_offset("all"), [], gap
        for n in sizes:
            spans.append((start + at, n))
            at += n + gap
        array = (_native.Span * len(spans))(*spans)
        _native.check(_native.load().odc_clear(arena.handle, array, len(spans), ctypes.c_void_p(
            torch.cuda.current_stream().cuda_stream)))
        want = torch.full((total,), 7, dtype=torch.uint8)
        for offset, n in spans:
            want[offset - start : offset - start + n] = 0
        for r, peer in enumerate(registry.peer_tensors["all"]):
            assert torch.equal(peer.cpu(), want), f"rank {r}"
    finally:
        _native.set_option("through_clear_bytes", saved)
