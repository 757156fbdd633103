"""Which launches write through the L2s, on dry-run arenas: from which size on, up to which, and by which option."""

import ctypes

import pytest

from odc_amd import _native

W, MiB = 8, 1 << 20
BF16, F32 = _native.DTYPE_BF16, _native.DTYPE_F32


@pytest.fixture
def through():
    """through(kind, bytes written) -> whether the launch, of one item, writes through the L2s; nothing is allocated,
    so all symmetric memory in use fits the cache."""
    lib, handle = _native.load(), ctypes.c_void_p()
    _native.check(lib.odc_arena_create(W, 1 << 30, _native.ODC_ARENA_DRY_RUN, ctypes.byref(handle)))

    def launch(kind, nbytes):
        per_rank, far = nbytes // W, 1 << 40
        accum = (_native.AccumItem * 1)(_native.AccumItem(far, nbytes // 4, 0, per_rank // 4))
        calls = {
            "gather": lambda: lib.odc_gather(handle, (_native.GatherItem * 1)(_native.GatherItem(far, 0, per_rank)), 1, 0, None),
            "accumulate": lambda: lib.odc_scatter_accumulate(handle, accum, 1, BF16, F32, None),
            "store": lambda: lib.odc_scatter_store(handle, accum, 1, BF16, F32, None),
            "clear": lambda: lib.odc_clear(handle, (_native.Span * 1)((0, per_rank)), 1, None),
        }
        _native.set_option("dry_run_reset", 0)
        _native.check(calls[kind]())
        assert _native.get_option("dry_run_launches") == 1
        return bool(_native.get_option("dry_run_through_launches"))

    names = ("plain_output_bytes", "cached_output_bytes", "plain_accumulation_bytes", "through_store_bytes",
             "through_clear_bytes", "cached_gradient_bytes", "cached_arena_bytes")
    saved = {name: _native.get_option(name) for name in names}
    launch.arena = handle
    yield launch
    for name, value in saved.items():
        _native.set_option(name, value)
    _native.check(lib.odc_arena_destroy(handle))


@pytest.mark.parametrize("kind,sizes", [
    ("gather", {3 * MiB: False, 3 * MiB + 128: True, 64 * MiB: True, 64 * MiB + 128: False}),
    ("accumulate", {3 * MiB: False, 3 * MiB + 128: True, 256 * MiB: True, 256 * MiB + 128: False}),
    ("store", {3 * MiB: False, 3 * MiB + 128: True, 44 * MiB: True, 44 * MiB + 128: False, 48 * MiB: False, 64 * MiB: False}),
    ("clear", {4096: True, 256 * MiB: True, 256 * MiB + 128: False}),
])
def test_lines(through, kind, sizes):
    """(an accumulate's end where its gradient, of half the bytes, no longer fits)"""
    assert {n: through(kind, n) for n in sizes} == sizes


def test_accumulations_and_outputs_have_options_of_their_own(through):
    """A program whose gathered parameters are not read soon streams them ("cached_output_bytes" = 0); its stores and
    accumulates stay as they are."""
    for name, value in {"cached_output_bytes": 0, "plain_output_bytes": 1 << 40}.items():
        _native.set_option(name, value)
    assert not through("gather", 16 * MiB)
    assert through("store", 16 * MiB) and through("accumulate", 16 * MiB)
    _native.set_option("through_store_bytes", 0)
    assert not through("store", 16 * MiB) and through("accumulate", 16 * MiB)
    _native.set_option("plain_accumulation_bytes", 1 << 40)
    assert not through("accumulate", 16 * MiB) and through("clear", 16 * MiB)


def test_accumulations_that_do_not_stay_in_the_caches(through):
    assert through("accumulate", 16 * MiB) and through("store", 16 * MiB)
    _native.set_option("cached_gradient_bytes", 8 * MiB - 1)
    assert not through("accumulate", 16 * MiB) and not through("store", 16 * MiB)
    _native.set_option("cached_gradient_bytes", 8 * MiB)
    assert through("accumulate", 16 * MiB) and through("store", 16 * MiB)
    _native.check(_native.load().odc_arena_alloc(through.arena, 25 * MiB, ctypes.byref(ctypes.c_uint64())))  # of every rank
    assert not through("accumulate", 16 * MiB) and not through("store", 16 * MiB)
    assert through("gather", 16 * MiB)
