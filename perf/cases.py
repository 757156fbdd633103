"""The work that a user has this package do, as cases to be measured.

A case is a set of sizes, world size, data types and options; ``run`` is one pass over it through
the public entry points, as a training program calls them. Three kinds of program are covered:

* ``tensors``: the primitives called directly, one key per parameter: ``gather_into_tensor(s)``,
  then ``scatter_accumulate`` / ``scatter_accumulate_multi``, for one or more microbatches, with or
  without the minibatch's ``clear_accumulations`` and final ``publish``;
* ``slices``: the primitives' group form, every parameter a slice of one symmetric buffer
  (``gather_slices``, ``scatter_accumulate_slices``);
* ``fsdp2`` / ``fsdp1``: a whole minibatch of the two FSDP modules: ``pre_minibatch_start``, per
  microbatch one unshard for the forward and one for the backward and one reduction, then
  ``pre_optimizer_step``.
"""

import math
import random
import types
import weakref

import torch

import odc_amd as odc
from odc_amd.fsdp import fsdp1, fsdp2
from odc_amd.primitives.utils import get_world
from odc_amd.workloads import HIDDEN, FFN, KV_HEADS, HEAD_DIM, VOCAB, shard_numel

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
LARGEST_NUMEL = VOCAB * HIDDEN


def _case(kind, world, **over):
    """A case with the options a program leaves alone filled in: bf16 parameters and gradients,
    fp32 accumulations, one microbatch, no clear and publish around it."""
    case = {"kind": kind, "world": world, "shard": "bf16", "compute": "bf16", "reduce": "fp32",
            "microbatches": 1, "minibatch": kind in ("fsdp1", "fsdp2"), "lazy_clear": False,
            "shard_copies": False, "padded": False}
    case.update(over)
    return case


def _layer(hidden=HIDDEN, ffn=FFN, kv=KV_HEADS * HEAD_DIM):
    return {"sizes": "layer", "hidden": hidden, "ffn": ffn, "kv": kv}


def _block(hidden):
    return {"sizes": "block", "hidden": hidden}


def _list(tensors, low, high, sizes_seed=0):
    return {"sizes": "list", "tensors": tensors, "low": low, "high": high, "sizes_seed": sizes_seed}


def listed():
    return [
        # The smallest call there is: one RMSNorm vector of the decoder layer on its own, gathered and
        # its gradient accumulated. Latency, launches and host time are all of it.
        dict(_case("tensors", 8, **_list(1, HIDDEN, HIDDEN)), name="norm_vector_w8"),
        # A flat parameter of 4 Mi elements at W=4, a minibatch of four microbatches: small enough
        # for the caches, where launch gaps and the ramp of each kernel count.
        dict(_case("tensors", 4, microbatches=4, minibatch=True, **_list(1, 1 << 22, 1 << 22)), name="flat_4m_minibatch_w4"),
        # The ordinary call: one microbatch over a decoder layer, nine parameters in one list.
        dict(_case("tensors", 8, **_layer()), name="layer_w8"),
        # The same layer sharded finely: 576 segments from 917 504 elements down to 64.
        dict(_case("tensors", 64, **_layer()), name="layer_w64"),
        # Uneven flat parameters, none divisible by W: unaligned segments, zero padded shards,
        # gradients that end before the padding.
        dict(_case("tensors", 12, padded=True, **_list(40, 4096, 58_720_256)), name="uneven_w12"),
        # The largest single parameter: a token embedding.
        dict(_case("tensors", 8, **_list(1, LARGEST_NUMEL, LARGEST_NUMEL)), name="embedding_w8"),
        # A minibatch over the layer with lazy clears (the first accumulate stores) and the publish.
        dict(_case("tensors", 8, microbatches=4, minibatch=True, lazy_clear=True, **_layer()), name="layer_minibatch_lazy_w8"),
        # The usual mixed precision of FSDP2: fp32 master shards, bf16 compute, fp32 reduction. The
        # gather converts.
        dict(_case("fsdp2", 8, shard="fp32", microbatches=2, **_layer()), name="fsdp2_layer_mixed_w8"),
        # FSDP2 with everything in bf16: no reduce_dtype given, so the accumulation is bf16 too.
        dict(_case("fsdp2", 8, reduce="bf16", microbatches=2, **_layer()), name="fsdp2_layer_bf16_w8"),
        # FSDP2 over one block of a toy transformer of width 256 in full precision: ten small parameters.
        dict(_case("fsdp2", 8, shard="fp32", compute="fp32", microbatches=2, **_block(256)), name="fsdp2_toy_block_fp32_w8"),
        # FSDP1: a flat parameter of odd size under fp16 mixed precision, with the shards kept a
        # second time in fp16 (converted once per minibatch, then gathered as they are).
        dict(_case("fsdp1", 8, shard="fp32", compute="fp16", microbatches=2, shard_copies=True, padded=True,
                   **_list(1, 25_000_001, 25_000_001)), name="fsdp1_flat_fp16_w8"),
        # Many small parameters as slices of one group (biases, norms, adapters): more than one
        # launch's worth of items, most of them less than a tile per rank.
        dict(_case("slices", 16, **_list(300, 64, 65_536)), name="many_small_slices_w16"),
    ]


def _log_uniform(rng, low, high):
    return int(math.exp(rng.uniform(math.log(low), math.log(high))))


def draw(rng):
    kind = rng.choice(["tensors", "tensors", "tensors", "slices", "fsdp2", "fsdp2", "fsdp1"])
    world = rng.choice([2, 4, 8, 8, 12, 16, 32, 64])
    shard, compute, reduce_ = rng.choice([
        ("bf16", "bf16", "fp32"), ("bf16", "bf16", "fp32"), ("bf16", "bf16", "bf16"), ("fp32", "bf16", "fp32"),
        ("fp16", "fp16", "fp32"), ("fp32", "fp16", "fp32"), ("fp32", "fp32", "fp32"),
    ])
    microbatches = rng.randint(1, 3)
    # one pass moves at most what the embedding's does: 14 bytes for each of its elements
    most = 14 * LARGEST_NUMEL // (microbatches * (2 * 8 + 12) + 16)
    form = rng.choice(["one", "layer", "list"]) if kind != "fsdp1" else "one"
    if form == "one":
        n = _log_uniform(rng, 1000, most)
        sizes = _list(1, n, n)
    elif form == "layer":
        hidden = 64 * rng.randint(2, 64)
        heads = rng.choice([1, 2, 4, 8])
        sizes = _layer(hidden, 64 * rng.randint(hidden // 64, 4 * hidden // 64), max(1, hidden // heads))
        if 8 * hidden * hidden + 3 * hidden * sizes["ffn"] > most:
            sizes = _block(hidden // 4)
    else:
        tensors = rng.randint(2, 60) if kind == "tensors" else rng.randint(2, 20) if kind == "fsdp2" else rng.randint(2, 400)
        high = _log_uniform(rng, 1000, max(2000, most // tensors))
        sizes = _list(tensors, max(64, high // rng.choice([4, 64, 1000])), high, rng.randrange(1 << 20))
    minibatch = kind in ("fsdp1", "fsdp2") or (kind == "tensors" and sizes.get("tensors", 9) <= 16 and rng.random() < 0.4)
    return _case(kind, world, shard=shard, compute=compute, reduce=reduce_, microbatches=microbatches, minibatch=minibatch,
                 lazy_clear=minibatch and kind == "tensors" and rng.random() < 0.4,
                 shard_copies=kind in ("fsdp1", "fsdp2") and shard != compute and rng.random() < 0.4,
                 padded=kind in ("slices", "fsdp1") or (kind == "tensors" and rng.random() < 0.5), **sizes)


def _shapes(case):
    """The parameters' shapes."""
    if case["sizes"] == "layer":
        h, f, kv = case["hidden"], case["ffn"], case["kv"]
        return [(h,), (h, h), (kv, h), (kv, h), (h, h), (h,), (f, h), (f, h), (h, f)]
    if case["sizes"] == "block":
        h = case["hidden"]
        return [(h,), (h,), (3 * h, h), (h, h), (h,), (h,), (4 * h, h), (4 * h,), (h, 4 * h), (h,)]
    rng = random.Random(case["sizes_seed"])
    return [(_log_uniform(rng, case["low"], case["high"]) if case["low"] < case["high"] else case["low"],)
            for _ in range(case["tensors"])]


def _numels(case):
    """(valid elements, elements per rank) of every parameter."""
    W, out = case["world"], []
    for shape in _shapes(case):
        n = math.prod(shape)
        if case["kind"] == "fsdp2":
            shard = -(-shape[0] // W) * math.prod(shape[1:])
        elif case["padded"]:
            shard = shard_numel(n, W)
        else:  # callers of the unpadded form pass what divides evenly
            shard = max(1, n // W)
            n = shard * W
        out.append((n, shard))
    return out


def work(case):
    """Per microbatch: the gather reads every shard and writes every full parameter, the
    accumulate reads the valid gradients and reads and writes the accumulations. A minibatch
    starts from zeros (its first accumulate need not read them) and ends with one rank's pass."""
    W, M = case["world"], case["microbatches"]
    sb, cb, rb = (DTYPES[case[k]].itemsize for k in ("shard", "compute", "reduce"))
    valid = sum(n for n, _ in _numels(case))
    full = sum(W * s for _, s in _numels(case))
    gathers = M * (2 if case["kind"] in ("fsdp1", "fsdp2") else 1)
    if case["shard_copies"]:
        nbytes = full * (sb + cb) + gathers * full * 2 * cb
    else:
        nbytes = gathers * full * (sb + cb)
    nbytes += M * (valid * cb + full * 2 * rb)
    if case["minibatch"]:
        nbytes += -full * rb + (full // W) * (2 * rb + (sb if sb != rb else 0))
    return {"bytes": nbytes, "flops": M * full}


def tolerance(case):
    """Every element of a result is a copy, one correctly rounded conversion, or a chain of
    correctly rounded additions in the order of the calls: there is one right answer. Two passes,
    and a pass against the same sums done with torch's fp32 adds, agree in every bit."""
    return "exact"


# ---- preparation --------------------------------------------------------------------------------
class _State:
    """What the program holds: its services, symmetric buffers, gradients and output buffers."""


_live = weakref.WeakSet()  # states whose buffers lie in the present arena
_units = []  # parameter groups and flat parameters of the present arena: their ids are its keys
_serial = 0
_STATES_PER_ARENA = 10


def _rank_bytes(case):
    sb, cb, rb = (DTYPES[case[k]].itemsize for k in ("shard", "compute", "reduce"))
    per_elem = sb + rb + (cb if case["shard_copies"] else 0)
    return sum(s * per_elem + 3 * 16384 + 4096 * 4 for _, s in _numels(case)) + (1 << 20)


def _world_for(case):
    """The symmetric arena, kept from state to state; made anew for another world size."""
    need = _rank_bytes(case) * _STATES_PER_ARENA
    registry = odc.SymmBufferRegistry.get_instance()
    try:
        world = get_world()
    except RuntimeError:
        world = None
    if world is not None:
        fits = world.world_size == case["world"] and world.arena.bytes_per_rank >= need
        if not fits or not len(_live):
            registry.finalize()
            _units.clear()
            _live.clear()
            if not fits or world.arena.bytes_per_rank > 16 * need + (1 << 28):
                odc.finalize_distributed()
                world = None
    if world is None:
        odc.init_nvshmem(world_size=case["world"], symmetric_size=need)
    return get_world()


class _EveryRank:
    """A symmetric buffer of all W ranks as one [W, bytes] array (no copy)."""

    def __init__(self, arena, offset, nbytes):
        self.__cuda_array_interface__ = {"shape": (arena.world_size, nbytes), "typestr": "|u1", "version": 2,
                                         "data": (arena.base + offset, False), "strides": (arena.rank_stride, 1)}


def _every_rank(world, key):
    offset, shape, dtype = odc.SymmBufferRegistry.get_instance().offsets[key]
    mem = _EveryRank(world.arena, offset, shape[0] * dtype.itemsize)
    return torch.as_tensor(mem, device="cuda").view(dtype)


def _fill_shards(key, full, shard, W):
    """Rank r publishes the r-th ``shard`` elements of ``full``, zero padded."""
    registry = odc.SymmBufferRegistry.get_instance()
    registry.get_or_create_symm_buffer(key, (shard,), full.dtype)
    for r, peer in enumerate(registry.peer_tensors[key]):
        piece = full[r * shard : (r + 1) * shard]
        peer[: piece.numel()].copy_(piece)
        peer[piece.numel() :].zero_()


def _views(numels, dtype):
    """One buffer and a view of it for every size, each on a 512-byte boundary as the allocator
    would place it."""
    at, where = 0, []
    for n in numels:
        where.append(at)
        at += -(-n * dtype.itemsize // 512) * 512 // dtype.itemsize
    flat = torch.zeros(max(1, at), dtype=dtype, device="cuda")
    return flat, [flat[a : a + n] for a, n in zip(where, numels)]


def prepare(case, seed):
    global _serial
    _serial += 1
    world = _world_for(case)
    W, s = case["world"], _State()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shard_t, compute_t, reduce_t = (DTYPES[case[k]] for k in ("shard", "compute", "reduce"))
    shapes, numels = _shapes(case), _numels(case)

    def values(shape, scale, dtype):
        return torch.randn(shape, generator=gen, device="cuda").mul_(scale).to(dtype)

    s.case, s.world, s.group = case, W, world.group
    s.valid = [n for n, _ in numels]
    s.shards = [m for _, m in numels]
    sets = min(2, case["microbatches"])
    if case["kind"] == "fsdp2":
        fsdp2.patch_fsdp2(compute_dtype_shards=case["shard_copies"])
        s.gather, s.reduction = fsdp2.get_gather_service(), fsdp2.get_reduction_service()
        s.unit = fsdp2.ParamGroup(shapes, shard_t, s.group, param_dtype=compute_t,
                                  reduce_dtype=None if reduce_t == compute_t else reduce_t, name="unit",
                                  compute_dtype_shards=case["shard_copies"])
        _units.append(s.unit)
        s.unit.load_full_params([values(shape, 0.02, shard_t) for shape in shapes])
        s.module = types.SimpleNamespace(_odc_param_groups=[s.unit])
        s.grads = [[values(shape, 1e-3, compute_t) for shape in shapes] for _ in range(sets)]
        s.unit.reduce(s.grads[0])  # the first microbatch of a program registers the accumulation
        s.accumulations = [_every_rank(world, f"rs_accumulation_{id(s.unit)}")]
    elif case["kind"] == "fsdp1":
        fsdp1.patch_fsdp1(reduce_dtype=reduce_t, compute_dtype_shards=case["shard_copies"])
        fsdp1.unpatch_fsdp1()  # the unit below is driven directly, torch's own classes stay as they are
        s.gather, s.reduction = fsdp1.get_gather_service(), fsdp1.get_reduction_service()
        (valid,), (shard,) = s.valid, s.shards
        s.unit = torch.nn.Parameter(values((valid,), 0.02, shard_t), requires_grad=False)
        _units.append(s.unit)
        _fill_shards(id(s.unit), s.unit.data, shard, W)
        s.unit.data = odc.SymmBufferRegistry.get_instance().get_symm_buffer(id(s.unit))
        s.module = types.SimpleNamespace(process_group=s.group, _gradient_postdivide_factor=float(W),
                                         _all_handles=[types.SimpleNamespace(flat_param=s.unit)])
        s.padded_param = torch.empty(W * shard, dtype=compute_t, device="cuda")
        s.grads = [values((valid,), 1e-3, compute_t) for _ in range(sets)]
        fsdp1.reduce_grad(s.unit, s.grads[0], s.group)
        s.accumulations = [_every_rank(world, f"rs_accumulation_{id(s.unit)}")]
    else:
        s.gather = odc.GatherService()
        s.reduction = odc.ReductionService(accumulation_dtype=reduce_t, lazy_clear=case["lazy_clear"])
        s.params, s.outs = _views([W * m for m in s.shards], compute_t)
        s.grads = [[values((n,), 1e-3, compute_t) for n in s.valid] for _ in range(sets)]
        if case["kind"] == "slices":
            s.key = (_serial, "group")
            s.offsets = [0]
            for m in s.shards:
                s.offsets.append(s.offsets[-1] + m)
            total = s.offsets.pop()
            _fill_shards(s.key, values((W * total,), 0.02, shard_t), total, W)
            s.source = odc.SymmBufferRegistry.get_instance().get_symm_buffer(s.key)
            s.acc_offsets, s.acc_total = fsdp2.tile_aligned_offsets(s.shards)
            s.reduction.register(s.key, (s.acc_total,), compute_t, reduce_t, s.group)
            s.accumulations = [_every_rank(world, f"rs_accumulation_{s.key}")]
        else:
            s.keys = [(_serial, i) for i in range(len(numels))]
            s.sources = []
            for key, n, m in zip(s.keys, s.valid, s.shards):
                _fill_shards(key, values((n,), 0.02, shard_t), m, W)
                s.sources.append(odc.SymmBufferRegistry.get_instance().get_symm_buffer(key))
                s.reduction.register(key, (m,), compute_t, reduce_t, s.group)
            s.accumulations = [_every_rank(world, f"rs_accumulation_{key}") for key in s.keys]
            # a list without padding is passed as it is, a single tensor through the single form
            s.valid_numels = s.valid if case["padded"] else None
            s.single = len(numels) == 1 and not case["padded"]
    _live.add(s)
    return s


# ---- one pass -----------------------------------------------------------------------------------
def _run_tensors(s):
    case, gather, reduction, group = s.case, s.gather, s.reduction, s.group
    if case["minibatch"]:
        reduction.clear_accumulations()
    for m in range(case["microbatches"]):
        grads = s.grads[m % len(s.grads)]
        if s.single:
            gather.gather_into_tensor(s.outs[0], s.sources[0], group)
            reduction.scatter_accumulate(s.keys[0], grads[0], group)
        else:
            gather.gather_into_tensors(s.outs, s.sources, group)
            reduction.scatter_accumulate_multi(s.keys, grads, group, s.valid_numels)
    result = {"params": s.params, "accumulations": s.accumulations}
    if case["minibatch"]:
        result["published"] = reduction.publish(s.keys, out_dtype=DTYPES[case["shard"]], divisor=float(s.world))
    return result


def _run_slices(s):
    for m in range(s.case["microbatches"]):
        s.gather.gather_slices(s.outs, s.source, s.offsets, s.shards, s.group)
        s.reduction.scatter_accumulate_slices(s.key, s.grads[m % len(s.grads)], s.acc_offsets, s.shards, s.group)
    return {"params": s.params, "accumulations": s.accumulations}


def _run_fsdp2(s):
    fsdp2.gather_service, fsdp2.reduction_service = s.gather, s.reduction
    unit = s.unit
    fsdp2.pre_minibatch_start(s.module)
    for m in range(s.case["microbatches"]):
        unit.unshard()  # forward
        unit.reshard()
        params = unit.unshard()  # backward
        unit.reduce(s.grads[m % len(s.grads)])
        unit.reshard()
    fsdp2.pre_optimizer_step(s.module)
    return {"params": params, "grads": unit.sharded_grads, "accumulations": s.accumulations}


def _run_fsdp1(s):
    fsdp1.gather_service, fsdp1.reduction_service = s.gather, s.reduction
    unit = s.unit
    fsdp1.pre_minibatch_start(s.module)
    for m in range(s.case["microbatches"]):
        fsdp1.all_gather_flat_param(s.padded_param, unit.data, s.group, watch=(unit,))  # forward
        fsdp1.all_gather_flat_param(s.padded_param, unit.data, s.group, watch=(unit,))  # backward
        fsdp1.reduce_grad(unit, s.grads[m % len(s.grads)], s.group)
    fsdp1.pre_optimizer_step(s.module)
    return {"params": s.padded_param, "grad": unit.grad, "accumulations": s.accumulations}


_RUN = {"tensors": _run_tensors, "slices": _run_slices, "fsdp2": _run_fsdp2, "fsdp1": _run_fsdp1}


def run(state):
    return _RUN[state.case["kind"]](state)
