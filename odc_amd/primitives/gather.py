"""On-demand gather: W sharded buffers -> one full flat buffer, one fused HIP launch.

Mirror of ``odc/primitives/gather.py`` (``GatherService.gather_into_tensor``, :76-127,176). The
reference issues W peer ``copy_``s on a side stream; here the same result comes from
``odc_gather`` (include/odc_hip.h), whose work list covers all W shards of all tensors of the
call. The inter-node NVSHMEM branch of the reference (:129-175) has no counterpart on one GPU.
"""

from __future__ import annotations

import ctypes
import logging
import threading
from typing import Sequence

import torch
from torch import Tensor

from odc_amd import _native
from odc_amd.primitives.utils import (
    BufferSplitter,
    SymmBufferRegistry,
    _launch_streams,
    comm_stream_section,
    get_world,
    group_size,
    native_dtype,
    note_launch,
    plain_launch_stream,
    stream_from_handle,
)

logger = logging.getLogger(__name__)

_host_path = _native.load_torch_binding()


class GatherService:
    def __init__(self):
        self.buffer_splitter = BufferSplitter()
        self._lock = threading.Lock()
        self._conversion = None  # (stream handle, event) of the latest convert_symm_buffer
        self._met_conversion = frozenset()  # streams ordered after it (replaced, never mutated)

    def gather_into_tensor(self, output_tensor: Tensor, input_tensor: Tensor, pg) -> None:
        """``output_tensor.view(W, -1)[r] = rank r's copy of input_tensor`` for every r.

        ``input_tensor`` is the calling rank's shard and must live in a registered symmetric
        buffer; ``pg`` is a process group or ``VirtualGroup`` of the arena's W ranks.
        """
        self.gather_into_tensors([output_tensor], [input_tensor], pg)

    def gather_into_tensors(
        self, output_tensors: Sequence[Tensor], input_tensors: Sequence[Tensor], pg
    ) -> None:
        """Multi-tensor form: every (output, input) pair of the lists in ONE launch (per 112
        pairs). Equivalent to calling ``gather_into_tensor`` pair by pair. When the outputs'
        dtype differs from the shards' (bf16/fp16/fp32 only) the conversion is fused in."""
        assert len(output_tensors) == len(input_tensors)
        world = get_world()  # raises when there is no arena (no GPU, or init_nvshmem not called)
        if not len(input_tensors):
            return
        self._launch(_host_path.gather, world, pg, output_tensors, input_tensors)

    def _launch(self, entry, world, pg, *call) -> None:
        """``entry`` (odc_torch.cpp) checks its tensors, fills the item array and launches."""
        W = world.world_size
        assert pg is world.group or group_size(pg) == W, f"group size {group_size(pg)} != arena world size {W}"
        stream = plain_launch_stream(world)
        if stream is not None:
            if self._conversion is not None:
                self._order_after_conversion(stream)
            status = entry(world.arena.raw_handle, W, world.rank, stream, *call)
            if stream not in _launch_streams:
                note_launch(stream)
        else:
            with comm_stream_section("odc.gather") as comm:
                if self._conversion is not None:
                    self._order_after_conversion(comm.cuda_stream)
                status = entry(world.arena.raw_handle, W, world.rank, comm.cuda_stream, *call)
        if status:
            _native.check(status)

    def gather_slices(
        self,
        output_tensors: Sequence[Tensor],
        input_tensor: Tensor,
        slice_offsets: Sequence[int],
        slice_numels: Sequence[int],
        pg,
    ) -> None:
        """Gather slices of ONE symmetric buffer straight into separate outputs, in one launch:
        ``output_i.view(W, -1)[r] = rank r's input_tensor[off_i : off_i + n_i]``.

        With the FSDP2 group layout (``odc/fsdp/fsdp2.py:146-196``: the group buffer is the
        concatenation of every parameter's padded shard) this is ``gather_into_tensor`` followed
        by ``split_with_sizes_copy(dim=1)`` (``fsdp2.py:378-401``) without the intermediate
        ``[W, sum n_i]`` buffer.
        """
        assert len(output_tensors) == len(slice_offsets) == len(slice_numels)
        assert input_tensor.is_cuda and input_tensor.is_contiguous()
        if not len(output_tensors):
            return
        self._launch(_host_path.gather_slices, get_world(), pg, output_tensors, input_tensor, slice_offsets,
                     slice_numels)

    def convert_symm_buffer(self, dst_key, src_key, ranks: Sequence[int] = None) -> None:
        """Rank r's symmetric buffer ``dst_key`` = rank r's ``src_key`` converted to the
        destination's dtype (round to nearest even), for every rank whose memory this process
        holds, in ONE launch over all W regions (``odc_convert``); ``ranks`` narrows it to some
        ranks, one launch each (with one process per GPU a rank converts its own shard). On the
        launch stream of the other primitives; a gather issued later on another stream first
        waits for the conversion.

        It is what keeps a copy of the sharded parameters in the compute dtype: converted once
        after the optimizer step (4 + 2 bytes per element of ONE shard), so that every gather of
        the minibatch moves 2 + 2 bytes per element instead of converting on the way (4 + 2),
        the FSDP2 counterpart of the copy-once-until-flush of ``odc/primitives/utils.py:103-116``
        that ``odc/fsdp/fsdp1.py:239-247`` uses for the low-precision shard."""
        registry = SymmBufferRegistry.get_instance()
        world = get_world()
        src_offset, src_shape, src_dtype = registry.offsets[src_key]
        dst_offset, dst_shape, dst_dtype = registry.offsets[dst_key]
        assert tuple(src_shape) == tuple(dst_shape), f"{src_key}: {src_shape} != {dst_key}: {dst_shape}"
        numel = 1
        for d in src_shape:
            numel *= d
        if not numel:
            return
        lib = _native.load()
        with comm_stream_section("odc.convert") as comm:
            stream = ctypes.c_void_p(comm.cuda_stream)
            if ranks is None:
                item = (_native.ConvertItem * 1)()
                item[0].src_offset, item[0].dst_offset, item[0].elems = src_offset, dst_offset, numel
                _native.check(
                    lib.odc_convert(world.arena.handle, item, 1, native_dtype(src_dtype), native_dtype(dst_dtype), stream)
                )
            else:
                item = (_native.PublishItem * 1)()
                item[0].acc_offset = src_offset
                item[0].elems = numel
                peers = registry.peer_tensors[dst_key]
                for r in ranks:
                    item[0].out = peers[r].data_ptr()
                    _native.check(
                        lib.odc_publish(
                            world.arena.handle, r, item, 1, native_dtype(src_dtype), native_dtype(dst_dtype), 1.0, stream
                        )
                    )
            self._note_conversion(comm.cuda_stream)

    def _note_conversion(self, stream_handle: int) -> None:
        """A conversion was just launched on ``stream_handle``: gathers on other streams must
        not read its output before it is written. Conversions are rare (one per group and
        minibatch), so the event is recorded here, eagerly; a gather only looks at it when its
        own stream has not met this conversion yet."""
        if torch.cuda.is_current_stream_capturing():
            return  # inside a graph the capture's own stream order is all there is
        event = torch.cuda.Event()
        event.record(stream_from_handle(stream_handle))
        with self._lock:
            self._conversion = (stream_handle, event)
            self._met_conversion = {stream_handle}

    def _order_after_conversion(self, stream_handle: int) -> None:
        """Before a gather on ``stream_handle``: wait for the latest conversion if it ran on
        another stream and this stream has not waited for it yet."""
        if stream_handle in self._met_conversion:
            return
        with self._lock:
            if self._conversion is None or stream_handle in self._met_conversion:
                return
            if not torch.cuda.is_current_stream_capturing():
                stream_from_handle(stream_handle).wait_event(self._conversion[1])
                self._met_conversion = self._met_conversion | {stream_handle}
