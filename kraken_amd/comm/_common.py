"""Shared argument handling of the W-way reduce wrappers."""
from __future__ import annotations

import ctypes
from typing import Sequence

import torch
from torch.autograd import forward_ad

from .. import _lib, _waits


class PeerBuffers:
    """The W buffers a reduce reads: one per rank, all on this GPU (``shape``: of one of them).

    Stands in for the peers' symmetric-memory buffers of the reference
    (``symm_mem_hdl.buffer_ptrs_dev``, ``kraken/comm/one_shot_all_reduce.py:96-99``).
    Two forms are accepted wherever the reference takes its symmetric buffer:

    * one ``[W, ...]`` tensor whose slices are the W buffers (slices must be
      contiguous, the stride between them is free) — goes to the stacked entry
      points of the library;
    * a list or tuple of W separately allocated tensors of one shape — goes to
      the pointer-table entry points (``kr_*_ptrs_bf16``), which is also how W
      real peer mappings would be handed over.

    Both forms give bit-identical results: the kernels are the same.
    """

    def __init__(self, buffers: torch.Tensor | Sequence[torch.Tensor], dtypes=(torch.bfloat16,)):
        if isinstance(buffers, torch.Tensor):
            assert buffers.dim() >= 2, "expected a stacked tensor of shape [W, ...]"
            assert buffers.dtype in dtypes, "Only bfloat16 is supported for now."
            self.W = buffers.shape[0]
            assert self.W >= 1
            assert buffers.is_contiguous() or buffers[0].is_contiguous(), "each of the W slices must be contiguous"
            self.cap = buffers.numel() // self.W
            self.stride = buffers.stride(0) if self.W > 1 else self.cap
            self.stacked = buffers
            self.tensors = [buffers]
            self.shape = buffers.shape[1:]
        else:
            bufs = list(buffers)
            assert len(bufs) >= 1, "expected W >= 1 buffers"
            assert isinstance(bufs[0], torch.Tensor), "expected a tensor or a sequence of tensors"
            dtype, shape = bufs[0].dtype, bufs[0].shape
            assert dtype in dtypes, "Only bfloat16 is supported for now."
            for t in bufs:
                assert isinstance(t, torch.Tensor), "expected a tensor or a sequence of tensors"
                assert t.dtype == dtype, "Only bfloat16 is supported for now."
                assert t.is_contiguous(), "each of the W buffers must be contiguous"
                assert t.shape == shape, "the W buffers must have one shape"
            self.W = len(bufs)
            self.cap = bufs[0].numel()
            self.stride = None
            self.stacked = None
            self.tensors = bufs
            self.shape = bufs[0].shape

    def slice(self, rank: int) -> torch.Tensor:
        """Buffer of rank ``rank``."""
        return self.stacked[rank] if self.stacked is not None else self.tensors[rank]

    def pointers(self) -> list[int]:
        """Device address of every rank's buffer."""
        if self.stacked is None:
            return [t.data_ptr() for t in self.tensors]
        base, step = self.stacked.data_ptr(), self.stride * self.stacked.element_size()
        return [base + r * step for r in range(self.W)]

    def _table(self, elem_off: int):
        # host array of W device pointers, each moved on by elem_off bf16 elements
        return (ctypes.c_void_p * self.W)(*[p + 2 * elem_off for p in self.pointers()])

    def reduce(self, elem_off, numel, bias_ptr, bias_numel, D, bias_first, out_ptr, stream) -> int:
        """``kr_reduce_bf16`` / ``kr_reduce_ptrs_bf16`` on elements [elem_off, elem_off + numel)."""
        lib = _lib.load()
        if self.stacked is not None:
            return lib.kr_reduce_bf16(self.stacked.data_ptr() + 2 * elem_off, self.W, self.stride, numel,
                                      bias_ptr, bias_numel, D, bias_first, out_ptr, stream)
        return lib.kr_reduce_ptrs_bf16(self._table(elem_off), self.W, numel, bias_ptr, bias_numel, D,
                                       bias_first, out_ptr, stream)

    def reduce_striped(self, numel, bias_ptr, block, rank, out_ptr, stream) -> int:
        lib = _lib.load()
        if self.stacked is not None:
            return lib.kr_reduce_striped_bf16(self.stacked.data_ptr(), self.W, self.stride, numel, bias_ptr,
                                              block, rank, out_ptr, stream)
        return lib.kr_reduce_striped_ptrs_bf16(self._table(0), self.W, numel, bias_ptr, block, rank, out_ptr,
                                               stream)

    def reduce_rmsnorm(self, rows, D, bias_ptr, bias_is_vector, w_ptr, eps, y_ptr, stream) -> int:
        lib = _lib.load()
        dev = self.tensors[0].device
        ws = row_workspace(dev, lib.kr_rmsnorm_workspace_bytes(self.W, rows, D), stream)
        ws_ptr, ws_bytes = (ws.data_ptr(), ws.numel()) if ws is not None else (None, 0)
        # a few long rows: their wavefronts meet in the workspace, a bounded wait that reports through
        # the stream's status word like the flag waits of the overlap paths
        status = _waits.new_status(dev, stream) if ws is not None else None
        if self.stacked is not None:
            rc = lib.kr_reduce_rmsnorm_ws_bf16(self.stacked.data_ptr(), self.W, self.stride, rows, D, bias_ptr,
                                               bias_is_vector, w_ptr, eps, y_ptr, ws_ptr, ws_bytes, _lib.ptr(status),
                                               stream)
        else:
            rc = lib.kr_reduce_rmsnorm_ptrs_ws_bf16(self._table(0), self.W, rows, D, bias_ptr, bias_is_vector,
                                                    w_ptr, eps, y_ptr, ws_ptr, ws_bytes, _lib.ptr(status), stream)
        if status is not None and rc == 0:
            row_watch(status)
        return rc


_row_workspaces: dict[tuple[int, int], tuple[torch.Tensor, torch.cuda.Stream]] = {}


def row_workspace(dev: torch.device, nbytes: int, stream_handle: int) -> torch.Tensor | None:
    """Workspace of the split-row RMSNorm kernel: one zero-initialised buffer per (device, stream
    that is current at the call, ``stream_handle``), so that eager calls on different streams never share one; the
    kernels keep it consistent afterwards.  A call that is captured into a graph bakes in the
    workspace of the capture stream, whatever stream the graph is later replayed on: replays of
    that graph must not overlap each other, other graphs captured on the same stream, or eager
    calls on the capture stream (calls that share a workspace and overlap give NaN rows or wrong
    ones).  After a reported time-out of the rows' exchange every workspace is zeroed again."""
    if nbytes <= 0:
        return None
    key = (dev.index if dev.index is not None else torch.cuda.current_device(), stream_handle)
    entry = _row_workspaces.get(key)
    if entry is None or entry[0].numel() < nbytes:
        entry = (torch.zeros(nbytes, dtype=torch.uint8, device=dev), torch.cuda.current_stream(dev))
        _row_workspaces[key] = entry
    return entry[0]


def row_exchange(index: int, nbytes: int, stream_handle: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Workspace and status word of the split-row kernel for a device index and stream."""
    dev = torch.device("cuda", index)
    return row_workspace(dev, nbytes, stream_handle), _waits.new_status(dev, stream_handle)


def row_watch(status: torch.Tensor) -> None:
    # (the word is sticky and these calls take microseconds: mirroring it to the host now and
    # then is enough to report a time-out, every call would cost more than the kernel)
    _waits.watch(status, "reduce + RMSNorm of a few long rows (rows spread over many compute units)", min_interval_s=0.05)


def _zero_row_workspaces() -> None:
    # after a time-out the slots of a workspace may carry tags that a later call would take for fresh ones
    for ws, stream in _row_workspaces.values():
        with torch.cuda.stream(stream):
            ws.zero_()


_waits.on_failure(_zero_row_workspaces)


def has_tangent(*tensors: torch.Tensor) -> bool:
    """Whether a tensor carries a forward-mode tangent: only copies by torch hand it on, or clear it."""
    return forward_ad._current_level >= 0 and any(forward_ad.unpack_dual(t).tangent is not None for t in tensors)


def check_stack(stacked: torch.Tensor | Sequence[torch.Tensor]) -> PeerBuffers:
    """Validate the W buffers (stacked tensor or sequence of tensors).

    Mirrors the dtype/alignment asserts of ``kraken/comm/one_shot_all_reduce.py:79-80``.
    """
    return PeerBuffers(stacked)


def stage_input(peers: PeerBuffers, input_tensor: torch.Tensor | None, rank: int, stage: bool = False) -> PeerBuffers:
    """Make ``input_tensor`` the source of rank ``rank`` and return the buffers to reduce.

    The reference kernels first copy the input into this rank's symmetric buffer, where the
    peers read it (``kraken/fused/one_shot_all_reduce_bias.py:56-65``,
    ``one_shot_all_reduce_bias_rms_norm.py:57-61``).  On one GPU nobody else reads that buffer, so
    by default the input is read in place: the returned buffers are the W sources as a pointer
    table whose entry ``rank`` is the input itself -- no copy, no extra launch, the same bits.
    ``stage=True`` keeps the side effect for callers who want the buffer to hold the input
    afterwards: one device copy into the buffer in front of the kernel.  An input that is not
    contiguous or not 16-byte aligned is always copied.
    """
    if input_tensor is None:
        return peers
    pointers = peers.pointers()
    address = input_tensor.data_ptr()
    if pointers[rank] == address:
        return peers
    if stage or not input_tensor.is_contiguous() or address % 16 != 0:
        peers.slice(rank).reshape(-1)[:input_tensor.numel()].copy_(input_tensor.reshape(-1))
        return peers
    pointers[rank] = address
    return _Sources(peers, pointers)


class _Sources(PeerBuffers):
    """The buffers of ``peers`` with some of their addresses replaced (by sources at least as long as the message).

    Addresses only: a view of every slice costs the host more than the kernel takes (W = 8, 512 x 5120 with an
    input of its own: 30.7 us a call with views, 12.4 with addresses)."""

    def __init__(self, peers: PeerBuffers, pointers: list[int]):
        self.W = peers.W
        self.cap = peers.cap
        self.stride = None
        self.stacked = None
        self.tensors = peers.tensors
        self.shape = peers.shape
        self._pointers = pointers

    def pointers(self) -> list[int]:
        return list(self._pointers)

    def slice(self, rank: int) -> torch.Tensor:
        raise NotImplementedError("the sources of a reduce are known by address only")


def bias_args(bias: torch.Tensor | None, numel: int, D: int) -> tuple[int | None, int]:
    """Return (pointer, bias_numel) for a bias of the input's shape or of shape [D]."""
    if bias is None:
        return None, 0
    assert bias.dtype == torch.bfloat16, "Only bfloat16 is supported for now."
    assert bias.is_contiguous()
    assert bias.numel() in (numel, D), (
        f"bias must have the shape of the input ({numel} elements) or be a vector of the last dim ({D})"
    )
    return _lib.ptr(bias), bias.numel()
