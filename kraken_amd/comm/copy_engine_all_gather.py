"""Chunked all-gather with arrival flags (``kraken/comm/copy_engine_all_gather.py``)."""
from __future__ import annotations

import ctypes

import torch

from .. import _lib
from ._common import PeerBuffers, has_tangent

# Up to here all copies and flags of a gather on a side stream are one launch.  What that gives depends on how long the product
# beside it takes next to the launches of the loop (about 120 us of host time and 9 per chunk).  Time in one launch over time
# with a copy and a flag per chunk, 2, 4 and 8 ranks, 4 to 47 MiB, K = 1024 to 8192, N = 1024 to 28672, one and two chunks a rank:
# a call that is waited for 0.39 to 1.00 at all 216 shapes (W = 8, 1024 x 1024, N = 1024 0.59; N = 28672 0.87); calls one
# behind the other 0.38 to 0.9 where the launches are the longer part, 0.94 to 1.03 where the product is, up to 1.07 with two
# or four ranks and N = 7168 (2 x 1024 x 8192 200 -> 215 us, alone 284 -> 260).  Above, copies that come one behind the other leave
# the product more of the memory (8 x 1024 x 8192, N = 3584 405 / 438 us; the same kernel once per chunk 424).
# (all_gather_matmul takes this way only for copies that the caller wants on the copy engines, or that one launch cannot take.)
ONE_LAUNCH_BYTES = 48 << 20

_backend_streams: dict[int, torch.cuda.Stream] = {}


def _get_backend_stream(dev: torch.device) -> torch.cuda.Stream:
    """One side stream per device for the copies (default priority)."""
    idx = dev.index if dev.index is not None else torch.cuda.current_device()
    if idx not in _backend_streams:
        _backend_streams[idx] = torch.cuda.Stream(device=dev)
    return _backend_streams[idx]


def _check_progress(progress: torch.Tensor, n: int) -> None:
    assert progress.dtype in (torch.int32, torch.uint32), "progress must be a 32-bit integer tensor"
    assert progress.is_contiguous() and progress.numel() >= n


def followed(output: torch.Tensor, peers: PeerBuffers) -> bool:
    """Whether autograd has to know of the gather: copies by torch tell it, a kernel or a copy engine does not."""
    return ((torch.is_grad_enabled() and (output.requires_grad or any(t.requires_grad for t in peers.tensors)))
            or has_tangent(output, *peers.tensors))


def _takes_copies(output: torch.Tensor) -> bool:
    """Whether torch copies into ``output`` (with gradients enabled, not into a leaf that requires one, nor a view of it)."""
    base = output._base if output._is_view() else output
    return not (torch.is_grad_enabled() and base.is_leaf and base.requires_grad)


def in_own_place(sources: list[int], output: torch.Tensor) -> list[bool]:
    """For each shard's address whether it overlaps the gathered matrix nowhere but in its own place."""
    W = len(sources)
    out, size = output.data_ptr(), output.numel() * output.element_size() // W
    return [p + size <= out or p >= out + W * size or p == out + r * size for r, p in enumerate(sources)]


def gather_chunks(output: torch.Tensor, peers: PeerBuffers, progress: torch.Tensor, splits: int, rank: int, stream: int) -> bool:
    """All chunks and flags in one launch (``kr_gather_chunks``) on the stream given; False, and nothing launched, where
    addresses or chunks are no multiples of 16 bytes, or a shard lies where another one's copy goes (its workgroups
    run in no order).  Of the arguments' checks only these are made here."""
    W = peers.W
    chunk_bytes = peers.cap // splits * output.element_size()
    sources = peers.pointers()
    if (W > _lib.KR_MAX_WORLD or chunk_bytes % 16 != 0 or output.data_ptr() % 16 != 0 or any(p % 16 != 0 for p in sources)
            or not all(in_own_place(sources, output))):
        return False
    rc = _lib.load().kr_gather_chunks((ctypes.c_void_p * W)(*sources), W, splits, rank, chunk_bytes, output.data_ptr(),
                                      progress.data_ptr(), stream)
    _lib.check(rc, "gather_chunks")
    torch.autograd.graph.increment_version(output)
    return True


def _copy_engine_all_gather_w_progress(
    output: torch.Tensor,
    inp,
    progress: torch.Tensor,
    splits_per_rank: int,
    backend_stream: torch.cuda.Stream | None = None,
    *,
    rank: int = 0,
    copy_engine: bool = False,
) -> torch.cuda.Stream:
    """Copy the W shards into ``output`` chunk by chunk on a side stream, flagging each chunk.

    Counterpart of ``_copy_engine_all_gather_w_progress``
    (``kraken/comm/copy_engine_all_gather.py:6-60``).  ``inp`` holds the W
    ranks' shards — the ``[W, m, ...]`` stack or a list of W tensors, standing
    in for the peers' symmetric buffers (``:41-43``).  On the side stream, in
    the reference's order (source ranks ``rank+1, rank+2, ..., rank``, ``:38-39``),
    every one of the ``W * splits_per_rank`` chunks is copied into its place in
    ``output`` and then ``progress[chunk]`` is set to 1 by a stream-ordered
    flag write (``:47-53``).  The side stream first waits for the current
    stream (``:35``); the caller makes the current stream wait for the returned
    stream when it needs the gathered tensor (``:118``).  All chunks and flags
    of a gather of up to ``ONE_LAUNCH_BYTES`` are one launch (``kr_gather_chunks``); larger ones,
    chunks that are no multiple of 16 bytes, shards that lie in another one's place of ``output`` (they are
    set aside first) and shards that autograd follows (they require a gradient, or carry a forward-mode tangent)
    are copied one by one by ordinary device-to-device copies, which autograd records,
    with a flag write behind each; ``copy_engine=True`` hands them to the GPU's
    copy engines (``kr_copy_engine_memcpy``), which take no compute units but
    are slower within one GPU and, like the one launch, only mark ``output`` as written.  ``progress``
    must have been zeroed on the current stream beforehand.
    """
    peers = PeerBuffers(inp, dtypes=(torch.bfloat16, torch.float8_e4m3fn))
    W = peers.W
    assert 0 <= rank < W
    assert peers.cap % splits_per_rank == 0
    n_chunks = W * splits_per_rank
    _check_progress(progress, n_chunks)
    out_shape = list(peers.shape)
    out_shape[0] *= W
    assert list(output.shape) == out_shape, (list(output.shape), out_shape)
    assert output.is_contiguous() and output.dtype == peers.tensors[0].dtype
    dev = _lib.require_device(*peers.tensors, output, progress)
    if backend_stream is None:
        backend_stream = _get_backend_stream(dev)
    lib = _lib.load()
    chunk = peers.cap // splits_per_rank
    current = torch.cuda.current_stream(dev)
    if backend_stream != current:
        backend_stream.wait_stream(current)
    recorded = not copy_engine and followed(output, peers)
    if (not copy_engine and output.numel() * output.element_size() <= ONE_LAUNCH_BYTES and not (recorded and _takes_copies(output))
            and gather_chunks(output, peers, progress, splits_per_rank, rank, backend_stream.cuda_stream)):
        return backend_stream
    if (recorded and torch.is_grad_enabled() and output.grad_fn is not None and not output._is_view()
            and all(t.untyped_storage().data_ptr() != output.untyped_storage().data_ptr() for t in peers.tensors)):
        output.detach_()     # every element is written below: a matrix that is kept does not keep the history of earlier gathers
    flat_out = output.view(-1)
    with torch.cuda.stream(backend_stream):
        shards = [peers.slice(r) if kept else peers.slice(r).clone() for r, kept in enumerate(in_own_place(peers.pointers(), output))]
        for step in range(W):
            src_rank = (rank + step + 1) % W
            src = shards[src_rank].reshape(-1)
            for split_id in range(splits_per_rank):
                c = src_rank * splits_per_rank + split_id
                dst_c, src_c = flat_out[c * chunk:(c + 1) * chunk], src[split_id * chunk:(split_id + 1) * chunk]
                if copy_engine:
                    _lib.copy_engine_copy(dst_c, src_c, backend_stream.cuda_stream)
                else:
                    dst_c.copy_(src_c)
                rc = lib.kr_stream_write_value32(progress.data_ptr() + 4 * c, 1, backend_stream.cuda_stream)
                _lib.check(rc, "stream_write_value32")
    if copy_engine:
        torch.autograd.graph.increment_version(output)
    return backend_stream


def all_gather_w_progress(a_shared, a_out: torch.Tensor | None = None, progress: torch.Tensor | None = None,
                          **kwargs) -> torch.Tensor:
    """All-gather of the W shards into one tensor, chunk flags in ``progress``.

    Counterpart of ``all_gather_w_progress``
    (``kraken/comm/copy_engine_all_gather.py:63-120``): allocates ``a_out`` and
    ``progress`` when not given, zeroes ``progress`` (``:108``), runs the chunked
    copy.  The current stream would wait for a side stream at once, so the copies run on it
    (``copy_engine=True``: on the side stream).  kwargs:
    ``splits_per_rank`` (default 1), ``rank`` (default 0), ``copy_engine`` (default False).
    """
    peers = PeerBuffers(a_shared)
    splits = kwargs.get("splits_per_rank", 1)
    rank = kwargs.get("rank", 0)
    dev = _lib.require_device(*peers.tensors)
    shape = list(peers.shape)
    shape[0] *= peers.W
    if a_out is None:
        a_out = torch.empty(shape, dtype=torch.bfloat16, device=dev)
    if progress is None:
        progress = torch.zeros(peers.W * splits, dtype=torch.int32, device=dev)
    else:
        progress.fill_(0)
    copy_engine, current = kwargs.get("copy_engine", False), torch.cuda.current_stream(dev)
    stream = _copy_engine_all_gather_w_progress(a_out, a_shared, progress, splits, None if copy_engine else current, rank=rank,
                                                copy_engine=copy_engine)
    if stream != current:
        current.wait_stream(stream)
    return a_out
