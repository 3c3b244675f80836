"""GEMM + copy-engine reduce-scatter, local arithmetic (``kraken/fused/gemm_reduce_scatter_ce_persistent.py``)."""
from __future__ import annotations

import ctypes

import torch
from torch.autograd import forward_ad

from .. import _lib, _waits
from ..comm._common import has_tangent
from ..comm.copy_engine_all_gather import _get_backend_stream
from . import _gemm


def reduce(inp: torch.Tensor, output: torch.Tensor, configs: dict) -> torch.Tensor:
    """Rotated-order W-way band reduce of ``inp [M, N]`` into ``output [M/W, N]``.

    Counterpart of ``reduce`` / ``_reduce_persistent_kernel``
    (``kraken/fused/gemm_reduce_scatter_ce_persistent.py:245-321``):
    ``output = sum_i inp[band (i + RANK + 1) % W]``, accumulated in the input
    dtype (bf16 rounding after every add) unless ``configs["fp32_acc"]``.
    """
    M, N = inp.shape
    W, rank = configs["WORLD_SIZE"], configs["RANK"]
    m_per_rank = M // W
    assert output.shape[0] == m_per_rank and M % W == 0
    assert inp.dtype == torch.bfloat16 and output.dtype == torch.bfloat16
    assert inp.is_contiguous() and output.is_contiguous()
    dev = _lib.require_device(inp, output)
    rc = _lib.load().kr_reduce_rotated_bf16(
        inp.data_ptr(), W, m_per_rank, N, rank, int(not configs.get("fp32_acc", False)),
        output.data_ptr(), _lib.current_stream(dev),
    )
    _lib.check(rc, "gemm_reduce_scatter_ce_persistent.reduce")
    return output


def gemm_producer_w_progress(
    a: torch.Tensor,
    b: torch.Tensor,
    gemm_out: torch.Tensor,
    progress: torch.Tensor,
    signal_pad: torch.Tensor,
    configs: dict,
    group=None,
) -> None:
    """``gemm_out = a @ b`` with one completion flag per destination rank's band.

    Counterpart of ``gemm_producer_w_progress`` / ``_gemm_producer_persistent_kernel``
    (``kraken/fused/gemm_reduce_scatter_ce_persistent.py:46-134,178-242``): the M
    tiles are processed starting at the band of ``RANK + 1`` (``:88,102``); every
    finished tile is counted into ``progress[r]`` of the bands it touches and the
    tile that completes band ``r`` sets ``signal_pad[r] = 1`` (``:117-132``).  Both
    are 32-bit integer tensors of ``WORLD_SIZE`` elements, zeroed by the caller
    (``:364-365``).  Shapes whose output tiles all run at once (one round of the
    compute units or less) finish all bands together, so for those the library's
    fastest GEMM is used when it is a split one (K loop shared between workgroups):
    their flags are set by a stream-ordered fill behind the GEMM and ``progress``
    is not counted.  Every larger shape runs the producer kernel, whose bands
    finish, and are flagged, one after the other.
    """
    a2, b2 = _gemm.prepare_operands(a, b)
    M, N = a2.shape[0], b2.shape[1]
    W, rank = configs["WORLD_SIZE"], configs["RANK"]
    assert M % W == 0 and 0 <= rank < W
    assert gemm_out.shape == (M, N) and gemm_out.dtype == torch.bfloat16 and gemm_out.is_contiguous()
    for t in (progress, signal_pad):
        assert t.dtype in (torch.int32, torch.uint32) and t.is_contiguous() and t.numel() >= W
    dev = _lib.require_device(a2, b2, gemm_out, progress, signal_pad)
    lib = _lib.load()
    pivot = ((rank + 1) % W) * (M // W)
    if _one_round(dev, M, N) and lib.kr_gemm_workspace_bytes(M, N, a2.shape[1]) > 0:
        _gemm.launch("gemm_producer_w_progress", a2, b2, M, N, None, 0, 0, None, 0, 0, gemm_out, None, pivot)
        signal_pad.fill_(1)
        return
    rc = lib.kr_gemm_producer_bf16(
        a2.data_ptr(), a2.stride(0), a2.stride(1), b2.data_ptr(), b2.stride(0), b2.stride(1),
        M, N, a2.shape[1], gemm_out.data_ptr(), W, rank, progress.data_ptr(), signal_pad.data_ptr(),
        _lib.current_stream(dev),
    )
    _lib.check(rc, "gemm_producer_w_progress")


def _one_round(dev: torch.device, M: int, N: int) -> bool:
    """Whether all output tiles run at once, so that all bands finish together."""
    return -(-M // 256) * -(-N // 256) <= torch.cuda.get_device_properties(dev).multi_processor_count


def _byte_range(t: torch.Tensor) -> tuple[int, int]:
    """First and past-the-last byte a tensor's elements lie in."""
    if t.is_contiguous():
        return t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()
    last = sum((n - 1) * s for n, s in zip(t.shape, t.stride()))
    return t.data_ptr(), t.data_ptr() + (last + 1) * t.element_size()


def _readable_in_place(bands: list[torch.Tensor], written: list[torch.Tensor]) -> bool:
    """Whether the reduce may read the bands where they are while ``written`` is being written."""
    if any(t.data_ptr() % 16 != 0 or t.device != bands[0].device for t in bands):
        return False
    reads = [_byte_range(t) for t in bands]
    return all(hi <= r_lo or r_hi <= lo for lo, hi in map(_byte_range, written) for r_lo, r_hi in reads)


def _sends_direct(sent, a: torch.Tensor, b: torch.Tensor, world_size: int, m_per_rank: int, N: int) -> bool:
    """Whether the GEMM may store the other ranks' bands in ``sent`` itself: one matrix of contiguous bands, apart from
    the operands, and nothing autograd would have to know of."""
    if not (isinstance(sent, torch.Tensor) and tuple(sent.shape) == (world_size, m_per_rank, N) and sent.is_contiguous()
            and sent.dtype == a.dtype and sent.device == a.device and sent.data_ptr() % 16 == 0
            and not sent.requires_grad and not has_tangent(sent)):
        return False
    lo, hi = _byte_range(sent)
    return all(hi <= t_lo or t_hi <= lo for t_lo, t_hi in (_byte_range(a), _byte_range(b)))


def _stacked_peers_apart(peers, sent: torch.Tensor, rows: int, N: int) -> list[int] | None:
    """Addresses of the peers' bands where they come as one tensor that the reduce may read in place whatever is
    written to ``sent``; ``None`` where that needs a closer look (a view per band costs the host more than the launch)."""
    if not isinstance(peers, torch.Tensor) or peers.device != sent.device:
        return None
    base, step, P = peers.data_ptr(), 2 * peers.stride(0), peers.shape[0]
    end, (lo, hi) = base + (P - 1) * step + 2 * rows * N, _byte_range(sent)
    if base % 16 != 0 or step % 16 != 0 or (base < hi and lo < end):
        return None
    return [base + r * step for r in range(P)]


def _reduce_sources(sources: list[int], rows: int, N: int, output: torch.Tensor, configs: dict) -> torch.Tensor:
    """``reduce`` of W bands given by their addresses, all on the device of ``output``."""
    rc = _lib.load().kr_reduce_rotated_ptrs_bf16(
        (ctypes.c_void_p * len(sources))(*sources), len(sources), rows, N, configs["RANK"],
        int(not configs["fp32_acc"]), output.data_ptr(), _lib.current_stream(output.device),
    )
    _lib.check(rc, "gemm_reduce_scatter_ce_persistent")
    return output


def _reduce_bands(bands: list[torch.Tensor], rows: int, N: int, output: torch.Tensor, configs: dict) -> torch.Tensor:
    """``reduce`` of W bands in buffers of their own."""
    _lib.require_device(output, *bands)
    return _reduce_sources([t.data_ptr() for t in bands], rows, N, output, configs)


def copy_engine_scatter(
    inp: torch.Tensor,
    output,
    signal_pad: torch.Tensor,
    group=None,
    *,
    rank: int = 0,
    wait_limit_us: int = 0,
    status: torch.Tensor | None = None,
    copy_engine: bool = False,
) -> None:
    """Copy every finished band of ``inp [M, N]`` to its destination, on the current stream.

    Counterpart of ``copy_engine_scatter``
    (``kraken/fused/gemm_reduce_scatter_ce_persistent.py:137-175``): for
    ``step = 0..W-1`` the band of ``remote = (rank + step + 1) % W`` is copied once
    ``signal_pad[remote] == 1`` — a stream-ordered wait in front of each copy
    (``:153-163``), so the copies start while the producer GEMM is still running on
    another stream.  ``output`` holds the W destinations: a ``[W, M/W, N]`` tensor or
    a sequence of W tensors ``[M/W, N]`` (``None`` entries are skipped: no wait, no
    copy); ``output[r]`` stands for slot ``rank`` of rank r's symmetric buffer
    (``:165-169``).  The waits are bounded (``wait_limit_us``, default 5 s); a wait
    that runs out sets ``status`` (int32 ``[1]``, zeroed by the caller) to 1 and the bands copied
    behind it are invalid; without ``status`` the wrapper keeps a word of its own and the next call
    of an overlap function (or ``kraken_amd._waits.check()``) raises once the copies have run.  The
    copies are ordinary copy kernels; ``copy_engine=True`` hands them to the GPU's
    copy engines (``kr_copy_engine_memcpy``).
    """
    M, N = inp.shape
    W = len(output)
    assert M % W == 0 and 0 <= rank < W
    m_per_rank = M // W
    assert signal_pad.dtype in (torch.int32, torch.uint32) and signal_pad.is_contiguous() and signal_pad.numel() >= W
    dev = _lib.require_device(inp, signal_pad, status, *[t for t in output if t is not None])
    lib = _lib.load()
    stream = _lib.current_stream(dev)
    _waits.check()
    own_status = status is None
    if own_status:
        status = _waits.new_status(dev)     # shared by the W waits: after one runs out the others give up at once
    for step in range(W):
        remote = (rank + step + 1) % W
        dst = output[remote]
        if dst is None:
            continue
        assert tuple(dst.shape) == (m_per_rank, N) and dst.dtype == inp.dtype
        rc = lib.kr_stream_wait_value32(signal_pad.data_ptr() + 4 * remote, 1, wait_limit_us, _lib.ptr(status), stream)
        _lib.check(rc, "stream_wait_value32")
        band = inp[remote * m_per_rank:(remote + 1) * m_per_rank]
        if copy_engine and dst.is_contiguous() and band.is_contiguous():
            _lib.copy_engine_copy(dst, band, stream)
        else:
            dst.copy_(band)
    if own_status:
        _waits.watch(status, "copy_engine_scatter")


def _common_form(a, b, reduce_op, peers=None, rank=0, sent=None, fp32_acc=False, **kwargs):
    """The call in native code where its arguments are of the common form: all peers in one tensor, the destinations in another,
    nothing else named, and no tangents about."""
    if kwargs or reduce_op != "sum" or type(fp32_acc) is not bool or forward_ad._current_level >= 0:
        return None
    return _lib.calls().reduce_scatter_sent(a, b, peers, sent, rank, not fp32_acc)


def gemm_reduce_scatter_ce_persistent(
    a: torch.Tensor,
    b: torch.Tensor,
    reduce_op: str = "sum",
    group=None,
    **kwargs,
) -> torch.Tensor:
    """Producer GEMM, band exchange on a side stream, then the rotated-order band reduce.

    Counterpart of ``kraken.fused.gemm_reduce_scatter_ce_persistent``
    (``kraken/fused/gemm_reduce_scatter_ce_persistent.py:324-375``).  The producer
    GEMM writes the full bf16 ``C = a @ b`` on the current stream and flags every
    band as it completes; with the kwarg ``sent`` (``[W, M/W, N]`` tensor or sequence) a side
    stream, which first waits for the current stream (``:345-346``), copies the flagged band of
    every other rank r to ``sent[r]`` (``:367-368``).  A contiguous ``sent`` tensor takes no copies: the GEMM
    stores the other ranks' bands there, nothing is flagged or waited for, and ``wait_limit_us`` and ``status``
    stay unused.  What the other ranks would push is in the
    pre-staged ``peers`` (kwarg, ``[W-1, M/W, N]`` or a sequence, the other ranks in ascending
    order).  The reduce (``:258-279``) sums the W bands starting at ``rank + 1`` and reads them where
    they are, the peers in their own buffers and the own band in ``C``, instead of through a
    scatter buffer they are first copied to; peers that overlap ``sent`` or are not 16-byte
    aligned are copied in front of the GEMM.  Where all bands finish together (one round of
    output tiles or less) the copies follow the GEMM on the current stream.  It otherwise
    waits for the side stream (``:370``).  kwargs ``rank`` (default 0), ``world_size``, ``fp32_acc``,
    ``wait_limit_us``, ``status``, ``copy_engine``.
    """
    out = _common_form(a, b, reduce_op, **kwargs)
    if out is not None:
        return out
    assert reduce_op == "sum", "only support sum for now"
    assert a.dtype == torch.bfloat16 and b.dtype == torch.bfloat16, "Only bfloat16 is supported for now."
    M, N = a.shape[0], b.shape[1]
    peers = kwargs.get("peers")
    world_size = kwargs.get("world_size", _gemm.n_peers_of(peers) + 1)
    rank = kwargs.get("rank", 0)
    assert M % world_size == 0
    m_per_rank = M // world_size
    P, _ = _gemm.check_peers(peers, m_per_rank, N)
    assert P == world_size - 1
    dev = _lib.require_device(a, b)
    _waits.check()      # an earlier call's failed wait is reported before anything of this call is enqueued
    output = torch.empty((m_per_rank, N), dtype=a.dtype, device=dev)
    configs = {"RANK": rank, "WORLD_SIZE": world_size, "fp32_acc": kwargs.get("fp32_acc", False)}
    if M == 0 or N == 0:
        return output
    sent = kwargs.get("sent")
    # Destinations that make up one matrix: the GEMM stores every tile where it has to go, the own band in a buffer of its
    # own (the reduce-scatter epilogue without peers), and may be any.  On one GPU the copies find compute units only as
    # the last tiles end, and bands that finish one by one cost the product its best tile order.  W = 8, all bands sent, us, copies
    # behind the bands' flags (one round of tiles: behind the GEMM) / stores of the GEMM:
    # 8192 x 4096 x 14336 735 / 658, 8192 x 8192 x 3584 (row-major B) 434 / 363, 4096 x 4096 x 4096 120 / 103,
    # 2704 x 2816 x 2304 71 / 56, 8 x 1600 x 768 73 / 58.
    direct = world_size > 1 and not kwargs.get("copy_engine", False) and _sends_direct(sent, a, b, world_size, m_per_rank, N)
    if direct:
        pivot = ((rank + 1) % world_size) * m_per_rank
        sources = _stacked_peers_apart(peers, sent, m_per_rank, N)
        if sources is None:
            bands = list(peers)
            if not _readable_in_place([a, *bands], [sent[r] for r in range(world_size) if r != rank]):
                bands = [torch.empty((m_per_rank, N), dtype=a.dtype, device=dev).copy_(t) for t in bands]
            sources = [t.data_ptr() for t in bands]
        own = _lib.calls().gemm(a, b, None, None, sent.view(M, N), rank * m_per_rank, m_per_rank, False, pivot)
        if own is None:
            own = torch.empty((m_per_rank, N), dtype=a.dtype, device=dev)
            _gemm.launch("gemm_reduce_scatter_ce_persistent", *_gemm.prepare_operands(a, b), M, N, None, 0, 0, None,
                         rank * m_per_rank, m_per_rank, sent.view(M, N), own, pivot)
        torch.autograd.graph.increment_version(sent)
        sources.insert(rank, own.data_ptr())
        return _reduce_sources(sources, m_per_rank, N, output, configs)
    dests = [None if sent is None or r == rank else sent[r] for r in range(world_size)]
    written = [t for t in dests if t is not None]
    gemm_out = torch.empty((M, N), dtype=a.dtype, device=dev)
    bands = list(peers) if peers is not None else []
    bands.insert(rank, gemm_out[rank * m_per_rank:(rank + 1) * m_per_rank])

    if not _readable_in_place(bands, written):
        scatter_out = torch.empty((world_size, m_per_rank, N), dtype=a.dtype, device=dev)
        for r, t in enumerate(bands):
            if r != rank:
                scatter_out[r].copy_(t)
                bands[r] = scatter_out[r]
    # One round of tiles or less: all bands finish together, so they leave behind the GEMM in stream order, without
    # flags, and the GEMM may be any (W = 8, 2048 x 4096 x 4096 with all bands sent: 219 us with a wait and a copy per
    # band on a side stream, 74 us with two copies).
    if _one_round(dev, M, N) and not (written and kwargs.get("copy_engine", False)):
        for t in written:
            assert tuple(t.shape) == (m_per_rank, N) and t.dtype == a.dtype
        _lib.require_device(a, *written)
        _gemm.launch("gemm_reduce_scatter_ce_persistent", *_gemm.prepare_operands(a, b), M, N, None, 0, 0, None, 0, 0,
                     gemm_out, None, ((rank + 1) % world_size) * m_per_rank)
        by_rank = gemm_out.view(world_size, m_per_rank, N)
        if (written and isinstance(sent, torch.Tensor) and sent.shape[0] == world_size
                and written[0].is_contiguous() and sent.stride(0) >= m_per_rank * N):
            for run in (slice(0, rank), slice(rank + 1, world_size)):
                if run.start < run.stop:
                    sent[run].copy_(by_rank[run])
        else:
            # (destinations may share memory, one scratch band for all: the order is that of copy_engine_scatter)
            for r in (*range(rank + 1, world_size), *range(rank)):
                if dests[r] is not None:
                    dests[r].copy_(by_rank[r])
        return _reduce_bands(bands, m_per_rank, N, output, configs)
    progress = torch.zeros(world_size, dtype=torch.int32, device=dev)
    signal_pad = torch.zeros(world_size, dtype=torch.int32, device=dev)
    current = torch.cuda.current_stream(dev)
    if written:
        backend_stream = _get_backend_stream(dev)
        backend_stream.wait_stream(current)
    gemm_producer_w_progress(a, b, gemm_out, progress, signal_pad, configs)
    if written:
        with torch.cuda.stream(backend_stream):
            copy_engine_scatter(gemm_out, dests, signal_pad, rank=rank,
                                wait_limit_us=kwargs.get("wait_limit_us", 0), status=kwargs.get("status"),
                                copy_engine=kwargs.get("copy_engine", False))
    # the own band is complete behind the GEMM in stream order: the reduce runs while the last bands leave
    _reduce_bands(bands, m_per_rank, N, output, configs)
    if written:
        current.wait_stream(backend_stream)
    return output
