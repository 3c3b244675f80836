"""All-gather + matmul, local arithmetic (``kraken/fused/all_gather_matmul.py``)."""
from __future__ import annotations

import ctypes

import torch
from torch.autograd import forward_ad

from .. import _lib, _waits
from ..comm._common import PeerBuffers, has_tangent
from ..comm.copy_engine_all_gather import _check_progress, _copy_engine_all_gather_w_progress, followed, gather_chunks, in_own_place
from . import _gemm


def _matmul_w_progress(a, a_local, b, progress, configs, status=None) -> torch.Tensor:
    """``c = a @ b`` where the rows of ``a`` arrive while the kernel runs.

    Counterpart of ``_matmul_w_progress`` (``kraken/fused/all_gather_matmul.py:147-219``):
    tiles of the local shard read ``a_local``, all others wait for
    ``progress[chunk] == 1`` (``:95-110``).  ``configs``: ``RANK``, ``WORLD_SIZE``,
    ``SPLITS_PER_RANK``, optional ``wait_limit_us``.
    """
    M, K = a.shape
    assert b.shape[0] == K
    if not b.T.is_contiguous():
        raise ValueError("b.T must be contiguous")
    N = b.shape[1]
    assert K % 8 == 0 and N % 8 == 0, "K and N must be multiples of 8"
    assert a.dtype == torch.bfloat16 and b.dtype == torch.bfloat16, "Only bfloat16 is supported for now."
    assert a.stride(1) == 1 and (a_local is None or a_local.stride(1) == 1)
    dev = _lib.require_device(a, a_local, b, progress, status)
    c = torch.empty((M, N), device=dev, dtype=a.dtype)
    rc = _lib.load().kr_all_gather_matmul_bf16(
        a.data_ptr(), a.stride(0), _lib.ptr(a_local), 0 if a_local is None else a_local.stride(0),
        b.data_ptr(), b.stride(0), b.stride(1), M, N, K,
        configs["WORLD_SIZE"], configs["RANK"], configs["SPLITS_PER_RANK"],
        _lib.ptr(progress), int(configs.get("wait_limit_us", 0)), _lib.ptr(status),
        c.data_ptr(), _lib.current_stream(dev),
    )
    _lib.check(rc, "all_gather_matmul")
    return c


def _direct(sources: list[int], a_out: torch.Tensor, b: torch.Tensor, W: int, m: int, N: int, K: int) -> bool:
    """Whether the product gathers the shards itself (``kr_gather_matmul_bf16``): enough large tiles, each inside one
    shard, and shards apart from the gathered matrix (a tile may read a row after another one has written it)."""
    return (W <= _lib.KR_MAX_WORLD and _lib.load().kr_gather_matmul_direct(W, m, N, K) == 1
            and all(p % 16 == 0 for p in (a_out.data_ptr(), b.data_ptr(), *sources)) and all(in_own_place(sources, a_out)))


def _copies_stream(peers: PeerBuffers, a_out: torch.Tensor, copy_engine: bool, dev: torch.device) -> torch.cuda.Stream | None:
    """The stream of the copies, ``None`` for the side stream.  Copies that make a tangent of ``a_out`` run on the caller's, whose
    memory it then is."""
    return torch.cuda.current_stream(dev) if not copy_engine and has_tangent(a_out, *peers.tensors) else None


def _local_shard(peers: PeerBuffers, rank: int, a_out: torch.Tensor) -> torch.Tensor | None:
    """The shard that tiles read without waiting; ``None`` where another one's copy overwrites it meanwhile (its tiles then
    wait for their flags and read ``a_out``)."""
    return peers.slice(rank) if in_own_place(peers.pointers(), a_out)[rank] else None


def _gathered_first(a_out, peers: PeerBuffers, progress, splits: int, rank: int, dev) -> bool:
    """Gather on the current stream in one launch, in front of a product that then waits for nothing and may be any;
    False, and nothing done, where ``kr_gather_chunks`` does not take the addresses or a shard overlaps the gathered matrix.

    On one GPU nothing is gained by the side stream: its copies wait for compute units of the running product, and
    its events, flags and status word cost the host 100 us.  Calls one behind the other, us, with the side stream /
    in front: W = 8, 1 x 1024, N = 1024 125 / 38; 8 x 130 x 8192, N = 8192 205 / 176; 8 x 500 x 4096, N = 6656 232 / 188;
    8 x 1000 x 8192, N = 1024 286 / 185, N = 3584 450 / 389; 2 x 1000 x 16384, N = 8192 429 / 393.
    fp8 of whole tiles, whose product could follow the flags: 8 x 32 x 1024, N = 1024 104 / 29; 8 x 1024 x 4096, N = 3584 153 / 106,
    K = 8192 266 / 184; N = 8192, K = 16384 760 / 722; 63 shapes 0.25 to 0.96."""
    flags = progress
    if progress is None:
        flags = torch.empty(peers.W * splits, dtype=torch.int32, device=dev)     # counted in, read by nobody
    else:
        _check_progress(progress, peers.W * splits)
        progress.fill_(0)
    return gather_chunks(a_out, peers, flags, splits, rank, _lib.current_stream(dev))


def _all_gather_matmul_fp8(a_shared, peers: PeerBuffers, b, a_out, progress, **kwargs):
    """The fp8 branch of ``all_gather_matmul`` (``all_gather_matmul.py:53,121,213``): fp8 product, rounded to
    fp8 once.  Shapes of whole tiles (M, N multiples of 256, K of 128) run on
    the fp8 matrix-core instruction (``kr_gemm_fp8_ws``, or ``kr_all_gather_matmul_fp8`` where ``gather=True`` takes the
    side stream: the tiles wait for their chunk's flag, as in the
    bf16 form); others run on the bf16 instruction, their operands widened in registers (``kr_gemm_fp8_wide_ws``).  The
    shards are gathered in front of it.  ``fp8_kernel=False`` forces the widening kernel.

    The two differ in the precision of the sums: the fp8 instruction keeps about 16 bits of them (1.2e-5 in the
    2-norm against 64 bits, K = 128 .. 16384; both the 16x16x32 and the 16x16x128 form, to the same bits), the bf16
    instruction all 24 (2e-9 at K = 4096), so ragged shapes are not sent to the fp8 kernel although its C entry points
    take them: 4000 x 6656 x 4096 takes 83 us there and 139 us here, with 5e-4 of the results one fp8 step off."""
    fp8 = torch.float8_e4m3fn
    W = peers.W
    m, K = peers.shape
    assert b.dtype == fp8, "fp8 shards need an fp8 b"
    assert b.dim() == 2 and b.shape[0] == K
    if not b.T.is_contiguous():
        raise ValueError("b.T must be contiguous")
    stacked = peers.stacked is not None and peers.stacked.is_contiguous()
    gather = kwargs.get("gather", not stacked)
    M, N = W * m, b.shape[1]
    assert K % 16 == 0 and N % 16 == 0 and (M * N) % 16 == 0, "fp8 operands: sizes must be multiples of 16"
    rank = kwargs.get("rank", 0)
    assert 0 <= rank < W
    splits = kwargs.get("splits_per_rank", 1)
    dev = _lib.require_device(*peers.tensors, b, a_out, progress)
    lib = _lib.load()
    stream = _lib.current_stream(dev)
    native = kwargs.get("fp8_kernel", True) and M % 256 == 0 and N % 256 == 0 and K % 128 == 0
    if gather:
        assert m % splits == 0, "splits_per_rank must divide the rows of a shard"
        _waits.check()      # an earlier call's failed wait is reported before anything of this call is enqueued
        if a_out is None:
            a_out = torch.empty((M, K), dtype=fp8, device=dev)
        else:
            assert tuple(a_out.shape) == (M, K) and a_out.dtype == fp8 and a_out.is_contiguous()
        copy_engine = kwargs.get("copy_engine", False)
        if copy_engine or followed(a_out, peers) or not _gathered_first(a_out, peers, progress, splits, rank, dev):
            if progress is None:
                progress = torch.zeros(W * splits, dtype=torch.int32, device=dev)
            else:
                progress.fill_(0)
            backend_stream = _copy_engine_all_gather_w_progress(
                a_out, a_shared, progress, splits, _copies_stream(peers, a_out, copy_engine, dev), rank=rank, copy_engine=copy_engine)
            if native:
                status = kwargs.get("status")
                own_status = status is None
                if own_status:
                    status = _waits.new_status(dev)
                a_local = _local_shard(peers, rank, a_out)
                assert a_local is None or a_local.stride(1) == 1
                c = torch.empty((M, N), dtype=fp8, device=dev)
                rc = lib.kr_all_gather_matmul_fp8(
                    a_out.data_ptr(), K, _lib.ptr(a_local), 0 if a_local is None else a_local.stride(0), b.T.data_ptr(), K, M, N, K, W, rank, splits,
                    progress.data_ptr(), int(kwargs.get("wait_limit_us", 0)), _lib.ptr(status), c.data_ptr(), 2, stream)
                _lib.check(rc, "all_gather_matmul(fp8)")
                torch.cuda.current_stream(dev).wait_stream(backend_stream)
                if own_status:
                    _waits.watch(status, "all_gather_matmul")
                return a_out, c
            torch.cuda.current_stream(dev).wait_stream(backend_stream)   # no overlap on the widening path
        a_full = a_out
    else:
        assert stacked, "gather=False needs the shards as one contiguous [W, m, K] tensor"
        a_full = peers.stacked.reshape(M, K)
        if a_out is not None:
            assert a_out.shape == a_full.shape and a_out.dtype == fp8
            a_out.copy_(a_full)
        else:
            a_out = a_full
        if progress is not None:
            progress.fill_(1)
    if native:
        c = torch.empty((M, N), dtype=fp8, device=dev)
        ws = _gemm.workspace(dev, lib.kr_gemm_fp8_workspace_bytes(M, N, K))
        ws_ptr, ws_bytes = (ws.data_ptr(), ws.numel()) if ws is not None else (None, 0)
        _lib.check(lib.kr_gemm_fp8_ws(a_full.data_ptr(), K, b.T.data_ptr(), K, M, N, K, c.data_ptr(), 2, ws_ptr, ws_bytes, stream),
                   "all_gather_matmul(fp8)")
        return a_out, c
    c = torch.empty((M, N), dtype=fp8, device=dev)
    ws = _gemm.workspace(dev, lib.kr_gemm_fp8_wide_workspace_bytes(M, N, K))
    ws_ptr, ws_bytes = (ws.data_ptr(), ws.numel()) if ws is not None else (None, 0)
    _lib.check(lib.kr_gemm_fp8_wide_ws(a_full.data_ptr(), K, b.T.data_ptr(), K, M, N, K, c.data_ptr(), rank * m, ws_ptr, ws_bytes, stream),
               "all_gather_matmul(fp8)")
    return a_out, c


_DEFAULT = object()     # (None that is named means gather=False)


def _common_form(a_shared, b, a_out, progress, rank=0, splits_per_rank=1, gather=_DEFAULT, **kwargs):
    """The call in native code where its arguments are of the common form: nothing but sizes named, and no tangents about."""
    if kwargs or forward_ad._current_level >= 0:
        return None
    if gather is _DEFAULT:
        gather = not isinstance(a_shared, torch.Tensor)     # (a stack that is not contiguous goes the general way in any case)
    if type(gather) is not bool:
        return None
    return _lib.calls().gather_matmul(a_shared, b, a_out, progress, rank, splits_per_rank, gather)


def all_gather_matmul(
    a_shared,
    b: torch.Tensor,
    a_out: torch.Tensor | None = None,
    progress: torch.Tensor | None = None,
    **kwargs,
) -> tuple[torch.Tensor, torch.Tensor]:
    """``c = concat_r(a_shared[r]) @ b``; returns ``(a_gathered, c)``.

    Counterpart of ``kraken.fused.all_gather_matmul``
    (``kraken/fused/all_gather_matmul.py:222-325``; arithmetic ``:87-123``).
    ``a_shared`` holds all ranks' shards: the ``[W, m, K]`` stack or a list of
    W separate ``[m, K]`` tensors.  ``b`` must satisfy ``b.T.is_contiguous()``
    like in the reference (``:158-160``).  Two modes (kwarg ``gather``):

    * ``gather=False`` (default for a contiguous stack): the stack already is
      the gathered matrix, so ``a_gathered`` is its zero-copy ``[W*m, K]`` view
      (copied into ``a_out`` when one is passed), ``progress`` is set to 1
      everywhere and the GEMM waits for nothing.
    * ``gather=True`` (default for a list of shards): the reference's overlap.  With more than 128
      tiles of 256 x 256 and shards of whole tiles the product gathers the shards itself
      (``kr_gather_matmul_bf16``): tiles read their rows where the shards lie and write what they
      read to ``a_out`` while they multiply; the flags of ``progress`` are set behind it, no tile waits and
      ``status`` is not touched.  8 shards of 1024 x 8192, N = 3584: 397 us with copies and flags, 346 so.
      Other shapes are gathered by one launch in front of the product.
      With ``copy_engine=True``, and where shards are not 16-byte aligned, overlap ``a_out`` or are followed by autograd
      (they require a gradient, with gradients enabled, or carry a forward-mode tangent),
      the shards are copied chunk by chunk into ``a_out`` on a side stream,
      each chunk followed by its flag in ``progress`` (``:308-311``), while the
      GEMM on the current stream consumes them: tiles of the local shard
      (``rank``) read it in place, every other tile waits for its chunk's flag
      (``:95-110``).  The current stream then waits for the side stream
      (``:316``).  ``status`` (int32 ``[1]``, zeroed by the caller) receives a
      non-zero value if a tile's wait ran out (``wait_limit_us``, default 5 s) and
      ``c`` is then invalid; without ``status`` the wrapper keeps a word of its own
      and the next call of an overlap function (or ``kraken_amd._waits.check()``)
      raises once the failed call has finished.
      ``copy_engine=True`` hands the copies to the GPU's copy engines.

    In both modes the order of the M tiles is rotated so that the shard of
    ``rank`` (kwarg, default 0) is consumed first and the others in the order
    the copies are issued (``:93``).  ``splits_per_rank`` (default 1) chunks per
    shard; the remaining tile-size kwargs are accepted and ignored.

    fp8 operands (``torch.float8_e4m3fn`` for the shards and ``b``) give an fp8 ``c``
    like in the reference (``:53,121,213``): fp32 accumulate, one rounding to fp8
    (nearest even, magnitudes of 448 and more saturate to 448), in both modes.
    With M and N multiples of 256 and K of 128 the product runs on the fp8
    matrix-core instruction, whose sums keep about 16 bits; other sizes (multiples of 16,
    and ``fp8_kernel=False``) run on the bf16 instruction, after the gather has finished, their
    operands widened to bf16 in registers (exact: every e4m3 value is a bf16 value) and the
    fp32 sums rounded to fp8 once.
    ``a_gathered`` stays fp8.
    """
    out = _common_form(a_shared, b, a_out, progress, **kwargs)
    if out is not None:
        return out
    fp8 = torch.float8_e4m3fn
    peers = PeerBuffers(a_shared, dtypes=(torch.bfloat16, fp8))
    if peers.tensors[0].dtype == fp8:
        return _all_gather_matmul_fp8(a_shared, peers, b, a_out, progress, **kwargs)
    W = peers.W
    assert len(peers.shape) == 2, "expected shards of shape [m, K]"
    assert b.dtype == torch.bfloat16, "Only bfloat16 is supported for now."
    m, K = peers.shape
    assert b.dim() == 2 and b.shape[0] == K
    if not b.T.is_contiguous():
        raise ValueError("b.T must be contiguous")
    rank = kwargs.get("rank", 0)
    assert 0 <= rank < W
    splits = kwargs.get("splits_per_rank", 1)
    M, N = W * m, b.shape[1]
    assert N % 8 == 0, "N must be a multiple of 8"
    stacked = peers.stacked is not None and peers.stacked.is_contiguous()
    gather = kwargs.get("gather", not stacked)
    dev = _lib.require_device(*peers.tensors, b, a_out, progress)

    if not gather:
        assert stacked, "gather=False needs the shards as one contiguous [W, m, K] tensor"
        a_full = peers.stacked.reshape(M, K)
        if a_out is not None:
            assert a_out.shape == a_full.shape and a_out.dtype == a_full.dtype
            a_out.copy_(a_full)
        else:
            a_out = a_full
        if progress is not None:
            progress.fill_(1)
        c = _lib.calls().gemm(a_full, b, None, None, None, 0, M, False, rank * m)
        if c is None:
            a2, b2 = _gemm.prepare_operands(a_full, b)
            c = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
            _gemm.launch("all_gather_matmul", a2, b2, M, N, None, 0, 0, None, 0, M, None, c, rank * m)
        return a_out, c

    assert K % 8 == 0, "K must be a multiple of 8"
    assert m % splits == 0, "splits_per_rank must divide the rows of a shard"
    _waits.check()      # an earlier call's failed wait is reported before anything of this call is enqueued
    if a_out is None:
        a_out = torch.empty((M, K), dtype=torch.bfloat16, device=dev)
    else:
        assert tuple(a_out.shape) == (M, K) and a_out.dtype == torch.bfloat16 and a_out.is_contiguous()
    sources = peers.pointers()
    copy_engine = kwargs.get("copy_engine", False)
    side_stream = copy_engine or followed(a_out, peers)
    if not side_stream and _direct(sources, a_out, b, W, m, N, K):
        if progress is not None:
            _check_progress(progress, W * splits)
            progress.fill_(0)
        c = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
        rc = _lib.load().kr_gather_matmul_bf16((ctypes.c_void_p * W)(*sources), W, rank, m, a_out.data_ptr(), b.data_ptr(), b.stride(1),
                                               N, K, c.data_ptr(), _lib.current_stream(dev))
        _lib.check(rc, "all_gather_matmul")
        torch.autograd.graph.increment_version(a_out)
        if progress is not None:
            progress.view(-1)[:W * splits].fill_(1)
        return a_out, c
    if not side_stream and _gathered_first(a_out, peers, progress, splits, rank, dev):
        c = _lib.calls().gemm(a_out, b, None, None, None, 0, M, False, rank * m)
        if c is None:
            c = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
            _gemm.launch("all_gather_matmul", a_out, b, M, N, None, 0, 0, None, 0, M, None, c, rank * m)
        return a_out, c
    if progress is None:
        progress = torch.zeros(W * splits, dtype=torch.int32, device=dev)
    else:
        progress.fill_(0)
    backend_stream = _copy_engine_all_gather_w_progress(
        a_out, a_shared, progress, splits, _copies_stream(peers, a_out, copy_engine, dev), rank=rank, copy_engine=copy_engine)
    configs = {"RANK": rank, "WORLD_SIZE": W, "SPLITS_PER_RANK": splits,
               "wait_limit_us": kwargs.get("wait_limit_us", 0)}
    status = kwargs.get("status")
    own_status = status is None
    if own_status:
        status = _waits.new_status(dev)
    c = _matmul_w_progress(a_out, _local_shard(peers, rank, a_out), b, progress, configs, status)
    torch.cuda.current_stream(dev).wait_stream(backend_stream)
    if own_status:
        _waits.watch(status, "all_gather_matmul")
    return a_out, c
