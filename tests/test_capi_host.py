"""Host side of the C ABI, exercised without a GPU: the library loads, exports every symbol
include/kraken_amd.h declares, and rejects bad arguments before any launch.  The Python
wrappers raise like the reference's asserts and refuse host tensors (no CPU fallback)."""
import ctypes
import re
from pathlib import Path

import pytest
import torch

import kraken_amd
from kraken_amd import _lib, comm, fused

ROOT = Path(__file__).resolve().parent.parent
BF16 = torch.bfloat16
FAKE = 0x10000  # aligned, non-null; never dereferenced because validation fails first


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def test_library_exports_every_declared_symbol(lib):
    header = (ROOT / "include" / "kraken_amd.h").read_text()
    declared = set(re.findall(r"\b(kr_[a-z0-9_]+)\s*\(", header))
    assert declared, "no declarations found"
    assert declared == set(_lib.EXPORTS)
    raw = ctypes.CDLL(str(_lib.LIB_PATH))
    for name in declared:
        assert hasattr(raw, name), f"{name} not exported"
    assert lib.kr_version() >= 100


def test_strerror_known_and_unknown(lib):
    assert "128-bit" in _lib.strerror(_lib.KR_ERR_NUMEL_MOD8)
    assert _lib.strerror(0) == "success"
    assert "unknown" in _lib.strerror(-999)


def test_reduce_argument_errors(lib):
    f = lib.kr_reduce_bf16
    assert f(FAKE, 8, 64, 12, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_NUMEL_MOD8
    assert f(FAKE, 0, 64, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_WORLD_SIZE
    assert f(FAKE, 17, 64, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_WORLD_SIZE
    assert f(None, 8, 64, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(FAKE, 8, 64, 16, None, 0, 0, 1, None, None) == _lib.KR_ERR_NULL_POINTER
    assert f(FAKE + 2, 8, 64, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_ALIGNMENT
    assert f(FAKE, 8, 60, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_ALIGNMENT
    assert f(FAKE, 8, 64, -8, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_BAD_DIM
    assert f(FAKE, 8, 64, 64, FAKE, 24, 16, 1, FAKE, None) == _lib.KR_ERR_BIAS_SHAPE
    assert f(FAKE, 8, 64, 64, FAKE + 4, 64, 16, 1, FAKE, None) == _lib.KR_ERR_ALIGNMENT
    # empty input: nothing to do, nothing launched
    assert f(None, 8, 0, 0, None, 0, 0, 1, None, None) == 0


def test_rmsnorm_argument_errors(lib):
    f = lib.kr_reduce_rmsnorm_bf16
    assert f(FAKE, 8, 4096, 1, 4100, None, 0, FAKE, 1e-5, FAKE, None) == _lib.KR_ERR_NUMEL_MOD8
    assert f(FAKE, 8, 1 << 20, 1, 65536 + 8, None, 0, FAKE, 1e-5, FAKE, None) == _lib.KR_ERR_ROW_TOO_LONG
    assert f(FAKE, 8, 4096, 1, 4096, None, 0, None, 1e-5, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(FAKE, 99, 4096, 1, 4096, None, 0, FAKE, 1e-5, FAKE, None) == _lib.KR_ERR_WORLD_SIZE
    assert f(FAKE, 8, 4096, 0, 4096, None, 0, FAKE, 1e-5, FAKE, None) == 0
    g = lib.kr_rmsnorm_bf16
    assert g(FAKE, FAKE, 1e-5, 4, 0, FAKE, None) == _lib.KR_ERR_BAD_DIM
    assert g(FAKE, FAKE + 8, 1e-5, 4, 64, FAKE, None) == _lib.KR_ERR_ALIGNMENT


def test_rmsnorm_workspace_entries(lib, monkeypatch):
    """Which shapes the split-row kernel takes (a few long rows), and that the workspace forms
    validate like the plain ones."""
    q = lib.kr_rmsnorm_workspace_bytes
    need = q(8, 16, 8192)
    assert need > 0 and q(8, 1, 8192) == need and q(4, 16, 32768) == need
    assert q(8, 256, 4096) == 0 and q(8, 16, 1024) == 0 and q(3, 16, 8192) == 0 and q(8, 128, 8192) == 0
    assert q(8, 16, 8190) == 0 and q(8, 0, 8192) == 0 and q(8, 2, 65536) == 0
    f = lib.kr_reduce_rmsnorm_ws_bf16
    assert f(FAKE, 8, 8192 * 16, 16, 8192, None, 0, FAKE, 1e-5, FAKE, FAKE + 8, need, None, None) == _lib.KR_ERR_ALIGNMENT
    assert f(FAKE, 8, 8192 * 16, 16, 8196, None, 0, FAKE, 1e-5, FAKE, FAKE, need, None, None) == _lib.KR_ERR_NUMEL_MOD8
    assert f(None, 8, 8192 * 16, 16, 8192, None, 0, FAKE, 1e-5, FAKE, FAKE, need, None, None) == _lib.KR_ERR_NULL_POINTER
    # the status word of the bounded exchange: 4-byte aligned or NULL
    assert f(FAKE, 8, 8192 * 16, 16, 8192, None, 0, FAKE, 1e-5, FAKE, FAKE, need, FAKE + 2, None) == _lib.KR_ERR_ALIGNMENT
    assert f(FAKE, 8, 8192 * 16, 0, 8192, None, 0, FAKE, 1e-5, FAKE, FAKE, need, FAKE, None) == 0
    g = lib.kr_reduce_rmsnorm_ptrs_ws_bf16
    assert g(None, 8, 16, 8192, None, 0, FAKE, 1e-5, FAKE, FAKE, need, None, None) == _lib.KR_ERR_NULL_POINTER
    monkeypatch.setenv("KRAKEN_AMD_ROW_SPLIT", "0")
    assert q(8, 16, 8192) == 0
    monkeypatch.setenv("KRAKEN_AMD_ROW_SPLIT", "1")
    assert q(8, 64, 1024) == need and q(8, 65, 1024) == 0 and q(8, 1, 512) == 0   # 64 rows at most, two wavefronts at least


def test_gemm_argument_errors(lib):
    f = lib.kr_gemm_reduce_bf16

    def call(**kw):
        a = dict(A=FAKE, lda_m=64, lda_k=1, B=FAKE, ldb_k=64, ldb_n=1, M=64, N=64, K=64, peers=None,
                 n_peers=0, pstride=0, bias=None, band0=0, band=64, c_full=None, out=FAKE, f32=0, pivot=0)
        a.update(kw)
        return f(a["A"], a["lda_m"], a["lda_k"], a["B"], a["ldb_k"], a["ldb_n"], a["M"], a["N"], a["K"],
                 a["peers"], a["n_peers"], a["pstride"], a["bias"], a["band0"], a["band"], a["c_full"],
                 a["out"], a["f32"], a["pivot"], None)

    assert call(K=60) == _lib.KR_ERR_NUMEL_MOD8
    assert call(N=60) == _lib.KR_ERR_NUMEL_MOD8
    assert call(lda_k=2) == _lib.KR_ERR_LAYOUT
    assert call(ldb_k=3, ldb_n=5) == _lib.KR_ERR_LAYOUT
    assert call(band0=32, band=64) == _lib.KR_ERR_BAND
    assert call(A=None) == _lib.KR_ERR_NULL_POINTER
    assert call(out=None) == _lib.KR_ERR_NULL_POINTER
    assert call(n_peers=3, peers=None) == _lib.KR_ERR_NULL_POINTER
    assert call(n_peers=3, peers=FAKE, pstride=64) == _lib.KR_ERR_BAD_DIM
    assert call(lda_m=68) == _lib.KR_ERR_ALIGNMENT
    assert call(M=-1) == _lib.KR_ERR_BAD_DIM
    assert call(M=0, band=0) == 0


def _table(*ptrs):
    return (ctypes.c_void_p * len(ptrs))(*ptrs)


def test_pointer_table_argument_errors(lib):
    """The kr_*_ptrs_bf16 forms reject what their stacked forms reject, and a bad table entry."""
    good = _table(*[FAKE + 4096 * r for r in range(8)])
    f = lib.kr_reduce_ptrs_bf16
    assert f(good, 8, 12, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_NUMEL_MOD8
    assert f(good, 0, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_WORLD_SIZE
    assert f(good, 17, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_WORLD_SIZE
    assert f(None, 8, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(good, 8, 16, None, 0, 0, 1, None, None) == _lib.KR_ERR_NULL_POINTER
    assert f(_table(FAKE, None), 2, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(_table(FAKE, FAKE + 8), 2, 16, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_ALIGNMENT
    assert f(good, 8, 64, FAKE, 24, 16, 1, FAKE, None) == _lib.KR_ERR_BIAS_SHAPE
    assert f(good, 8, -8, None, 0, 0, 1, FAKE, None) == _lib.KR_ERR_BAD_DIM
    assert f(None, 8, 0, None, 0, 0, 1, None, None) == 0

    f = lib.kr_reduce_striped_ptrs_bf16
    assert f(good, 8, 4096, None, 12, 0, FAKE, None) == _lib.KR_ERR_STRIPE
    assert f(good, 8, 4096, None, 256, 8, FAKE, None) == _lib.KR_ERR_STRIPE
    assert f(_table(FAKE, FAKE + 2), 2, 4096, None, 256, 0, FAKE, None) == _lib.KR_ERR_ALIGNMENT
    assert f(None, 8, 4096, None, 256, 0, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(good, 8, 256, None, 256, 3, FAKE, None) == 0   # rank 3 owns nothing of a 256-element input

    f = lib.kr_reduce_rmsnorm_ptrs_bf16
    assert f(good, 8, 1, 4100, None, 0, FAKE, 1e-5, FAKE, None) == _lib.KR_ERR_NUMEL_MOD8
    assert f(good, 8, 1, 65536 + 8, None, 0, FAKE, 1e-5, FAKE, None) == _lib.KR_ERR_ROW_TOO_LONG
    assert f(good, 8, 1, 4096, None, 0, None, 1e-5, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(None, 8, 1, 4096, None, 0, FAKE, 1e-5, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(_table(FAKE + 6), 1, 1, 4096, None, 0, FAKE, 1e-5, FAKE, None) == _lib.KR_ERR_ALIGNMENT
    assert f(good, 8, 0, 4096, None, 0, None, 1e-5, None, None) == 0

    f = lib.kr_gemm_reduce_ptrs_bf16
    def args(**kw):
        a = dict(A=FAKE, lda_m=64, lda_k=1, B=FAKE, ldb_k=64, ldb_n=1, M=64, N=64, K=64, peers=None, n_peers=0,
                 bias=None, band_row0=0, band_rows=64, c_full=None, out=FAKE, out_is_fp32=0, tile_pivot=0,
                 stream=None)
        a.update(kw)
        return tuple(a.values())
    assert f(*args(n_peers=2, peers=None)) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(n_peers=2, peers=_table(FAKE, None))) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(n_peers=2, peers=_table(FAKE, FAKE + 4))) == _lib.KR_ERR_ALIGNMENT
    assert f(*args(n_peers=16, peers=good)) == _lib.KR_ERR_WORLD_SIZE
    assert f(*args(n_peers=2, peers=good, band_row0=32, band_rows=64)) == _lib.KR_ERR_BAND
    assert f(*args(n_peers=2, peers=good, lda_k=2)) == _lib.KR_ERR_LAYOUT
    assert f(*args(n_peers=2, peers=good, M=0, band_rows=0)) == 0


def test_wrappers_accept_a_list_of_buffers_and_check_it():
    bufs = [torch.zeros(4, 16, dtype=BF16) for _ in range(3)]
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        comm.one_shot_all_reduce(bufs)
    with pytest.raises(AssertionError, match="one shape"):
        comm.one_shot_all_reduce([bufs[0], torch.zeros(4, 8, dtype=BF16)])
    with pytest.raises(AssertionError, match="bfloat16"):
        comm.one_shot_all_reduce([bufs[0], torch.zeros(4, 16)])
    with pytest.raises(AssertionError, match="contiguous"):
        comm.one_shot_all_reduce([bufs[0], torch.zeros(16, 4, dtype=BF16).T])
    a = torch.zeros(8, 16, dtype=BF16)
    b = torch.zeros(16, 8, dtype=BF16)
    with pytest.raises(AssertionError, match="every peer"):
        fused.gemm_one_shot_all_reduce_fused(a, b, peers=[torch.zeros(8, 16, dtype=BF16)])
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        fused.gemm_one_shot_all_reduce_fused(a, b, peers=[torch.zeros(8, 8, dtype=BF16)])


def test_all_gather_matmul_argument_errors(lib):
    f = lib.kr_all_gather_matmul_bf16
    def args(**kw):
        a = dict(A=FAKE, lda_m=64, A_local=FAKE, lda_local=64, B=FAKE, ldb_k=1, ldb_n=64, M=512, N=64, K=64,
                 W=4, rank=1, splits=2, progress=FAKE, wait_us=0, status=FAKE, C=FAKE, stream=None)
        a.update(kw)
        return tuple(a.values())
    assert f(*args(W=0)) == _lib.KR_ERR_WORLD_SIZE
    assert f(*args(W=17)) == _lib.KR_ERR_WORLD_SIZE
    assert f(*args(rank=4)) == _lib.KR_ERR_STRIPE
    assert f(*args(splits=0)) == _lib.KR_ERR_STRIPE
    assert f(*args(M=500)) == _lib.KR_ERR_BAND             # 500 rows do not split into 4*2 chunks
    assert f(*args(A_local=FAKE + 2)) == _lib.KR_ERR_ALIGNMENT
    assert f(*args(lda_local=32)) == _lib.KR_ERR_LAYOUT      # shorter than K
    assert f(*args(progress=FAKE + 2)) == _lib.KR_ERR_ALIGNMENT
    assert f(*args(status=FAKE + 1)) == _lib.KR_ERR_ALIGNMENT
    assert f(*args(A=None)) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(C=None)) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(K=60)) == _lib.KR_ERR_NUMEL_MOD8
    assert f(*args(ldb_k=2, ldb_n=3)) == _lib.KR_ERR_LAYOUT
    assert f(*args(M=0)) == 0
    g = lib.kr_stream_write_value32
    assert g(None, 1, None) == _lib.KR_ERR_NULL_POINTER
    assert g(FAKE + 2, 1, None) == _lib.KR_ERR_ALIGNMENT


def test_gemm_row_stride_beyond_the_kernels_reach(lib):
    # a row stride of 2^24 elements: 128 rows of a tile span 4 GiB, more than the operand descriptors cover
    f = lib.kr_gemm_reduce_bf16
    assert f(FAKE, 1 << 24, 1, FAKE, 64, 1, 128, 64, 64, None, 0, 0, None, 0, 128, None, FAKE, 0, 0,
             None) == _lib.KR_ERR_LAYOUT
    assert f(FAKE, 64, 1, FAKE, 1, 1 << 24, 128, 64, 64, None, 0, 0, None, 0, 128, None, FAKE, 0, 0,
             None) == _lib.KR_ERR_LAYOUT


@pytest.mark.parametrize("M", [1, 16, 64, 65, 128])
def test_gemm_row_stride_rule_does_not_depend_on_the_rows(lib, M):
    """128 rows of an operand must lie within 2 GiB, as the header says, also for a product of a few rows."""
    f, N, K, wide = lib.kr_gemm_reduce_bf16, 256, 64, (1 << 23) + 8
    for lda, lk, ln in ((wide, N, 1), (K, wide, 1), (K, 1, wide)):
        assert f(FAKE, lda, 1, FAKE, lk, ln, M, N, K, None, 0, 0, None, 0, M, None, FAKE, 0, 0, None) == _lib.KR_ERR_LAYOUT
    f32 = lib.kr_gemm_reduce_f32_ws
    for lda, lk, ln in ((wide // 2, N, 1), (K, wide // 2, 1), (K, 1, wide // 2)):
        assert f32(FAKE, lda, 1, FAKE, lk, ln, M, N, K, None, 0, None, 0, M, None, FAKE, 1, 0, None, 0, None) == _lib.KR_ERR_LAYOUT


def test_gemm_producer_argument_errors(lib):
    f = lib.kr_gemm_producer_bf16
    def args(**kw):
        a = dict(A=FAKE, lda_m=64, lda_k=1, B=FAKE, ldb_k=64, ldb_n=1, M=512, N=64, K=64, C=FAKE, W=4, rank=1,
                 progress=FAKE, signal=FAKE, stream=None)
        a.update(kw)
        return tuple(a.values())
    assert f(*args(W=0)) == _lib.KR_ERR_WORLD_SIZE
    assert f(*args(W=17)) == _lib.KR_ERR_WORLD_SIZE
    assert f(*args(rank=4)) == _lib.KR_ERR_BAND
    assert f(*args(rank=-1)) == _lib.KR_ERR_BAND
    assert f(*args(M=510)) == _lib.KR_ERR_BAD_DIM             # 510 rows do not split into 4 bands
    assert f(*args(progress=None)) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(signal=None)) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(C=None)) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(progress=FAKE + 2)) == _lib.KR_ERR_ALIGNMENT
    assert f(*args(signal=FAKE + 1)) == _lib.KR_ERR_ALIGNMENT
    assert f(*args(A=None)) == _lib.KR_ERR_NULL_POINTER
    assert f(*args(K=60)) == _lib.KR_ERR_NUMEL_MOD8
    assert f(*args(lda_k=2)) == _lib.KR_ERR_LAYOUT
    assert f(*args(C=FAKE + 8)) == _lib.KR_ERR_ALIGNMENT
    assert f(*args(M=0)) == 0                                 # nothing to compute, nothing launched
    g = lib.kr_stream_wait_value32
    assert g(None, 1, 0, None, None) == _lib.KR_ERR_NULL_POINTER
    assert g(FAKE + 2, 1, 0, None, None) == _lib.KR_ERR_ALIGNMENT
    assert g(FAKE, 1, 0, FAKE + 1, None) == _lib.KR_ERR_ALIGNMENT
    assert g(FAKE, 1, -5, None, None) == _lib.KR_ERR_BAD_DIM
    k = lib.kr_flag_arrive_wait
    assert k(None, 8, 32, 0, None, None) == _lib.KR_ERR_NULL_POINTER
    assert k(FAKE, 0, 32, 0, None, None) == _lib.KR_ERR_BAD_DIM
    assert k(FAKE, 8, 30, 0, None, None) == _lib.KR_ERR_STRIPE          # consumers per producer must be whole
    assert k(FAKE + 2, 8, 32, 0, None, None) == _lib.KR_ERR_ALIGNMENT
    h = lib.kr_copy_engine_memcpy
    assert h(FAKE, FAKE + 64, -1, None) == _lib.KR_ERR_BAD_DIM
    assert h(None, None, 0, None) == 0                        # nothing to copy
    assert h(None, FAKE, 16, None) == _lib.KR_ERR_NULL_POINTER
    assert h(FAKE, None, 16, None) == _lib.KR_ERR_NULL_POINTER


def test_gemm_workspace_entries(lib):
    assert lib.kr_gemm_workspace_bytes(0, 128, 128) == 0
    assert lib.kr_gemm_workspace_bytes(8192, 8192, 8192) == 0
    need = lib.kr_gemm_workspace_bytes(128, 6656, 4096)
    assert need >= 2 * 128 * 6656 * 4 and need % (128 * 6656 * 4) == 0   # S fp32 partial products
    f = lib.kr_gemm_reduce_ws_bf16
    base = (FAKE, 4096, 1, FAKE, 6656, 1, 128, 6656, 4096, None, 0, 0, None, 0, 128, None, FAKE, 0, 0)
    assert f(*base, FAKE + 8, need, None) == _lib.KR_ERR_ALIGNMENT     # workspace not 16-byte aligned
    assert f(FAKE, 4096, 2, *base[3:], FAKE, need, None) == _lib.KR_ERR_LAYOUT
    g = lib.kr_gemm_reduce_ptrs_ws_bf16
    assert g(FAKE, 4096, 1, FAKE, 6656, 1, 128, 6656, 4096, None, 2, None, 0, 128, None, FAKE, 0, 0,
             FAKE, need, None) == _lib.KR_ERR_NULL_POINTER


def test_gemm_noalloc_entry_checks_arguments_first(lib, monkeypatch):
    """The allocation-free form validates like the others (nothing is looked up or launched for
    a rejected call) and refuses a split that its static scratch cannot hold."""
    f = lib.kr_gemm_reduce_noalloc_bf16
    base = (FAKE, 4096, 1, FAKE, 6656, 1, 128, 6656, 4096, None, 0, 0, None, 0, 128, None, FAKE, 0, 0)
    assert f(FAKE, 4096, 2, *base[3:], None) == _lib.KR_ERR_LAYOUT
    assert f(None, *base[1:], None) == _lib.KR_ERR_NULL_POINTER
    assert f(FAKE + 4, *base[1:], None) == _lib.KR_ERR_ALIGNMENT
    assert f(*base[:6], 0, 6656, 4096, None, 0, 0, None, 0, 0, None, FAKE, 0, 0, None) == 0   # M == 0: nothing to do
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "128")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_SPLITK", "16")                  # 16 partial products of 1024 x 2048 fp32
    assert lib.kr_gemm_workspace_bytes(1024, 2048, 4096) == 16 * 1024 * 2048 * 4 > (64 << 20)
    assert f(FAKE, 4096, 1, FAKE, 2048, 1, 1024, 2048, 4096, None, 0, 0, None, 0, 1024, None, FAKE, 0, 0,
             None) == _lib.KR_ERR_SCRATCH
    # an oversize shape with a bad argument reports the argument, as every other entry point would
    assert f(None, 4096, 1, FAKE, 2048, 1, 1024, 2048, 4096, None, 0, 0, None, 0, 1024, None, FAKE, 0, 0,
             None) == _lib.KR_ERR_NULL_POINTER
    assert f(FAKE + 2, 4096, 1, FAKE, 2048, 1, 1024, 2048, 4096, None, 0, 0, None, 0, 1024, None, FAKE, 0, 0,
             None) == _lib.KR_ERR_ALIGNMENT
    assert f(FAKE, 4096, 2, FAKE, 2048, 1, 1024, 2048, 4096, None, 0, 0, None, 0, 1024, None, FAKE, 0, 0,
             None) == _lib.KR_ERR_LAYOUT
    assert "scratch" in _lib.strerror(_lib.KR_ERR_SCRATCH)


def test_gemm_plan_reports_the_dispatch(lib, monkeypatch):
    """kr_gemm_plan names the kernel a shape gets, by the rule the launch itself uses."""
    p = _lib.gemm_plan(8192, 8192, 3584, False, 7, 1024, False, True)        # GEMM + reduce-scatter shape
    assert p["kernel"] == "gemm_dtl16_kernel" and p["tile"] == 256 and p["mfma"] == "16x16x32" and p["peers_on_mfma"]
    p = _lib.gemm_plan(4096, 8192, 1024, False, 7, 4096, True, False)        # every tile streams peers
    assert p["kernel"] == "gemm_dtl16_kernel" and p["mfma"] == "16x16x32" and p["peers_on_mfma"] and p["group_n"] == 16
    p = _lib.gemm_plan(8192, 3584, 8192, True)                               # all-gather matmul shape: 448 tiles of 256 columns
    assert p["kernel"] == "gemm_dtl16n7_kernel" and p["tile_n"] == 224 and p["group_n"] == 4 and p["tail_tiles"] == 0   # 512 of 224
    assert _lib.gemm_plan(8192, 3584, 8192, False)["tile_n"] == 256          # row-major B: no 224-column form
    assert _lib.gemm_plan(8192, 3584, 8192, True, 7, 8192)["tile_n"] == 256  # peers: not a plain product
    assert _lib.gemm_plan(8192, 3584, 8192, True, has_bias=True)["tile_n"] == 256
    assert _lib.gemm_plan(8192, 7168, 4096, True)["tile_n"] == 224           # 896 tiles = 3.5 rounds against 1024 = 4 rounds of 224
    assert _lib.gemm_plan(8192, 14336, 4096, True)["tile_n"] == 256          # 1792 tiles = 7 whole rounds already
    assert _lib.gemm_plan(8192, 4096, 8192, True)["tile_n"] == 256           # 224 does not divide N
    p = _lib.gemm_plan(256, 256, 100 * 8, False)                             # K not a multiple of 64
    assert p["kernel"] == "gemm_ks_kernel" and p["tile"] == 128 and p["k_splits"] == 1
    need = lib.kr_gemm_workspace_bytes(128, 6656, 4096)
    p = _lib.gemm_plan(128, 6656, 4096, False, workspace_bytes=need)         # few tiles: split K loop
    assert p["tile"] == 128 and p["k_splits"] > 1
    assert _lib.gemm_plan(128, 6656, 4096, False)["k_splits"] == 1           # no workspace, no split
    p = _lib.gemm_plan(4352, 4096, 8192, False, workspace_bytes=1 << 30)     # 272 tiles: 16 tail tiles split
    assert p["tile"] == 256 and p["tail_tiles"] == 16 and p["tail_splits"] == 8
    assert _lib.gemm_plan(300, 8192 + 8, 4096, False)["ragged"]
    plan = (ctypes.c_int32 * 8)()
    assert lib.kr_gemm_plan(0, 64, 64, 0, 0, 0, 0, 0, 0, plan) == _lib.KR_ERR_BAD_DIM
    assert lib.kr_gemm_plan(64, 64, 64, 0, 16, 0, 0, 0, 0, plan) == _lib.KR_ERR_WORLD_SIZE
    assert lib.kr_gemm_plan(64, 64, 64, 0, 0, 65, 0, 0, 0, plan) == _lib.KR_ERR_BAND
    assert lib.kr_gemm_plan(64, 64, 64, 0, 0, 0, 0, 0, 0, None) == _lib.KR_ERR_NULL_POINTER
    monkeypatch.setenv("KRAKEN_AMD_GEMM_MFMA", "32")
    _lib.reload_env()
    try:
        assert _lib.gemm_plan(8192, 4096, 8192, True)["kernel"] == "gemm_dtl_kernel"
    finally:
        monkeypatch.delenv("KRAKEN_AMD_GEMM_MFMA")
        _lib.reload_env()


@pytest.mark.parametrize("mode", [None, "mfma", "first", "last", "epilogue"])
def test_gemm_plan_peers_of_a_ragged_k_stay_in_the_epilogue(lib, monkeypatch, mode):
    """Peers are added on the matrix cores only where K is a multiple of 64, which is the condition the header gives
    for a non-finite partial sum spreading over its 16 columns."""
    if mode is not None:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_PEERS", mode)
    for b_t in (False, True):
        for K in (4112, 4104, 264):
            p = _lib.gemm_plan(4096, 4096, K, b_t, 7, 4096)
            assert p["tile"] == 256 and not p["peers_on_mfma"]
        assert _lib.gemm_plan(4096, 4096, 4096, b_t, 7, 4096)["peers_on_mfma"] == (mode != "epilogue")


@pytest.mark.parametrize("M,N,K,b_t,kernel,mfma", [
    (512, 4096, 1024, False, "gemm_ks_kernel", "16x16x32"),
    (128, 6656, 4096, False, "gemm_ks_kernel", "16x16x32"),
    (128, 6656, 4096, True, "gemm_reduce_kernel", "32x32x16"),        # transposed B and peers
    (256, 256, 800, False, "gemm_ks_kernel", "16x16x32"),
    (1000, 6656, 1024, True, "gemm_reduce_kernel", "32x32x16"),       # 416 tiles (transposed B)
    (1000, 6656, 12288, True, "gemm_reduce_kernel", "32x32x16"),
    (1000, 6656, 4096, False, "gemm_ks_kernel", "16x16x32"),
    (1000, 4096, 8192, True, "gemm_reduce_kernel", "32x32x16"),
    (1000, 4096, 12288, True, "gemm_reduce_kernel", "32x32x16"),      # 256 tiles, K above 8192 (transposed B)
    (1000, 4096, 12288, False, "gemm_ks_kernel", "16x16x32"),
    (2048, 4096, 512, False, "gemm_reduce_kernel", "32x32x16"),       # 512 tiles, K below 2048 (row-major B)
    (4352, 1496, 1984, False, "gemm_reduce_kernel", "32x32x16"),
    (4352, 1496, 2048, False, "gemm_ks_kernel", "16x16x32"),
    (4352, 1496, 4104, False, "gemm_reduce_kernel", "32x32x16"),      # 408 tiles, K no multiple of 64
    (1000, 4096, 1032, False, "gemm_ks_kernel", "16x16x32"),          # 256 tiles: any K
    (256, 256, 56, False, "gemm_reduce_kernel", "32x32x16"),          # no whole k-step
    (16, 8192, 3584, True, "gemm_skinny_kernel", "16x16x32"),
    (4096, 4096, 4096, True, "gemm_dtl16_kernel", "16x16x32"),
])
def test_gemm_plan_names_every_kernel(lib, M, N, K, b_t, kernel, mfma):
    p = _lib.gemm_plan(M, N, K, b_t, 7, M)
    assert (p["kernel"], p["mfma"]) == (kernel, mfma)


@pytest.mark.parametrize("M,N,K", [(256, 7168, 12928), (512, 5376, 6400), (768, 3584, 13760)])
def test_gemm_plan_few_tiles_stay_split_where_224_divides_n(lib, M, N, K):
    """A plain product with transposed B whose few 256 x 256 tiles share their K loops keeps them where N is also a
    multiple of 224."""
    p = _lib.gemm_plan(M, N, K, True, workspace_bytes=lib.kr_gemm_workspace_bytes(M, N, K))
    assert p["tile_n"] == 256 and p["tail_tiles"] == (M // 256) * (N // 256) and p["tail_splits"] > 1


@pytest.mark.parametrize("M,N,K,b_t,P,cols,ragged", [
    (512, 6656, 8192, True, 7, 224, True), (512, 6720, 8192, True, 7, 224, False), (512, 6656, 8192, False, 7, 256, False),
    (500, 6656, 8192, False, 7, 256, True),
])
def test_gemm_plan_names_the_launch_of_tiles_that_are_all_split(lib, M, N, K, b_t, P, cols, ragged):
    p = _lib.gemm_plan(M, N, K, b_t, P, M // 8, False, True, workspace_bytes=lib.kr_gemm_workspace_bytes(M, N, K))
    assert p["tail_tiles"] == -(-M // 256) * -(-N // cols) and p["tail_splits"] > 1
    assert (p["kernel"], p["tile_n"], p["ragged"]) == ("gemm_dtl_split_kernel", cols, ragged)


@pytest.mark.parametrize("M,N,K,b_t,P,band", [
    (1422, 1088, 7424, False, 0, 1),      # us, 128 x 128 tiles / 256 x 256 in parts: 40.7 / 47.1
    (632, 2304, 6208, False, 7, 8),       # 37.7 / 42.2
    (1208, 1216, 5696, False, 7, 8),      # 34.0 / 39.0
    (640, 4608, 5120, False, 7, 1),       # 50.4 / 57.2
    (512, 4352, 4096, False, 7, 8),       # 32.4 / 39.2
    (512, 4352, 3072, True, 7, 8),        # 29.5 / 33.9
    (2816, 2560, 3072, False, 7, 8),      # 52.9 / 63.5
])
def test_gemm_plan_keeps_small_tiles_where_large_ones_in_parts_are_slower(lib, M, N, K, b_t, P, band):
    p = _lib.gemm_plan(M, N, K, b_t, P, M // band, False, band > 1, workspace_bytes=lib.kr_gemm_workspace_bytes(M, N, K))
    assert p["tail_splits"] == 1


@pytest.mark.parametrize("M,N,K,b_t,tile", [
    (4096, 4672, 416, True, 128), (4096, 4672, 632, True, 128),      # 304 tiles of 256 x 256: a second round of 48
    (4096, 4672, 416, False, 256), (4096, 4672, 384, True, 256), (4096, 4672, 640, True, 256), (4096, 4672, 648, True, 256),
    (4096, 5120, 416, True, 128), (4096, 5376, 416, True, 256),      # 320, 336 tiles
])
def test_gemm_plan_of_a_short_ragged_k(lib, M, N, K, b_t, tile):
    """Transposed B, K below 640 and no multiple of 64: 128 x 128 tiles unless the rounds of large ones are 5/8 full."""
    need = lib.kr_gemm_workspace_bytes(M, N, K)
    p = _lib.gemm_plan(M, N, K, b_t, 3, M, workspace_bytes=need)
    assert p["tile"] == tile and p["k_splits"] == 1
    assert p == _lib.gemm_plan(M, N, K, b_t, 3, M, workspace_bytes=1 << 40)


@pytest.mark.parametrize("M,N,K,b_t,splits", [
    (1280, 2304, 14224, True, 2), (1272, 2304, 12296, True, 2), (1272, 2304, 12280, True, 1), (1280, 2304, 14224, False, 1),
    (2048, 2048, 12296, True, 2), (2048, 2056, 12296, True, 1),      # 256, 272 tiles
])
def test_gemm_plan_long_k_with_up_to_256_tiles(lib, M, N, K, b_t, splits):
    """Transposed B: two workgroups per tile, on one compute unit, from K = 12288 on."""
    need = lib.kr_gemm_workspace_bytes(M, N, K)
    p = _lib.gemm_plan(M, N, K, b_t, 1, M, workspace_bytes=need)
    assert (p["tile"], p["k_splits"]) == (128, splits)
    assert splits * M * N * 4 <= need or splits == 1
    assert p == _lib.gemm_plan(M, N, K, b_t, 1, M, workspace_bytes=1 << 40)
    assert _lib.gemm_plan(M, N, K, b_t, 1, M)["k_splits"] == 1       # no workspace


@pytest.mark.parametrize("M,N,K,b_t,few", [
    (64, 2048, 4096, True, True), (64, 2048, 4104, True, False), (64, 2040, 4104, True, True), (33, 2048, 4104, True, False),
    (64, 2048, 3584, False, True), (64, 2048, 3592, False, False), (64, 2040, 3592, False, True),
    (32, 2048, 11264, True, True), (32, 2048, 11272, True, False), (32, 2040, 11272, True, True), (17, 2048, 11272, True, False),
    (32, 2048, 16384, False, True), (16, 8192, 16384, True, True), (16, 8192, 16384, False, True),
])
def test_gemm_plan_few_rows_up_to_a_k(lib, M, N, K, b_t, few):
    """Wide outputs with a long K: from 17 rows on the few-rows kernel is left for one with 128 x 128 tiles."""
    need = lib.kr_gemm_workspace_bytes(M, N, K)
    p = _lib.gemm_plan(M, N, K, b_t, workspace_bytes=need)
    assert (p["kernel"] == "gemm_skinny_kernel") == few
    assert few or p["k_splits"] > 1
    assert p == _lib.gemm_plan(M, N, K, b_t, workspace_bytes=1 << 40)


@pytest.mark.parametrize("M,N,K,P,kernel", [
    (1000, 4096, 1984, 0, "gemm_ks_kernel"),         # one pass, no peers, whole k-steps
    (256, 512, 640, 0, "gemm_ks_kernel"),
    (256, 512, 576, 0, "gemm_reduce_kernel"),        # K below 640
    (256, 512, 648, 0, "gemm_reduce_kernel"),        # K no multiple of 64
    (1000, 4224, 1984, 0, "gemm_reduce_kernel"),     # 264 tiles
    (256, 512, 4096, 0, "gemm_reduce_kernel"),       # K loop in parts
    (256, 512, 640, 1, "gemm_reduce_kernel"),        # peers
    (384, 1712, 1024, 7, "gemm_reduce_kernel"),      # peers and sixteen k-steps: in parts
    (384, 1712, 960, 7, "gemm_reduce_kernel"),
])
def test_gemm_plan_of_transposed_b_with_few_tiles(lib, M, N, K, P, kernel):
    """With transposed B gemm_ks_kernel only where it is not slower than gemm_reduce_kernel, and parts of at least
    eight k-steps."""
    p = _lib.gemm_plan(M, N, K, True, P, M, workspace_bytes=lib.kr_gemm_workspace_bytes(M, N, K))
    assert (p["kernel"], p["tile"]) == (kernel, 128)
    assert p["k_splits"] == 1 or K // 64 >= 8 * p["k_splits"]
    assert (p["k_splits"] > 1) == ((M, N, K) in ((256, 512, 4096), (384, 1712, 1024)))


@pytest.mark.parametrize("M,N,K,kernel", [(1000, 4096, 8192, "gemm_ks_kernel"), (1000, 4096, 8256, "gemm_reduce_kernel"), (1000, 4224, 4096, "gemm_reduce_kernel")])
def test_gemm_plan_of_transposed_b_without_a_workspace(lib, M, N, K, kernel):
    """One pass over 128x128 tiles: gemm_ks_kernel up to 256 tiles and K = 8192."""
    p = _lib.gemm_plan(M, N, K, True)
    assert (p["kernel"], p["tile"], p["k_splits"]) == (kernel, 128, 1)


@pytest.mark.parametrize("M,N,K,P", [(1000, 4096, 8192, 0), (1000, 4096, 8256, 0), (1000, 4224, 4096, 0), (990, 4224, 4096, 0), (1272, 2304, 12288, 1)])
def test_gemm_plan_of_transposed_b_and_ragged_rows_in_parts(lib, M, N, K, P):
    """Large tiles in parts where the model has them ahead, however few rows the last 128 x 128 tiles miss.  us, those / in parts: 71.3 / 73.0,
    82.7 / 72.3, 55.1 / 48.1 for the first three."""
    p = _lib.gemm_plan(M, N, K, True, P, M, workspace_bytes=lib.kr_gemm_workspace_bytes(M, N, K))
    assert (p["kernel"], p["tile"]) == ("gemm_dtl_split_kernel", 256) and p["tail_splits"] >= 3


@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (2, 1216, 16384), (16, 1024, 16384), (16, 1024, 8192), (32, 512, 8192), (64, 1032, 16384), (64, 8192, 3584)])
def test_few_rows_workspace_covers_either_layout(lib, M, N, K):
    """kr_gemm_workspace_bytes does not know the layout of B: it is enough for the parts the rule takes with either one,
    so that the plan does not change when the workspace is larger, and no larger than the larger of the two."""
    need = lib.kr_gemm_workspace_bytes(M, N, K)
    largest = 0
    for b_t in (False, True):
        plan = _lib.gemm_plan(M, N, K, b_t, workspace_bytes=need)
        assert plan["kernel"] == "gemm_skinny_kernel"
        assert plan == _lib.gemm_plan(M, N, K, b_t, workspace_bytes=1 << 40)
        if plan["k_splits"] > 1:
            largest = max(largest, plan["k_splits"] * M * N * 4)
    assert need == largest
    assert (need > 0) == (K >= 8192)


@pytest.mark.parametrize("M,N,K,split", [(331, 2440, 1352, True), (382, 3536, 1848, True), (720, 1280, 1464, True), (300, 2048, 1024, False), (256, 8192, 1024, False)])
def test_workspace_covers_the_plan_with_peers(lib, M, N, K, split):
    """kr_gemm_workspace_bytes knows neither the layout of B nor the peers: it is enough for the parts of either plan.
    With row-major B, peers and more than 16 k-steps few tiles share their K loop where one pass is enough without peers."""
    need = lib.kr_gemm_workspace_bytes(M, N, K)
    for b_t in (False, True):
        for P in (0, 1, 7):
            plan = _lib.gemm_plan(M, N, K, b_t, P, M, workspace_bytes=need)
            assert plan == _lib.gemm_plan(M, N, K, b_t, P, M, workspace_bytes=1 << 40)
            assert plan["k_splits"] == 1 or plan["k_splits"] * M * N * 4 <= need
            assert b_t or (plan["k_splits"] > 1) == (split and P > 0)


def test_split_fp32_argument_errors(lib):
    f = lib.kr_split_fp32
    assert f(FAKE, 16, 12, 12, 1, 0, FAKE, 36, None) == _lib.KR_ERR_NUMEL_MOD8
    assert f(None, 16, 16, 16, 1, 0, FAKE, 48, None) == _lib.KR_ERR_NULL_POINTER
    assert f(FAKE, 16, 16, 8, 1, 0, FAKE, 48, None) == _lib.KR_ERR_LAYOUT          # row stride shorter than the row
    assert f(FAKE, 16, 16, 16, 1, 0, FAKE, 40, None) == _lib.KR_ERR_LAYOUT         # side by side needs 3 * cols
    assert f(FAKE + 4, 16, 16, 16, 1, 0, FAKE, 48, None) == _lib.KR_ERR_ALIGNMENT
    assert f(FAKE, 16, 16, 18, 1, 0, FAKE, 48, None) == _lib.KR_ERR_ALIGNMENT      # fp32 rows not 16-byte aligned
    assert f(FAKE, 16, 16, 16, 1, 2, FAKE, 48, None) == _lib.KR_ERR_BAD_DIM
    assert f(None, 0, 16, 16, 1, 0, None, 48, None) == 0


def test_fp8_cast_argument_errors(lib):
    for f in (lib.kr_cast_fp8_to_bf16, lib.kr_cast_f32_to_fp8):
        assert f(FAKE, 24, FAKE, None) == _lib.KR_ERR_NUMEL_MOD8
        assert f(FAKE, -16, FAKE, None) == _lib.KR_ERR_BAD_DIM
        assert f(None, 32, FAKE, None) == _lib.KR_ERR_NULL_POINTER
        assert f(FAKE, 32, None, None) == _lib.KR_ERR_NULL_POINTER
        assert f(FAKE + 4, 32, FAKE, None) == _lib.KR_ERR_ALIGNMENT
        assert f(None, 0, None, None) == 0


def test_gather_matmul_argument_errors(lib):
    import ctypes
    f, direct = lib.kr_gather_matmul_bf16, lib.kr_gather_matmul_direct
    table = (ctypes.c_void_p * 8)(*[FAKE] * 8)
    base = dict(shards=table, W=8, rank=1, rows=512, A_out=FAKE, B=FAKE, ldb=256, N=4096, K=256, C=FAKE, stream=None)
    def call(**kw):
        args = dict(base); args.update(kw)
        return f(*args.values())
    assert direct(8, 512, 4096, 256) == 1
    for W, rows, N, K in ((0, 512, 4096, 256), (17, 512, 4096, 256), (8, 500, 4096, 256), (8, 0, 4096, 256), (8, 256, 1024, 256),
                          (8, 512, 4096, 64), (8, 512, 4100, 256), (8, 512, 4096, 260), (8, 1 << 40, 4096, 256), (8, 512, 4096, 1 << 22)):
        assert direct(W, rows, N, K) == 0
    assert call(W=17) == _lib.KR_ERR_WORLD_SIZE
    assert call(rank=8) == _lib.KR_ERR_STRIPE
    assert call(shards=None) == _lib.KR_ERR_NULL_POINTER
    assert call(A_out=None) == _lib.KR_ERR_NULL_POINTER
    assert call(A_out=FAKE + 8) == _lib.KR_ERR_ALIGNMENT
    assert call(rows=500) == _lib.KR_ERR_BAD_DIM
    assert call(C=None) == _lib.KR_ERR_NULL_POINTER
    assert call(ldb=128) == _lib.KR_ERR_LAYOUT
    assert call(shards=(ctypes.c_void_p * 8)(*[FAKE] * 7, FAKE + 2)) == _lib.KR_ERR_ALIGNMENT


def test_gemm_fp8_wide_argument_errors(lib):
    f = lib.kr_gemm_fp8_wide_ws
    base = dict(A=FAKE, lda=512, Bt=FAKE, ldb=512, M=100, N=272, K=496, out=FAKE, pivot=0, ws=None, bytes=0, stream=None)
    def call(**kw):
        args = dict(base); args.update(kw)
        return f(*args.values())
    assert call(N=264) == _lib.KR_ERR_BAD_DIM
    assert call(K=488) == _lib.KR_ERR_BAD_DIM
    assert call(K=0) == _lib.KR_ERR_BAD_DIM
    assert call(M=-1) == _lib.KR_ERR_BAD_DIM
    assert call(Bt=None) == _lib.KR_ERR_NULL_POINTER
    assert call(lda=480) == _lib.KR_ERR_LAYOUT
    assert call(ldb=1 << 23) == _lib.KR_ERR_LAYOUT       # 256 rows beyond the reach of 32-bit offsets
    assert call(lda=520) == _lib.KR_ERR_ALIGNMENT
    assert call(out=FAKE + 8) == _lib.KR_ERR_ALIGNMENT
    assert call(ws=FAKE + 8) == _lib.KR_ERR_ALIGNMENT
    assert call(M=0, A=None, Bt=None, out=None) == 0
    need = lib.kr_gemm_fp8_wide_workspace_bytes
    assert need(0, 256, 256) == 0 and need(4000, 6656, 4096) == 0
    for M, N, K in ((1, 16, 16), (8, 8192, 16384), (512, 4096, 4096), (2000, 2048, 8192), (1, 16, 1 << 20)):
        assert 0 <= need(M, N, K) <= 64 << 20


def test_gemm_fp8_argument_errors(lib):
    f = lib.kr_gemm_fp8
    ok = (FAKE, 512, FAKE, 512, 256, 256, 512, FAKE, 2, None)
    def call(**kw):
        names = ("A", "lda", "Bt", "ldb", "M", "N", "K", "out", "kind", "stream")
        args = dict(zip(names, ok)); args.update(kw)
        return f(*[args[n] for n in names])
    assert call(M=128) == _lib.KR_ERR_BAD_DIM            # whole 256 x 256 tiles only
    assert call(N=384) == _lib.KR_ERR_BAD_DIM
    assert call(K=192, lda=192, ldb=192) == _lib.KR_ERR_BAD_DIM
    assert call(kind=3) == _lib.KR_ERR_BAD_DIM
    assert call(M=-256) == _lib.KR_ERR_BAD_DIM
    assert call(A=None) == _lib.KR_ERR_NULL_POINTER
    assert call(out=None) == _lib.KR_ERR_NULL_POINTER
    assert call(lda=256) == _lib.KR_ERR_LAYOUT           # rows shorter than K
    assert call(ldb=520) == _lib.KR_ERR_ALIGNMENT        # row stride not a multiple of 16 bytes
    assert call(Bt=FAKE + 8) == _lib.KR_ERR_ALIGNMENT
    assert call(M=0, A=None, Bt=None, out=None) == 0     # nothing to do, nothing launched
    g = lib.kr_all_gather_matmul_fp8
    base = dict(A=FAKE, lda=512, A_local=FAKE, lda_local=512, Bt=FAKE, ldb=512, M=2048, N=256, K=512, W=8, rank=3, splits=1,
                progress=FAKE, limit=0, status=None, out=FAKE, kind=2, stream=None)
    def gcall(**kw):
        args = dict(base); args.update(kw)
        return g(*args.values())
    assert gcall(W=0) == _lib.KR_ERR_WORLD_SIZE
    assert gcall(rank=8) == _lib.KR_ERR_STRIPE
    assert gcall(splits=3) == _lib.KR_ERR_BAND           # 2048 rows in 24 chunks
    assert gcall(lda_local=520) == _lib.KR_ERR_ALIGNMENT
    assert gcall(lda_local=256) == _lib.KR_ERR_LAYOUT
    assert gcall(progress=FAKE + 2) == _lib.KR_ERR_ALIGNMENT
    assert gcall(M=1024, N=384) == _lib.KR_ERR_BAD_DIM   # the product's own shape rule


def test_gather_chunks_argument_errors(lib):
    f = lib.kr_gather_chunks
    table = (ctypes.c_void_p * 2)(FAKE, FAKE)
    assert f(table, 0, 1, 0, 16, FAKE, FAKE, None) == _lib.KR_ERR_WORLD_SIZE
    assert f(table, 2, 1, 2, 16, FAKE, FAKE, None) == _lib.KR_ERR_STRIPE
    assert f(table, 2, 1, 0, 24, FAKE, FAKE, None) == _lib.KR_ERR_BAD_DIM
    assert f(table, 2, 1, 0, 16, None, FAKE, None) == _lib.KR_ERR_NULL_POINTER
    assert f(table, 2, 1, 0, 16, FAKE + 8, FAKE, None) == _lib.KR_ERR_ALIGNMENT
    assert f(table, 2, 1, 0, 16, FAKE, FAKE + 2, None) == _lib.KR_ERR_ALIGNMENT
    assert f(None, 2, 1, 0, 0, None, None, None) == _lib.KR_ERR_NULL_POINTER     # empty chunks still have flags


def test_probe_argument_errors(lib):
    assert lib.kr_probe_read(FAKE, 24, None, None) == _lib.KR_ERR_NUMEL_MOD8
    assert lib.kr_probe_read(None, 32, None, None) == _lib.KR_ERR_NULL_POINTER
    assert lib.kr_probe_read(FAKE + 4, 32, None, None) == _lib.KR_ERR_ALIGNMENT
    assert lib.kr_probe_read(None, 0, None, None) == 0
    assert lib.kr_probe_copy(FAKE, None, 32, None) == _lib.KR_ERR_NULL_POINTER
    assert lib.kr_probe_copy(FAKE, FAKE + 8, 32, None) == _lib.KR_ERR_ALIGNMENT
    assert lib.kr_probe_copy(None, None, 0, None) == 0


def test_striped_share_numel(lib):
    f = lib.kr_striped_share_numel
    numel, W, block = 8 * 37, 4, 16
    shares = [f(numel, W, block, r) for r in range(W)]
    assert sum(shares) == numel
    from oracle import oracle as orc
    assert shares == [orc.striped_indices(numel, W, block, r).numel() for r in range(W)]
    assert f(numel, W, 12, 0) == _lib.KR_ERR_STRIPE
    assert f(numel, W, 16, 4) == _lib.KR_ERR_STRIPE
    assert f(numel + 4, W, 16, 0) == _lib.KR_ERR_NUMEL_MOD8


def test_rotated_argument_errors(lib):
    f = lib.kr_reduce_rotated_bf16
    assert f(FAKE, 4, 3, 16, 4, 1, FAKE, None) == _lib.KR_ERR_STRIPE
    assert f(FAKE, 4, 3, 12, 0, 1, FAKE, None) == _lib.KR_ERR_NUMEL_MOD8
    assert f(None, 4, 3, 16, 0, 1, FAKE, None) == _lib.KR_ERR_NULL_POINTER


def test_check_maps_codes_to_reference_exceptions():
    with pytest.raises(AssertionError, match="128-bit"):
        _lib.check(_lib.KR_ERR_NUMEL_MOD8, "x")
    with pytest.raises(ValueError):
        _lib.check(_lib.KR_ERR_LAYOUT, "x")
    with pytest.raises(_lib.KrakenAmdError):
        _lib.check(1, "x")
    _lib.check(0, "x")


def test_public_names_match_reference_layout():
    # kraken/comm/__init__.py:12-17, kraken/fused/__init__.py:17-27
    assert set(comm.__all__) == {"_copy_engine_all_gather_w_progress", "all_gather_w_progress",
                                 "one_shot_all_reduce", "two_shot_all_reduce"}
    assert set(fused.__all__) == {
        "all_gather_matmul", "gemm_one_shot_all_reduce_fused", "gemm_reduce_scatter",
        "gemm_reduce_scatter_ce_persistent", "one_shot_all_reduce_bias",
        "one_shot_all_reduce_bias_rms_norm", "rms_norm", "two_shot_all_reduce_bias",
        "two_shot_all_reduce_bias_rms_norm",
    }
    assert kraken_amd.__all__ == ["_lib", "_logging", "comm", "fused"]
    # kraken/_logging/__init__.py:1-4 (the PTX dump helper has no counterpart: nothing is compiled at run time)
    from kraken_amd import _logging
    assert set(_logging.__all__) == {"benchmark_with_event", "benchmark_with_profiler", "plot_experiment_comparison"}


def test_plot_experiment_comparison_writes_the_chart(tmp_path):
    from kraken_amd._logging import plot_experiment_comparison
    out = tmp_path / "sweep.png"
    plot_experiment_comparison(["(1, 5k)", "(2, 5k)", "(4, 5k)"], ["hip", "torch"], [[6.3, 14.6], [6.3, 13.4], [6.4, 13.6]],
                               str(out))
    assert out.stat().st_size > 1000 and out.read_bytes()[:4] == b"\x89PNG"
    with pytest.raises(AssertionError):
        plot_experiment_comparison(["a"], ["x", "y"], [[1.0]], str(out))      # a row per size, a value per experiment


def test_wrappers_assert_like_the_reference_and_refuse_host_tensors():
    s32 = torch.zeros(8, 4, 64, dtype=torch.float32)
    with pytest.raises(AssertionError, match="bfloat16"):
        comm.one_shot_all_reduce(s32)                       # one_shot_all_reduce.py:79
    with pytest.raises(AssertionError, match="128-bit"):
        comm.one_shot_all_reduce(torch.zeros(8, 3, 4, dtype=BF16))   # :80
    with pytest.raises(AssertionError):
        comm.two_shot_all_reduce(torch.zeros(3, 8, 64, dtype=BF16), BLOCK_SIZE=2048)  # BLOCK % W
    s = torch.zeros(8, 4, 64, dtype=BF16)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        comm.one_shot_all_reduce(s)
    y = torch.empty(4, 64, dtype=BF16)
    w = torch.ones(64, dtype=BF16)
    with pytest.raises(AssertionError):
        fused.one_shot_all_reduce_bias_rms_norm(s, None, None, torch.ones(32, dtype=BF16), y)  # w.shape == (D,)
    with pytest.raises(AssertionError):
        fused.two_shot_all_reduce_bias_rms_norm(torch.zeros(8, 1, 72, dtype=BF16), None, None,
                                                torch.ones(72, dtype=BF16), torch.empty(1, 72, dtype=BF16))
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        fused.one_shot_all_reduce_bias_rms_norm(s, None, None, w, y)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        fused.rms_norm(torch.zeros(4, 64, dtype=BF16), w)
    a, b = torch.zeros(64, 32, dtype=BF16), torch.zeros(32, 64, dtype=BF16)
    with pytest.raises(AssertionError, match="Inner dimensions"):
        fused.gemm_one_shot_all_reduce_fused(a, torch.zeros(16, 64, dtype=BF16))
    with pytest.raises(AssertionError, match="divisible by world_size"):
        fused.gemm_reduce_scatter(torch.zeros(66, 32, dtype=BF16), b, world_size=4)
    with pytest.raises(ValueError, match="b.T must be contiguous"):
        fused.all_gather_matmul(torch.zeros(4, 16, 32, dtype=BF16), b)   # all_gather_matmul.py:158-160
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        fused.gemm_one_shot_all_reduce_fused(a, b)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "libkraken_amd.so")
    with pytest.raises(RuntimeError, match="kraken_amd.build"):
        _lib.load()


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one rank on one GPU: any other --gpus value ends with a message and exit status 2
    before anything touches a device."""
    import subprocess
    import sys
    r = subprocess.run([sys.executable, str(Path(__file__).resolve().parents[1] / "bench.py"), "--gpus", "2"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2
    assert "--gpus 2 is not supported" in r.stderr and r.stdout == ""


def test_shards_in_each_others_places_take_no_single_launch(monkeypatch):
    """The workgroups of kr_gather_chunks run in no order: it is not launched where a shard lies where another one's copy goes."""
    from kraken_amd.comm import copy_engine_all_gather as ag
    from kraken_amd.comm._common import PeerBuffers

    launched = []

    class Lib:
        def kr_gather_chunks(self, *args):
            launched.append(args)
            return 0

    monkeypatch.setattr(_lib, "load", Lib)
    W, m, K = 4, 6, 64
    out, progress, own = torch.zeros(W * m, K, dtype=torch.bfloat16), torch.zeros(W, dtype=torch.int32), torch.zeros(W, m, K, dtype=torch.bfloat16)
    for first, taken in ((own[0], True), (out[:m], True), (out[m:2 * m], False), (out[1:m + 1], False), (out[(W - 1) * m:], False)):
        launched.clear()
        assert ag.gather_chunks(out, PeerBuffers([first, *own[1:]]), progress, 1, 0, 0) == taken == bool(launched)


def test_tangents_keep_gathers_and_sends_from_the_kernels():
    """A forward-mode tangent is handed on, or cleared, by torch's copies only, whether gradients are enabled or not."""
    import torch.autograd.forward_ad as fw

    from kraken_amd.comm import copy_engine_all_gather as ag
    from kraken_amd.comm._common import PeerBuffers
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import _sends_direct

    W, m, K = 2, 4, 16
    out, a, b = torch.zeros(W * m, K, dtype=BF16), torch.zeros(W * m, K, dtype=BF16), torch.zeros(K, K, dtype=BF16)
    shards, sent = [torch.zeros(m, K, dtype=BF16) for _ in range(W)], torch.zeros(W, m, K, dtype=BF16)
    with fw.dual_level():
        assert not ag.followed(out, PeerBuffers(shards)) and _sends_direct(sent, a, b, W, m, K)
        for grad in (torch.no_grad, torch.enable_grad):
            with grad():
                dual = fw.make_dual(shards[1], torch.ones_like(shards[1]))
                assert ag.followed(out, PeerBuffers([shards[0], dual]))
                assert ag.followed(fw.make_dual(out, torch.ones_like(out)), PeerBuffers(shards))
                assert not _sends_direct(fw.make_dual(sent, torch.ones_like(sent)), a, b, W, m, K)
    with torch.no_grad():
        assert ag._takes_copies(out.requires_grad_())
    assert not ag._takes_copies(out)


def test_fp8_wide_empty_products_check_the_operand_that_has_elements(lib):
    f = lib.kr_gemm_fp8_wide_ws
    for off, M, N, want in ((8, 0, 64, 0), (8, 16, 0, _lib.KR_ERR_ALIGNMENT), (0, 16, 0, 0), (0, 0, 64, 0)):
        assert f(FAKE + off, 64, FAKE, 64, M, N, 64, FAKE, 0, None, 0, None) == want
        assert f(FAKE, 64, FAKE + off, 64, N, M, 64, FAKE, 0, None, 0, None) == want


@pytest.mark.parametrize("M,N,K,b_t,P", [(736, 6416, 5680, True, 7), (3224, 1248, 7136, False, 3), (3144, 1392, 15472, True, 0), (504, 6656, 8208, False, 1),
                                         (944, 4240, 13360, True, 1), (1100, 1856, 13616, True, 0)])
def test_gemm_plan_few_tiles_and_a_ragged_k_in_parts(lib, M, N, K, b_t, P):
    """256-row tiles in parts whether or not the last k-step is full, and the workspace for them."""
    need = lib.kr_gemm_workspace_bytes(M, N, K)
    p = _lib.gemm_plan(M, N, K, b_t, P, M // (P + 1) if P else M, False, P > 0, workspace_bytes=need)
    assert p["kernel"] == "gemm_dtl_split_kernel" and p["ragged"] and not p["peers_on_mfma"]
    assert p["tail_tiles"] * p["tail_splits"] * 1024 * p["tile_n"] <= need <= 64 << 20


@pytest.mark.parametrize("M,N,K", [(5486, 3456, 9984), (4360, 4096, 8200), (2312, 8000, 4096), (6080, 4096, 8192), (5632, 4224, 11264), (4104, 4096, 3072), (4864, 4096, 3648)])
def test_gemm_plan_ragged_shapes_share_their_last_round(lib, M, N, K):
    need, tiles = lib.kr_gemm_workspace_bytes(M, N, K), -(-M // 256) * -(-N // 256)
    for b_t in (False, True):
        p = _lib.gemm_plan(M, N, K, b_t, 7, M // 8, False, True, workspace_bytes=need)
        assert p["tile"] == 256 and p["tail_tiles"] == tiles % 256 and p["tail_splits"] > 1 and 0 < need <= 64 << 20
        assert _lib.gemm_plan(M, N, K, b_t, 7, M // 8, False, True)["tail_tiles"] == 0       # no workspace
