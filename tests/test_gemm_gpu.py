"""GPU parity of the bf16 MFMA GEMM with fused reduce(+bias) epilogue against the CPU oracle.
Gate: rtol = atol = 2e-2 for bf16 outputs vs the fp32-accumulated oracle."""
import ctypes
import importlib
import os

import pytest
import torch

from kraken_amd import _lib, comm, fused
from oracle import oracle as orc

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
TOL = dict(rtol=2e-2, atol=2e-2)


@pytest.fixture(params=["128", "128-staged", "256", "256-epilogue"])
def tile(request, monkeypatch):
    """Force each GEMM kernel in turn: with 128x128 tiles the deep-ring kernel (a K below 64 falls
    back to the register-staged one) and the register-staged one; the
    LDS-DMA kernel with 256x256 tiles (shapes it cannot take fall back to the others), with the
    peers' partial sums of whole-band tiles added on the matrix cores (default) or in the
    epilogue."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", request.param[:3])
    if request.param[:3] == "128":
        monkeypatch.setenv("KRAKEN_AMD_GEMM_KS", "0" if request.param == "128-staged" else "1")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_PEERS", "epilogue" if request.param.endswith("epilogue") else "mfma")
    return request.param


def mk(M, N, K, P, b_t=False, seed=0):
    a = orc.randn_bf16((M, K), 42 + seed)
    if b_t:
        b = orc.randn_bf16((N, K), 43 + seed, 0.05).T          # b.T contiguous
    else:
        b = orc.randn_bf16((K, N), 43 + seed, 0.05)
    peers = torch.stack([orc.randn_bf16((M, N), 100 + j) for j in range(P)]) if P else None
    return a, b, peers


def test_rank_specific_known_answer(dev, tile):
    # test/test_gemm_allreduce.py:92-117 (M=N=K=32, W=4): every element K*(1+2+3+4), at 1e-5
    M = N = K = 32
    a = torch.ones(M, K, dtype=BF16)
    b = torch.ones(K, N, dtype=BF16)
    peers = torch.stack([torch.full((M, N), float((r + 1) * K), dtype=BF16) for r in range(1, 4)])
    out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev), peers=peers.to(dev))
    assert out.dtype == torch.float32 and out.shape == (M, N)
    torch.testing.assert_close(out.cpu(), torch.full((M, N), float(K * 10)), rtol=1e-5, atol=1e-5)
    # same with fp32 operands, as the reference test passes them
    out32 = fused.gemm_one_shot_all_reduce_fused(a.float().to(dev), b.float().to(dev), peers=peers.to(dev))
    torch.testing.assert_close(out32.cpu(), torch.full((M, N), float(K * 10)), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("shape", [(512, 256, 128), (256, 256, 256), (128, 128, 64), (384, 640, 192),
                                   (100, 72, 40), (8, 8, 8), (1000, 264, 520)])
@pytest.mark.parametrize("b_t", [False, True])
def test_gemm_all_reduce_shapes(dev, tile, shape, b_t):
    M, N, K = shape
    a, b, peers = mk(M, N, K, 3, b_t)
    bias = orc.randn_bf16((N,), 42, 0.02)
    want = orc.gemm_all_reduce(a, b, peers, bias)
    out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev), peers=peers.to(dev), bias=bias.to(dev))
    torch.testing.assert_close(out.cpu(), want, rtol=1e-3, atol=1e-3)      # fp32 out: tight
    outb = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev), peers=peers.to(dev), bias=bias.to(dev),
                                                out_dtype=BF16)
    torch.testing.assert_close(outb.cpu(), want.to(BF16), **TOL)
    plain = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev))
    torch.testing.assert_close(plain.cpu(), orc.gemm_all_reduce(a, b), rtol=1e-3, atol=1e-3)


def test_all_gather_matmul_224_column_tiles(dev, monkeypatch):
    """A plain product with transposed-contiguous B whose 256-column tiles leave a partial round of
    compute units takes 256 x 224 tiles (4096 x 3584: 224 tiles against 256): the whole matrix against
    the oracle, and the same bits as the 256-column form (every element sums the same products in the
    same order)."""
    for name in ("TILE", "MFMA", "N224", "PEERS"):   # the rule under test, whatever the caller's environment forces
        monkeypatch.delenv("KRAKEN_AMD_GEMM_" + name, raising=False)
    W, m, K, N = 8, 512, 320, 3584
    assert _lib.gemm_plan(W * m, N, K, True)["kernel"] == "gemm_dtl16n7_kernel"
    stack = orc.make_stack(W, (m, K), seed0=21)
    bT = orc.randn_bf16((N, K), 22, 0.05)
    a_out, c = fused.all_gather_matmul(stack.to(dev), bT.to(dev).T, rank=5)
    _, want = orc.all_gather_matmul(stack, bT.T)
    torch.testing.assert_close(c.cpu().float(), want.float(), **TOL)
    assert torch.equal(a_out.cpu(), stack.reshape(W * m, K))
    # the overlapped form takes the same tiles (a tile waits for its rows' flags before its first load)
    a_g, c_g = fused.all_gather_matmul(stack.to(dev), bT.to(dev).T, rank=5, gather=True, splits_per_rank=2)
    assert torch.equal(c, c_g) and torch.equal(a_g.cpu(), stack.reshape(W * m, K))
    monkeypatch.setenv("KRAKEN_AMD_GEMM_N224", "0")
    assert _lib.gemm_plan(W * m, N, K, True)["kernel"] == "gemm_dtl16_kernel"
    _, c256 = fused.all_gather_matmul(stack.to(dev), bT.to(dev).T, rank=5)
    assert torch.equal(c, c256)
    # forced on where the rule would not pick it (64 tiles of 224 columns: one partial round either way), odd k-step count
    monkeypatch.setenv("KRAKEN_AMD_GEMM_N224", "1")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    W, m, K, N = 4, 256, 192, 896
    stack = orc.make_stack(W, (m, K), seed0=23)
    bT = orc.randn_bf16((N, K), 24, 0.05)
    assert _lib.gemm_plan(W * m, N, K, True)["kernel"] == "gemm_dtl16n7_kernel"
    _, c = fused.all_gather_matmul(stack.to(dev), bT.to(dev).T)
    _, want = orc.all_gather_matmul(stack, bT.T)
    torch.testing.assert_close(c.cpu().float(), want.float(), **TOL)


def test_fp8_conversions(dev):
    """kr_cast_fp8_to_bf16 on all 256 codes and kr_cast_f32_to_fp8 on random and boundary values,
    against torch's CPU conversions (nearest even); from magnitude 448 on the result saturates to
    448 where torch gives NaN (from 464 on)."""
    lib = _lib.load()
    stream = torch.cuda.current_stream(dev).cuda_stream
    fp8 = torch.float8_e4m3fn
    codes = torch.arange(256, dtype=torch.uint8).repeat(4)
    out = torch.empty(codes.numel(), dtype=BF16, device=dev)
    assert lib.kr_cast_fp8_to_bf16(codes.to(dev).data_ptr(), codes.numel(), out.data_ptr(), stream) == 0
    want = codes.view(fp8).to(BF16)
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(out.cpu()), nan) and torch.equal(out.cpu()[~nan].view(torch.int16), want[~nan].view(torch.int16))
    g = torch.Generator().manual_seed(3)
    x = torch.cat([torch.randn(1 << 16, generator=g) * s_ for s_ in (1e-3, 0.02, 1.0, 30.0, 300.0)])
    edge = torch.tensor([0.0, -0.0, 2.0 ** -9, 2.0 ** -10, 1.5 * 2.0 ** -9, 2.5 * 2.0 ** -9, 2.0 ** -6, 0.9375 * 2.0 ** -6,
                         447.9, 448.0, 463.9, 464.0, 1e9, -1e9, float("inf"), -float("inf")])
    x = torch.cat([x, edge, torch.zeros(-(x.numel() + edge.numel()) % 16)])
    y = torch.empty(x.numel(), dtype=torch.uint8, device=dev)
    assert lib.kr_cast_f32_to_fp8(x.to(dev).data_ptr(), x.numel(), y.data_ptr(), stream) == 0
    got = y.cpu()
    small = x.abs() < 448
    assert torch.equal(got[small], x[small].to(fp8).view(torch.uint8))
    assert torch.equal(got[~small] & 0x7f, torch.full_like(got[~small], 0x7e))           # saturated, sign kept
    assert torch.equal(got[~small] >> 7, (x[~small] < 0).to(torch.uint8))
    z = torch.full((16,), float("nan"))
    assert lib.kr_cast_f32_to_fp8(z.to(dev).data_ptr(), 16, y.data_ptr(), stream) == 0
    assert torch.isnan(y.cpu()[:16].view(fp8).float()).all()


def test_all_gather_matmul_fp8(dev):
    """The fp8 branch (kraken/fused/all_gather_matmul.py:53,121,213): fp8 shards and b, fp8 result.
    With small integers and halves every fp32 sum is exact whatever its order, so the result equals
    the oracle bit for bit, saturated elements included; with random operands it is within one fp8
    step of the oracle (the orders of the fp32 sums differ) and mostly equal."""
    fp8 = torch.float8_e4m3fn
    W, m, K, N = 8, 64, 512, 384
    g = torch.Generator().manual_seed(11)
    a = torch.randint(-2, 3, (W, m, K), generator=g).float().to(fp8)
    bT = (torch.randint(-3, 4, (N, K), generator=g).float() * 0.5).to(fp8)
    a_out, c = fused.all_gather_matmul(a.to(dev), bT.to(dev).T, rank=3)
    a_full, want = orc.all_gather_matmul_fp8(a, bT.T)
    assert c.dtype == fp8 and a_out.dtype == fp8
    assert torch.equal(a_out.cpu().view(torch.uint8), a_full.view(torch.uint8))
    assert torch.equal(c.cpu().view(torch.uint8), want.view(torch.uint8))
    # a shape the 256x256 kernel takes, random operands, one fp8 step of slack
    W, m, K, N = 8, 512, 1024, 4096
    a = (torch.randn(W, m, K, generator=g)).to(fp8)
    bT = (torch.randn(N, K, generator=g) * 0.05).to(fp8)
    _, c = fused.all_gather_matmul(a.to(dev), bT.to(dev).T)
    _, want = orc.all_gather_matmul_fp8(a, bT.T)
    got, ref = c.cpu().float(), want.float()
    assert (got == ref).float().mean() > 0.99
    step = torch.maximum(ref.abs(), torch.tensor(2.0 ** -6)) * 2.0 ** -3          # spacing of e4m3 at that magnitude
    assert ((got - ref).abs() <= step).all()


@pytest.mark.parametrize("K", [128, 256, 384, 1024])
def test_fp8_kernel_exact_sums(dev, K):
    """kr_gemm_fp8 (fp8 operands on the fp8 matrix-core instruction): with small integers and halves every
    fp32 sum is exact whatever its order, so all three result types equal the oracle bit for bit -- the fp8
    result with its saturated elements, through the wrapper and straight through the C ABI; one, two, an odd
    number and many k-steps."""
    fp8 = torch.float8_e4m3fn
    W, m, N = 8, 64, 768
    g = torch.Generator().manual_seed(31 + K)
    a = torch.randint(-2, 3, (W, m, K), generator=g).float().to(fp8)
    bT = (torch.randint(-3, 4, (N, K), generator=g).float() * 0.5).to(fp8)
    a[0], a[1], bT[:64] = 4.0, -4.0, 1.5            # sums of +-6K: beyond the largest fp8 value on both sides
    a_full, want = orc.all_gather_matmul_fp8(a, bT.T)
    exact = a.reshape(W * m, K).float() @ bT.float().T
    assert (exact > 448).any() and (exact < -448).any() and (exact.abs() < 448).any()      # the case has saturating and ordinary sums
    a_out, c = fused.all_gather_matmul(a.to(dev), bT.to(dev).T, rank=2)
    assert c.dtype == fp8 and torch.equal(a_out.cpu().view(torch.uint8), a_full.view(torch.uint8))
    assert torch.equal(c.cpu().view(torch.uint8), want.view(torch.uint8))
    lib = _lib.load()
    stream = torch.cuda.current_stream(dev).cuda_stream
    ad, bd = a.reshape(W * m, K).to(dev), bT.to(dev)
    for kind, dtype in ((1, torch.float32), (0, BF16)):
        out = torch.full((W * m, N), 7, dtype=dtype, device=dev)
        assert lib.kr_gemm_fp8(ad.data_ptr(), K, bd.data_ptr(), K, W * m, N, K, out.data_ptr(), kind, stream) == 0
        assert torch.equal(out.cpu(), exact.to(dtype))


def test_fp8_kernel_random_operands_and_nan(dev):
    """Random operands: within one fp8 step of the oracle and of the widening path (the orders of the fp32
    sums differ), mostly equal; the fp32 result against a double-precision product; row strides larger than
    K; a NaN operand element makes its row of the result NaN and nothing else."""
    fp8 = torch.float8_e4m3fn
    W, m, K, N = 8, 128, 2048, 1280
    g = torch.Generator().manual_seed(41)
    a = torch.randn(W, m, K, generator=g).to(fp8)
    bT = (torch.randn(N, K, generator=g) * 0.05).to(fp8)
    _, c = fused.all_gather_matmul(a.to(dev), bT.to(dev).T)
    _, c_wide = fused.all_gather_matmul(a.to(dev), bT.to(dev).T, fp8_kernel=False)
    _, want = orc.all_gather_matmul_fp8(a, bT.T)
    ref = want.float()
    step = torch.maximum(ref.abs(), torch.tensor(2.0 ** -6)) * 2.0 ** -3          # spacing of e4m3 at that magnitude
    for got in (c.cpu().float(), c_wide.cpu().float()):
        assert (got == ref).float().mean() > 0.99
        assert ((got - ref).abs() <= step).all()
    lib = _lib.load()
    stream = torch.cuda.current_stream(dev).cuda_stream
    M = W * m
    a_pad = torch.zeros(M, K + 64, dtype=torch.uint8).view(fp8)
    a_pad[:, :K] = a.reshape(M, K)
    b_pad = torch.zeros(N, K + 16, dtype=torch.uint8).view(fp8)
    b_pad[:, :K] = bT
    ad, bd = a_pad.to(dev), b_pad.to(dev)
    out = torch.empty(M, N, dtype=torch.float32, device=dev)
    assert lib.kr_gemm_fp8(ad.data_ptr(), K + 64, bd.data_ptr(), K + 16, M, N, K, out.data_ptr(), 1, stream) == 0
    exact = (a.reshape(M, K).double() @ bT.double().T)
    torch.testing.assert_close(out.cpu().double(), exact, rtol=1e-5, atol=1e-3)      # fp32 sums of 2048 products of size 0.05
    a_nan = a.reshape(M, K).clone()
    a_nan.view(torch.uint8)[300, 77] = 0x7f
    c = torch.empty(M, N, dtype=fp8, device=dev)
    assert lib.kr_gemm_fp8(a_nan.to(dev).data_ptr(), K, bT.to(dev).data_ptr(), K, M, N, K, c.data_ptr(), 2, stream) == 0
    nan = torch.isnan(c.cpu().float())
    assert nan[300].all() and not nan[:300].any() and not nan[301:].any()


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("as_list", [False, True])
def test_all_gather_matmul_fp8_overlapped(dev, splits, as_list):
    """gather=True with fp8 shards (the reference's overlap, all_gather_matmul.py:308-323, on its fp8 branch):
    the chunks are copied on the side stream and flagged while the fp8 kernel's tiles wait for them; the
    gathered matrix is the shards bit for bit, every flag ends at 1, and the product has the bits of the
    gather=False call (same kernel, same sums).  Also a shape the fp8 kernel does not take (the widening
    path behind the finished gather)."""
    from kraken_amd import _waits
    fp8 = torch.float8_e4m3fn
    W, m, K, N = 8, 256, 1024, 768
    g = torch.Generator().manual_seed(51)
    a = torch.randn(W, m, K, generator=g).to(fp8)
    bT = (torch.randn(N, K, generator=g) * 0.05).to(fp8)
    ad, bd = a.to(dev), bT.to(dev)
    _, want = fused.all_gather_matmul(ad, bd.T, rank=5)
    shards = [ad[r].clone() for r in range(W)] if as_list else ad
    progress = torch.zeros(W * splits, dtype=torch.int32, device=dev)
    a_out, c = fused.all_gather_matmul(shards, bd.T, None, progress, rank=5, splits_per_rank=splits, gather=True)
    torch.cuda.synchronize()
    _waits.check(block=True)
    assert a_out.dtype == fp8 and torch.equal(a_out.cpu().view(torch.uint8), a.reshape(W * m, K).view(torch.uint8))
    assert (progress.cpu() == 1).all()
    assert torch.equal(c.cpu().view(torch.uint8), want.cpu().view(torch.uint8))
    _, ref = orc.all_gather_matmul_fp8(a, bT.T)
    assert (c.cpu().float() == ref.float()).float().mean() > 0.99
    # 8 x 48 rows: not a multiple of 256
    a2, b2 = a[:, :48].contiguous(), bT[:400]
    a_out, c = fused.all_gather_matmul(a2.to(dev), b2.to(dev).T, rank=1, gather=True)
    _, ref = orc.all_gather_matmul_fp8(a2, b2.T)
    assert torch.equal(a_out.cpu().view(torch.uint8), a2.reshape(-1, K).view(torch.uint8))
    assert (c.cpu().float() == ref.float()).float().mean() > 0.99


def test_split_fp32_is_one_pass_and_bit_exact(dev):
    """kr_split_fp32 writes the hi / lo blocks of an fp32 operand in the three layouts the GEMM
    wrappers use, bit for bit what elementwise torch ops give (hi = bf16(x), lo = bf16(x - hi)),
    also for a row stride larger than the row."""
    from kraken_amd.fused import _gemm
    g = torch.Generator().manual_seed(7)
    for (M, K, N) in [(64, 128, 72), (300, 264, 136), (8, 8, 8)]:
        a = torch.randn(M, K + 8, generator=g).to(dev)[:, :K]            # row stride K + 8
        b = torch.randn(K, N, generator=g).to(dev)
        bt = torch.randn(N, K, generator=g).to(dev).T                     # transposed-contiguous [K, N]
        for (x, y) in ((a, b), (a, bt)):
            a3, b3 = _gemm.split_fp32(x, y)
            x_hi = x.to(BF16); x_lo = (x - x_hi.float()).to(BF16)
            y_hi = y.to(BF16); y_lo = (y - y_hi.float()).to(BF16)
            assert torch.equal(a3, torch.cat([x_hi, x_hi, x_lo], dim=1))
            assert torch.equal(b3, torch.cat([y_hi, y_lo, y_hi], dim=0))
            assert b3.T.is_contiguous() == (y is bt)                      # the operand's layout is kept
            # the 3K-long bf16 product is a @ b to ~16 mantissa bits
            ref = x.double() @ y.double()
            got = (a3.double() @ b3.double())
            assert (got - ref).abs().max() <= 2e-4 * ref.abs().max() + 1e-6
    # sizes the kernel does not take fall back to elementwise ops with the same result
    a = torch.randn(16, 12, generator=g).to(dev); b = torch.randn(12, 20, generator=g).to(dev)
    a3, b3 = _gemm.split_fp32(a, b)
    assert a3.shape == (16, 36) and b3.shape == (36, 20)
    assert torch.equal(a3[:, :12], a.to(BF16)) and torch.equal(b3[12:24], (b - b.to(BF16).float()).to(BF16))


def test_fp32_operands_reference_shapes(dev, tile):
    # test/test_gemm_allreduce.py:51-89: fp32 N(0,1) operands, (512,256,128) and (256,256,256), tol 1e-1
    for (M, N, K) in [(512, 256, 128), (256, 256, 256)]:
        g = torch.Generator().manual_seed(42)
        a = torch.randn(M, K, generator=g)
        b = torch.randn(K, N, generator=g)
        out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev))
        torch.testing.assert_close(out.cpu(), a @ b, rtol=1e-1, atol=1e-1)
        torch.testing.assert_close(out.cpu(), a @ b, rtol=2e-3, atol=2e-3)   # the split keeps ~16 bits


@pytest.mark.parametrize("rank", [0, 2, 3])
@pytest.mark.parametrize("b_t", [False, True])
def test_gemm_reduce_scatter(dev, tile, rank, b_t):
    M, N, K, W = 512, 256, 128, 4        # test/test_gemm_reduce_scatter.py:61-74
    a, b, _ = mk(M, N, K, 0, b_t)
    peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)])
    want, c_want = orc.gemm_reduce_scatter(a, b, peers, rank, W)
    c_scratch = torch.full((M, N), float("nan"), dtype=BF16, device=dev)
    out = fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=peers.to(dev), rank=rank, c_scratch=c_scratch)
    assert out.shape == (M // W, N) and out.dtype == BF16
    torch.testing.assert_close(out.cpu(), want, **TOL)
    rows = torch.ones(M, dtype=torch.bool)
    rows[rank * M // W:(rank + 1) * M // W] = False
    torch.testing.assert_close(c_scratch.cpu()[rows], c_want[rows], **TOL)
    assert torch.isnan(c_scratch.cpu()[~rows].float()).all()    # own band never makes the round trip


def test_gemm_reduce_scatter_rank_specific(dev, tile):
    # test/test_gemm_reduce_scatter.py:76-91
    M, N, K, W = 512, 256, 128, 4
    for rank in range(W):
        a = torch.full((M, K), float(rank + 1), dtype=BF16)
        b = torch.ones(K, N, dtype=BF16)
        others = [r for r in range(W) if r != rank]
        peers = torch.stack([torch.full((M // W, N), float((r + 1) * K), dtype=BF16) for r in others])
        out = fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=peers.to(dev), rank=rank)
        assert torch.equal(out.cpu().float(), torch.full((M // W, N), float(K * 10)))


@pytest.mark.parametrize("rank", [0, 3])
def test_all_gather_matmul(dev, tile, rank):
    W, m, K, N = 4, 128, 256, 384
    stack = orc.make_stack(W, (m, K))
    bT = orc.randn_bf16((N, K), 43, 0.05)
    sd = stack.to(dev)
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    ag, c = fused.all_gather_matmul(sd, bT.to(dev).T, progress=progress, rank=rank)
    a_want, c_want = orc.all_gather_matmul(stack, bT.T)
    assert torch.equal(ag.cpu(), a_want)                      # test/test_allgather_matmul.py:75: exact
    assert ag.data_ptr() == sd.data_ptr()                     # zero-copy view
    assert (progress != 0).all()                              # test/test_allgather.py:73
    torch.testing.assert_close(c.cpu(), c_want, **TOL)
    a_out = torch.empty(W * m, K, dtype=BF16, device=dev)
    ag2, c2 = fused.all_gather_matmul(sd, bT.to(dev).T, a_out=a_out, rank=rank)
    assert ag2 is a_out and torch.equal(a_out.cpu(), a_want) and torch.equal(c2, c)


@pytest.mark.parametrize("rank,splits", [(0, 1), (2, 2), (3, 4)])
@pytest.mark.parametrize("as_list", [False, True])
def test_all_gather_matmul_overlapped_with_the_copies(dev, tile, rank, splits, as_list):
    """The reference's overlap: chunk copies with arrival flags on a side stream, tiles that
    wait for their chunk (kraken/fused/all_gather_matmul.py:95-110); local shard read in place."""
    W, m, K, N = 4, 256, 320, 384
    stack = orc.make_stack(W, (m, K), seed0=7)
    bT = orc.randn_bf16((N, K), 43, 0.05)
    a_want, c_want = orc.all_gather_matmul(stack, bT.T)
    shards = [stack[r].to(dev) for r in range(W)] if as_list else stack.to(dev)
    progress = torch.full((W * splits,), 7, dtype=torch.int32, device=dev)       # stale values: must be reset
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    a_out = torch.full((W * m, K), float("nan"), dtype=BF16, device=dev)
    ag, c = fused.all_gather_matmul(shards, bT.to(dev).T, a_out=a_out, progress=progress, rank=rank,
                                    splits_per_rank=splits, gather=True, status=status)
    torch.cuda.synchronize()
    assert ag is a_out and torch.equal(ag.cpu(), a_want)          # test/test_allgather_matmul.py:75: exact
    assert (progress == 1).all()                                  # test/test_allgather.py:73
    assert status.item() == 0
    torch.testing.assert_close(c.cpu(), c_want, **TOL)
    # same bits as the GEMM on the already gathered matrix
    _, c_plain = fused.all_gather_matmul(stack.to(dev), bT.to(dev).T, rank=rank)
    assert torch.equal(c, c_plain)


@pytest.mark.parametrize("how", ["copy_engine", "misaligned"])
@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
def test_all_gather_matmul_on_the_side_stream(dev, tile, how, dtype):
    """The form with copies and flags on a side stream (asked for, or shards that one launch cannot take): the
    results of the form that gathers in front of the product, every flag at 1, no wait run out."""
    from kraken_amd import _waits
    W, m, K, N, rank, splits = 4, 256, 384, 512, 2, 2
    dt = BF16 if dtype == "bf16" else torch.float8_e4m3fn
    g = torch.Generator().manual_seed(3)
    a = torch.randn(W, m, K, generator=g).to(dt).to(dev)
    bT = (torch.randn(N, K, generator=g) * 0.05).to(dt).to(dev)
    bits = torch.int16 if dtype == "bf16" else torch.uint8
    want_a, want = fused.all_gather_matmul([t.clone() for t in a], bT.T, rank=rank, splits_per_rank=splits)
    assert torch.equal(want_a.view(bits), a.reshape(W * m, K).view(bits))
    shards = [t.clone() for t in a]
    if how == "misaligned":
        for r in range(W):
            mem = torch.empty(m * K + 8, dtype=dt, device=dev)
            shards[r] = mem[4:4 + m * K].view(m, K)
            shards[r].copy_(a[r])
        assert all(t.data_ptr() % 16 for t in shards)
        shards[rank] = a[rank].clone()            # (tiles read the local shard in place)
    progress = torch.full((W * splits,), 7, dtype=torch.int32, device=dev)
    got, c = fused.all_gather_matmul(shards, bT.T, None, progress, rank=rank, splits_per_rank=splits, copy_engine=how == "copy_engine")
    torch.cuda.synchronize()
    _waits.check(block=True)
    assert torch.equal(got.view(bits), a.reshape(W * m, K).view(bits)) and (progress == 1).all()
    assert torch.equal(c.view(bits), want.view(bits))


def test_all_gather_w_progress(dev):
    # test/test_allgather.py:50-75: gathered tensor exact, every flag set
    W, m, K = 8, 64, 128
    stack = orc.make_stack(W, (m, K), seed0=3)
    for splits, rank in ((1, 0), (4, 5)):
        progress = torch.zeros(W * splits, dtype=torch.int32, device=dev)
        out = comm.all_gather_w_progress([stack[r].to(dev) for r in range(W)], progress=progress,
                                         splits_per_rank=splits, rank=rank)
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), stack.reshape(W * m, K))
        assert (progress == 1).all()


def test_all_gather_matmul_wait_is_bounded(dev, tile):
    """A flag that never comes: every tile's wait ends at the limit, the kernel exits and the
    status names a chunk (no copy is enqueued here; the limit is 2 ms)."""
    from kraken_amd.fused.all_gather_matmul import _matmul_w_progress
    W, m, K, N = 4, 256, 128, 256
    a = orc.randn_bf16((W * m, K), 1).to(dev)
    bT = orc.randn_bf16((N, K), 2, 0.05).to(dev)
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    progress[1] = 1                                               # one chunk present, two missing
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    cfg = {"RANK": 0, "WORLD_SIZE": W, "SPLITS_PER_RANK": 1, "wait_limit_us": 2000}
    c = _matmul_w_progress(a, a[:m], bT.T, progress, cfg, status)
    torch.cuda.synchronize()
    assert status.item() in (3, 4)                                # 1 + index of a missing chunk
    want = (a.float().cpu() @ bT.float().cpu().T).to(BF16)
    torch.testing.assert_close(c[:2 * m].cpu(), want[:2 * m], **TOL)   # local shard and the present chunk
    # with every flag set the same call is complete and the status stays clear
    progress.fill_(1)
    status.zero_()
    c = _matmul_w_progress(a, a[:m], bT.T, progress, cfg, status)
    torch.cuda.synchronize()
    assert status.item() == 0
    torch.testing.assert_close(c.cpu(), want, **TOL)


def test_ce_persistent_variant(dev, tile):
    M, N, K, W = 512, 256, 128, 4
    a, b, _ = mk(M, N, K, 0, True)
    for rank in (0, 2):
        peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)])
        out = fused.gemm_reduce_scatter_ce_persistent(a.to(dev), b.to(dev), peers=peers.to(dev), rank=rank)
        c = (a.float() @ b.float()).to(BF16)
        bands = list(peers)
        bands.insert(rank, c[rank * M // W:(rank + 1) * M // W])
        want = orc.reduce_rotated(torch.cat(bands, 0), W, rank, acc_bf16=True)
        torch.testing.assert_close(out.cpu(), want, **TOL)


def test_split_k_loop_replays_from_a_graph(dev):
    """The GEMM entry points enqueue kernels only (the split K loop included: partial products,
    then the finishing pass): captured once, every replay reproduces the eager result bit for
    bit, with eager work between the replays."""
    M, N, K, W = 512, 256, 128, 4
    a, b, peers = mk(M, N, K, 3, True)
    bias = orc.randn_bf16((N,), 42, 0.02)
    ad, bd, pd, biasd = a.to(dev), b.to(dev), peers.to(dev), bias.to(dev)
    band_peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)]).to(dev)
    c_scratch = torch.zeros(M, N, dtype=BF16, device=dev)       # (the own band's rows are never written)
    stack = orc.make_stack(W, (M // W, K)).to(dev)
    a_few, b_few, _ = mk(128, 384, 1024, 0, False, seed=9)       # 3 tiles: its K loop is split
    a_few, b_few = a_few.to(dev), b_few.to(dev)
    assert _lib.load().kr_gemm_workspace_bytes(128, 384, 1024) > 0

    def run():
        o1 = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd)
        o2 = fused.gemm_reduce_scatter(ad, bd, peers=band_peers, rank=1, c_scratch=c_scratch)
        _, o3 = fused.all_gather_matmul(stack, bd, rank=2)
        o4 = fused.gemm_one_shot_all_reduce_fused(a_few, b_few)
        return o1, o2, c_scratch, o3, o4

    eager = [t.clone() for t in run()]
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        run()                                   # the stream's workspace exists before the capture
        side.synchronize()
        with torch.cuda.graph(g, stream=side):
            got = run()
    for rep in range(3):
        for t in got:
            t.zero_()
        _ = fused.gemm_one_shot_all_reduce_fused(a_few, b_few)   # eager work between the replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for e, r in zip(eager, got):
            assert torch.equal(e, r)


@pytest.mark.parametrize("b_t", [False, True])
def test_both_mfma_block_shapes_agree(dev, monkeypatch, b_t):
    """The 256 x 256 kernel's k loop on 16x16x32 blocks (default) and on 32x32x16 blocks: the same
    products, summed 32 or 16 at a time inside the matrix cores, so the fp32 results agree to
    rounding and the bf16 ones to an ulp -- for full and ragged shapes, the reduce-scatter form
    and the split launches."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    outs = {}
    for mfma in ("16", "32"):
        monkeypatch.setenv("KRAKEN_AMD_GEMM_MFMA", mfma)
        res = []
        for (M, N, K) in [(512, 768, 448), (520, 264, 192), (256, 256, 64)]:
            a, b, _ = mk(M, N, K, 0, b_t, seed=K)
            ad, bd = a.to(dev), b.to(dev)
            res.append(fused.gemm_one_shot_all_reduce_fused(ad, bd))
            res.append(fused.gemm_one_shot_all_reduce_fused(ad, bd, out_dtype=BF16))
        M, N, K, W = 1024, 512, 256, 4
        a, b, _ = mk(M, N, K, 0, b_t, seed=1)
        peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)]).to(dev)
        c_scratch = torch.zeros(M, N, dtype=BF16, device=dev)
        res.append(fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=peers, rank=2, c_scratch=c_scratch))
        res.append(c_scratch)
        monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", "4")      # 6 tiles, every one split four ways
        a, b, _ = mk(512, 768, 1024, 0, b_t, seed=2)
        res.append(fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev)))
        monkeypatch.delenv("KRAKEN_AMD_GEMM_TAILSPLIT")
        outs[mfma] = res
    for x, y in zip(outs["16"], outs["32"]):
        if x.dtype == torch.float32:
            torch.testing.assert_close(x, y, rtol=1e-5, atol=1e-4)
        else:
            # two bf16 ulps: in the reduce-scatter form the 32x32x16 kernel adds the band's peers on
            # the matrix cores (one rounding), the 16x16x32 kernel in the epilogue (product rounded first)
            torch.testing.assert_close(x, y, rtol=1.6e-2, atol=1e-2)
    a, b, _ = mk(512, 768, 448, 0, b_t, seed=448)
    torch.testing.assert_close(outs["16"][0].cpu(), a.float() @ b.float(), rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("mfma", ["16", "32"])
def test_split_parts_of_very_few_k_steps(dev, monkeypatch, b_t, mfma):
    """Forced splits that leave a workgroup one or two k-steps (and uneven shares): the prologue,
    the loads past the end and the waits of the k loop must still line up."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_MFMA", mfma)
    for (M, N, K, S) in [(512, 768, 256, 4), (512, 768, 192, 3), (256, 256, 64, 1), (512, 512, 128, 2), (768, 512, 320, 5),
                         (512, 768, 448, 2)]:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", str(S))
        a, b, _ = mk(M, N, K, 0, b_t, seed=S)
        out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev))
        torch.testing.assert_close(out.cpu(), a.float() @ b.float(), rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("cols", [256, 224])
@pytest.mark.parametrize("M,N,K,S", [(513, 776, 576, 3), (255, 224, 128, 2), (264, 456, 1024, 8), (512, 448, 320, 5), (8, 8, 192, 2), (520, 680, 64 * 17, 4),
                                     (513, 776, 600, 3), (264, 456, 1032, 5), (512, 448, 328, 2), (256, 256, 72, 2)])
def test_ragged_tiles_in_parts(dev, monkeypatch, M, N, K, S, cols):
    """Every 256 x 256 or 256 x 224 tile's K loop in parts, with edge tiles of one row, one 16-byte piece or all but one,
    and a last k-step of one 16-byte piece or more that is not full: all rows with peers and bias, and a band that starts inside a tile.  Small integers: every fp32 sum is exact."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", str(S))
    monkeypatch.setenv("KRAKEN_AMD_GEMM_N224", str(int(cols == 224)))
    _lib.reload_env()
    g = torch.Generator().manual_seed(K + N)
    a, b = torch.randint(-4, 5, (M, K), generator=g).float(), torch.randint(-4, 5, (K, N), generator=g).float()
    peers = torch.randint(-8, 9, (9, M, N), generator=g).to(BF16)
    bias = torch.randint(-8, 9, (N,), generator=g).to(BF16)
    for b_t in (True,) if cols == 224 else (False, True):
        p = _lib.gemm_plan(M, N, K, b_t, 9, M, workspace_bytes=1 << 40)
        assert (p["tile_n"], p["tail_tiles"], p["tail_splits"]) == (cols, -(-M // 256) * -(-N // cols), S)
        ad, bd = a.to(BF16).to(dev), b.T.contiguous().to(BF16).to(dev).T if b_t else b.to(BF16).to(dev)
        out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=peers.to(dev), bias=bias.to(dev))
        assert torch.equal(out.cpu(), a @ b + peers.float().sum(0) + bias.float())
        if M % 4 == 0:
            c = torch.zeros(M, N, dtype=BF16, device=dev)
            rows = slice(M // 4, M // 2)
            got = fused.gemm_reduce_scatter(ad, bd, peers=peers[:3, :M // 4].contiguous().to(dev), rank=1, c_scratch=c).cpu()
            product, summed = a @ b, peers[:3, :M // 4].float().sum(0)
            # (a tile wholly in the band rounds once, others round the product first)
            once, twice = (product[rows] + summed).to(BF16), (product[rows].to(BF16).float() + summed).to(BF16)
            assert ((got == once) | (got == twice)).all()
            c = c.cpu()
            assert (c[rows] == 0).all()
            c[rows] = product[rows].to(BF16)
            assert torch.equal(c, product.to(BF16))


@pytest.mark.parametrize("M,N,K,b_t,cols", [(500, 6656, 8192, True, 224), (576, 4608, 10560, False, 256), (300, 1032, 4096, True, 128)])
def test_ragged_tiles_in_parts_where_the_rule_takes_them(dev, M, N, K, b_t, cols):
    """Nothing forced: seven peers, bf16 result, against the exact sums."""
    plan = _lib.gemm_plan(M, N, K, b_t, 7, M, workspace_bytes=_lib.load().kr_gemm_workspace_bytes(M, N, K))
    assert plan["tile_n"] == cols and (plan["tail_splits"] > 1) == (cols != 128)
    g = torch.Generator().manual_seed(K)
    a = torch.randint(-2, 3, (M, K), generator=g).float().to(dev)
    b = torch.randint(-1, 2, (K, N), generator=g).float().to(dev)
    peers = torch.randint(-8, 9, (7, M, N), generator=g).to(BF16).to(dev)
    b16 = b.T.contiguous().to(BF16).T if b_t else b.to(BF16)
    out = fused.gemm_one_shot_all_reduce_fused(a.to(BF16), b16, peers=peers)
    assert torch.equal(out, a @ b + peers.float().sum(0))


def _band_tile_counts(M, N, W, bm):
    rows = M // W
    return [(((r + 1) * rows - 1) // bm - (r * rows) // bm + 1) * -(-N // bm) for r in range(W)]


@pytest.mark.parametrize("shape,W,rank", [((512, 256, 128), 4, 1), ((768, 384, 192), 3, 2), ((1024, 512, 256), 8, 7),
                                          ((1000, 264, 512), 4, 0), ((1000, 264, 520), 4, 3)])
def test_producer_gemm_flags_every_band(dev, tile, shape, W, rank):
    """Producer GEMM of the copy-engine reduce-scatter: all of C, one counter and one flag per
    destination rank's band (bands that start inside a tile included)."""
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import gemm_producer_w_progress
    M, N, K = shape
    a, b, _ = mk(M, N, K, 0, True, seed=W)
    gemm_out = torch.full((M, N), float("nan"), dtype=BF16, device=dev)
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    signal_pad = torch.zeros(W, dtype=torch.int32, device=dev)
    gemm_producer_w_progress(a.to(dev), b.to(dev), gemm_out, progress, signal_pad, {"RANK": rank, "WORLD_SIZE": W})
    torch.cuda.synchronize()
    assert signal_pad.tolist() == [1] * W
    assert progress.tolist() in (_band_tile_counts(M, N, W, 128), _band_tile_counts(M, N, W, 256))
    torch.testing.assert_close(gemm_out.cpu(), (a.float() @ b.float()).to(BF16), **TOL)


def test_producer_gemm_counts_bands_of_a_shape_with_a_partial_last_round(dev):
    """272 tiles of 256 x 256 = one round of the compute units and a partial second one: the plain GEMM
    would split that tail over idle compute units (a workspace is asked for), the producer keeps the
    one-pass kernel so that every band is counted and flagged when it is finished."""
    from kraken_amd import _lib
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import gemm_producer_w_progress
    M, N, K, W, rank = 4352, 4096, 4096, 8, 3
    assert _lib.load().kr_gemm_workspace_bytes(M, N, K) > 0
    g = torch.Generator().manual_seed(11)
    a = (torch.randn(M, K, generator=g) * 0.25).to(BF16)
    b = (torch.randn(K, N, generator=g) * 0.25).to(BF16)
    gemm_out = torch.full((M, N), float("nan"), dtype=BF16, device=dev)
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    signal_pad = torch.zeros(W, dtype=torch.int32, device=dev)
    gemm_producer_w_progress(a.to(dev), b.to(dev), gemm_out, progress, signal_pad, {"RANK": rank, "WORLD_SIZE": W})
    torch.cuda.synchronize()
    assert signal_pad.tolist() == [1] * W
    assert progress.tolist() == _band_tile_counts(M, N, W, 256)
    torch.testing.assert_close(gemm_out.cpu(), (a.float() @ b.float()).to(BF16), **TOL)


@pytest.mark.parametrize("rank", [0, 2])
def test_copy_engine_scatter_overlaps_the_producer(dev, tile, rank):
    """The reference's overlap: the band copies sit on a side stream behind stream-ordered waits
    for the producer's flags (kraken/fused/gemm_reduce_scatter_ce_persistent.py:137-175,343-370)."""
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import gemm_producer_w_progress
    M, N, K, W = 2048, 1024, 256, 4
    a, b, _ = mk(M, N, K, 0, True, seed=3)
    peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)])
    sent = torch.full((W, M // W, N), float("nan"), dtype=BF16, device=dev)
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    out = fused.gemm_reduce_scatter_ce_persistent(a.to(dev), b.to(dev), peers=peers.to(dev), rank=rank, sent=sent,
                                                  status=status)
    torch.cuda.synchronize()
    assert status.item() == 0
    c = (a.float() @ b.float()).to(BF16)
    bands = list(peers)
    bands.insert(rank, c[rank * M // W:(rank + 1) * M // W])
    want = orc.reduce_rotated(torch.cat(bands, 0), W, rank, acc_bf16=True)
    torch.testing.assert_close(out.cpu(), want, **TOL)
    # every other rank's band went out as the GEMM wrote it; the own band went to the scatter buffer
    gemm_out = torch.empty(M, N, dtype=BF16, device=dev)
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    signal_pad = torch.zeros(W, dtype=torch.int32, device=dev)
    gemm_producer_w_progress(a.to(dev), b.to(dev), gemm_out, progress, signal_pad, {"RANK": rank, "WORLD_SIZE": W})
    for r in range(W):
        if r != rank:
            assert torch.equal(sent[r], gemm_out[r * M // W:(r + 1) * M // W])
        else:
            assert torch.isnan(sent[r].float()).all()
    assert torch.equal(out, fused.gemm_reduce_scatter_ce_persistent(a.to(dev), b.to(dev), peers=peers.to(dev), rank=rank))


def test_copies_on_the_copy_engines(dev):
    """copy_engine=True: the chunk copies of the all-gather and the band copies of the scatter go
    through kr_copy_engine_memcpy (SDMA) instead of copy kernels; same bits either way."""
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import copy_engine_scatter, gemm_producer_w_progress
    W, m, K, N = 4, 256, 512, 384
    stack = orc.make_stack(W, (m, K), seed0=11)
    bT = orc.randn_bf16((N, K), 43, 0.05)
    shards = [stack[r].to(dev) for r in range(W)]
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    a_out = torch.full((W * m, K), float("nan"), dtype=BF16, device=dev)
    ag, c = fused.all_gather_matmul(shards, bT.to(dev).T, a_out=a_out, rank=1, splits_per_rank=2, copy_engine=True,
                                    status=status)
    torch.cuda.synchronize()
    assert status.item() == 0 and torch.equal(ag.cpu(), stack.reshape(W * m, K))
    assert torch.equal(c, fused.all_gather_matmul(stack.to(dev), bT.to(dev).T)[1])
    gemm_out = torch.empty(W * m, N, dtype=BF16, device=dev)
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    signal_pad = torch.zeros(W, dtype=torch.int32, device=dev)
    gemm_producer_w_progress(ag, bT.to(dev).T, gemm_out, progress, signal_pad, {"RANK": 2, "WORLD_SIZE": W})
    sent = torch.zeros(W, m, N, dtype=BF16, device=dev)
    copy_engine_scatter(gemm_out, sent, signal_pad, rank=2, status=status, copy_engine=True)
    torch.cuda.synchronize()
    assert status.item() == 0 and torch.equal(sent.view(W * m, N), gemm_out)


def test_flag_arrive_wait(dev):
    """test/test_ptx_utils.py:80-116: 8 producer workgroups set their flags, 32 consumers wait for
    them in the same launch; the flags end as 1 and no consumer runs into the limit."""
    lib = _lib.load()
    stream = torch.cuda.current_stream(dev).cuda_stream
    flags = torch.zeros(64, dtype=torch.int32, device=dev)
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    _lib.check(lib.kr_flag_arrive_wait(flags.data_ptr(), 8, 32, 0, status.data_ptr(), stream), "flag_arrive_wait")
    torch.cuda.synchronize()
    expect = torch.zeros_like(flags)
    expect[:8] = 1
    assert torch.equal(flags, expect) and status.item() == 0
    # one producer, four consumers, on a flag further into the array
    flags.zero_()
    _lib.check(lib.kr_flag_arrive_wait(flags.data_ptr() + 4, 1, 4, 2000, status.data_ptr(), stream), "flag_arrive_wait")
    torch.cuda.synchronize()
    assert flags.tolist() == [0, 1] + [0] * 62 and status.item() == 0


def test_copy_engine_scatter_wait_is_bounded(dev):
    """A flag that never comes: the stream-ordered wait gives up after its limit, records it in
    `status`, and the stream drains."""
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import copy_engine_scatter
    W, rows, N = 2, 64, 128
    inp = torch.ones(W * rows, N, dtype=BF16, device=dev)
    signal_pad = torch.tensor([1, 0], dtype=torch.int32, device=dev)      # band 1 is never flagged
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    outs = [torch.zeros(rows, N, dtype=BF16, device=dev) for _ in range(W)]
    copy_engine_scatter(inp, outs, signal_pad, rank=0, wait_limit_us=2000, status=status)
    torch.cuda.synchronize()
    assert status.item() == 1
    ok = torch.zeros(1, dtype=torch.int32, device=dev)
    copy_engine_scatter(inp, [outs[0], None], torch.ones(W, dtype=torch.int32, device=dev), rank=1,
                        wait_limit_us=2000, status=ok)
    torch.cuda.synchronize()
    assert ok.item() == 0 and torch.equal(outs[0], inp[:rows])


def test_bounded_waits_without_a_status_do_not_fail_silently(dev):
    """No `status` passed: the wrappers keep a word of their own, every wait of the call shares it
    (after the first one runs out the others give up at once), and the failure is raised on the
    next look -- here by an explicit check, in use by the next call of an overlap function."""
    import time
    from kraken_amd import _waits
    from kraken_amd._lib import KrakenAmdError
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import copy_engine_scatter
    W, rows, N = 8, 64, 128
    inp = torch.ones(W * rows, N, dtype=BF16, device=dev)
    outs = [torch.zeros(rows, N, dtype=BF16, device=dev) for _ in range(W)]
    _waits.check(block=True)                                              # nothing pending from earlier tests
    copy_engine_scatter(inp, outs, torch.ones(W, dtype=torch.int32, device=dev), rank=0)      # every flag is set
    _waits.check(block=True)
    never = torch.zeros(W, dtype=torch.int32, device=dev)                 # no flag ever comes: 8 waits of 20 ms
    t0 = time.perf_counter()
    copy_engine_scatter(inp, outs, never, rank=0, wait_limit_us=20000)
    with pytest.raises(KrakenAmdError, match="ran out in.*copy_engine_scatter"):
        _waits.check(block=True)
    assert time.perf_counter() - t0 < 0.1                                 # one limit, not eight
    _waits.check(block=True)                                              # reported once
    # two failing calls before anybody looks: both are named (the second gives up at once: the
    # stream's word is still set when its waits start)
    t0 = time.perf_counter()
    copy_engine_scatter(inp, outs, never, rank=0, wait_limit_us=20000)
    copy_engine_scatter(inp, outs, never, rank=0, wait_limit_us=20000)
    with pytest.raises(KrakenAmdError) as both:
        _waits.check(block=True)
    assert str(both.value).count("copy_engine_scatter") == 2
    assert time.perf_counter() - t0 < 0.1
    _waits.check(block=True)
    assert _waits.new_status(dev).item() == 0                             # cleared by the report
    # the all-gather matmul with chunks that never arrive (no copies are enqueued for this call)
    from kraken_amd.fused.all_gather_matmul import _matmul_w_progress
    m, K, Nn = 64, 128, 256
    a = orc.randn_bf16((4 * m, K), 1).to(dev)
    bT = orc.randn_bf16((Nn, K), 2, 0.05).to(dev)
    status = _waits.new_status(dev)
    _matmul_w_progress(a, a[:m], bT.T, torch.zeros(4, dtype=torch.int32, device=dev),
                       {"RANK": 0, "WORLD_SIZE": 4, "SPLITS_PER_RANK": 1, "wait_limit_us": 2000}, status)
    _waits.watch(status, "all_gather_matmul")
    with pytest.raises(KrakenAmdError, match="all_gather_matmul"):
        _waits.check(block=True)


def test_ce_persistent_reference_shape(dev):
    """(8192, 4096, 14336), the shape of test/test_gemm_reduce_scatter.py:93-111 (tolerance 1e-2
    there; the gate here is the library's 2e-2 on sampled rows)."""
    M, N, K, W, rank = 8192, 4096, 14336, 8, 5
    a = orc.randn_bf16((M, K), 42)
    b = orc.randn_bf16((N, K), 43, 0.02).T
    peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)])
    out = fused.gemm_reduce_scatter_ce_persistent(a.to(dev), b.to(dev), peers=peers.to(dev), rank=rank)
    pick = torch.tensor([0, 1, 127, 128, 255, 256, 700, 1023])
    own = (a[rank * 1024 + pick].float() @ b.float()).to(BF16)
    bands = [p[pick] for p in peers]
    bands.insert(rank, own)
    want = orc.reduce_rotated(torch.cat(bands, 0), W, rank, acc_bf16=True)
    torch.testing.assert_close(out.cpu()[pick], want, **TOL)


def _sampled_rows_check(got, rows, a, b, extra, tol=TOL):
    want = a[rows].float() @ b.float()
    if extra is not None:
        want = want + extra
    torch.testing.assert_close(got.cpu()[rows].float(), want.to(BF16).float(), **tol)


def test_baseline_config4_full_size(dev, monkeypatch):
    """A [8192,3584] @ B [3584,8192]; band of 1024 rows + 7 partials.  Oracle on sampled rows."""
    monkeypatch.delenv("KRAKEN_AMD_GEMM_TILE", raising=False)
    monkeypatch.delenv("KRAKEN_AMD_GEMM_PEERS", raising=False)
    M, N, K, W, rank = 8192, 8192, 3584, 8, 3
    a = orc.randn_bf16((M, K), 42)
    b = orc.randn_bf16((K, N), 43, 0.02)
    peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)])
    c_scratch = torch.empty(M, N, dtype=BF16, device=dev)
    out = fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=peers.to(dev), rank=rank, c_scratch=c_scratch)
    band = torch.arange(rank * 1024, (rank + 1) * 1024)
    pick = band[torch.tensor([0, 1, 31, 32, 255, 256, 511, 777, 1023])]
    want = a[pick].float() @ b.float() + peers[:, pick - rank * 1024].float().sum(0)
    torch.testing.assert_close(out.cpu()[pick - rank * 1024].float(), want.to(BF16).float(), **TOL)
    others = torch.tensor([0, 255, 256, 1023, 4096, 5000, 8191])
    _sampled_rows_check(c_scratch, others, a, b, None)
    # whole-matrix check against the device library GEMM in fp32
    ref = (a.to(dev).float() @ b.to(dev).float())
    ref_band = ref[band.to(dev)] + peers.to(dev).float().sum(0)
    torch.testing.assert_close(out.float(), ref_band.to(BF16).float(), **TOL)


def test_baseline_config5_full_size(dev, monkeypatch):
    monkeypatch.delenv("KRAKEN_AMD_GEMM_TILE", raising=False)
    monkeypatch.delenv("KRAKEN_AMD_GEMM_PEERS", raising=False)
    # fused all-reduce: A [4096,1024] @ B [1024,8192] + 7 partials + bias
    M, N, K, P = 4096, 8192, 1024, 7
    a = orc.randn_bf16((M, K), 42)
    b = orc.randn_bf16((K, N), 43, 0.02)
    peers = torch.stack([orc.randn_bf16((M, N), 100 + j) for j in range(P)])
    bias = orc.randn_bf16((N,), 42, 0.02)
    out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev), peers=peers.to(dev), bias=bias.to(dev),
                                               out_dtype=BF16)
    pick = torch.tensor([0, 63, 64, 127, 128, 2047, 4095])
    want = a[pick].float() @ b.float() + peers[:, pick].float().sum(0) + bias.float()
    torch.testing.assert_close(out.cpu()[pick].float(), want.to(BF16).float(), **TOL)
    ref = a.to(dev).float() @ b.to(dev).float() + peers.to(dev).float().sum(0) + bias.to(dev).float()
    torch.testing.assert_close(out.float(), ref.to(BF16).float(), **TOL)
    del peers, out, ref
    # all-gather matmul: A stack [8,1024,8192] @ B [8192,3584] (B.T contiguous)
    W, m, K2, N2 = 8, 1024, 8192, 3584
    stack = orc.make_stack(W, (m, K2), seed0=42)
    bT = orc.randn_bf16((N2, K2), 43, 0.02)
    ag, c = fused.all_gather_matmul(stack.to(dev), bT.to(dev).T, rank=5)
    assert torch.equal(ag.cpu(), stack.reshape(W * m, K2))
    rows = torch.tensor([0, 1023, 1024, 5 * 1024, 5 * 1024 + 17, 8191])
    _sampled_rows_check(c, rows, stack.reshape(W * m, K2), bT.T, None)
    ref = stack.to(dev).reshape(W * m, K2).float() @ bT.to(dev).T.float()
    torch.testing.assert_close(c.float(), ref.to(BF16).float(), **TOL)


def test_all_gather_matmul_reference_test_shape(dev, monkeypatch):
    """test/test_allgather_matmul.py:51-66: M=4096, N=6656, K=16384, bf16, B.T contiguous, here with W=8 shards of
    512 rows; the gathered A must be the exact stack, C within the gate of the sampled-row oracle
    and of the device's fp32 GEMM on the whole matrix."""
    monkeypatch.delenv("KRAKEN_AMD_GEMM_TILE", raising=False)
    monkeypatch.delenv("KRAKEN_AMD_GEMM_PEERS", raising=False)
    W, M, N, K = 8, 4096, 6656, 16384
    stack = orc.make_stack(W, (M // W, K), seed0=42)
    bT = orc.randn_bf16((N, K), 43, 0.02)
    sd = stack.to(dev)
    for rank in (0, 5):
        ag, c = fused.all_gather_matmul(sd, bT.to(dev).T, rank=rank)
        assert torch.equal(ag.cpu(), stack.reshape(M, K))
        rows = torch.tensor([0, 511, 512, 5 * 512 + 3, 4095])
        _sampled_rows_check(c, rows, stack.reshape(M, K), bT.T, None)
        ref = sd.reshape(M, K).float() @ bT.to(dev).T.float()
        torch.testing.assert_close(c.float(), ref.to(BF16).float(), **TOL)


@pytest.mark.parametrize("mode", ["mfma", "epilogue"])
def test_non_finite_partial_sum_stays_local(dev, monkeypatch, mode):
    """An Inf in one peer's partial sum: added in the epilogue it shows up in its own element
    only; added on the matrix cores (identity MFMA, 0 * Inf = NaN) it may also spoil the columns
    of its row that share its MFMA -- the aligned block of 32 -- and nothing else."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_PEERS", mode)
    M, N, K, P = 512, 512, 256, 3
    a, b, peers = mk(M, N, K, P)
    r, c = 300, 77
    peers[1, r, c] = float("inf")
    out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev), peers=peers.to(dev), out_dtype=BF16).cpu().float()
    clean = peers.clone()
    clean[1, r, c] = 0.0
    want = orc.gemm_all_reduce(a, b, clean).to(BF16).float()
    bad = ~torch.isfinite(out)
    assert bad[r, c]
    group = torch.zeros_like(bad)
    group[r, c // 32 * 32:c // 32 * 32 + 32] = True
    assert not (bad & ~group).any()
    if mode == "epilogue":
        assert bad.sum() == 1 and out[r, c] == float("inf")
    torch.testing.assert_close(out[~group], want[~group], **TOL)


@pytest.mark.parametrize("M,N,K", [(3072, 3072, 264), (3000, 3080, 328)])    # 144 tiles of 256 x 256, whole and ragged
@pytest.mark.parametrize("b_t", [False, True])
def test_non_finite_partial_sum_stays_in_its_element_with_a_ragged_k(dev, M, N, K, b_t):
    """K no multiple of 64: an Inf and a NaN in one peer each stay in their own element, and a bf16 result is the
    product rounded to bf16, then the sum with the peers rounded once more (small integers: all sums exact)."""
    g = torch.Generator().manual_seed(K)
    a = torch.randint(-4, 5, (M, K), generator=g).float()
    b = torch.randint(-4, 5, (K, N), generator=g).float()
    peers = torch.randint(-8, 9, (3, M, N), generator=g).float()
    product = a @ b
    once = product + peers.sum(0)
    twice = product.to(BF16).float() + peers.sum(0)
    assert not torch.equal(once.to(BF16), twice.to(BF16))
    peers[1, 300, 77], peers[2, 700, 1030] = float("inf"), float("nan")
    once[300, 77] = twice[300, 77] = float("inf")
    once[700, 1030] = twice[700, 1030] = float("nan")
    ad, pd = a.to(BF16).to(dev), peers.to(BF16).to(dev)
    bd = b.T.contiguous().to(BF16).to(dev).T if b_t else b.to(BF16).to(dev)
    for dtype, want in ((torch.float32, once), (BF16, twice.to(BF16))):
        out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, out_dtype=dtype).cpu()
        assert torch.equal(torch.isnan(out), torch.isnan(want))
        assert torch.equal(torch.nan_to_num(out.float(), nan=0.5), torch.nan_to_num(want.float(), nan=0.5))


@pytest.mark.parametrize("P", [1, 2, 7, 8, 15])
def test_gemm_all_reduce_world_sizes(dev, tile, P):
    """Every world size the C ABI accepts (W = P + 1 up to 16), on a shape with whole-band
    256-tiles (matrix-core or epilogue peer path) and on a ragged one (generic epilogue path)."""
    for (M, N, K) in [(512, 256, 160), (200, 136, 72)]:
        a, b, peers = mk(M, N, K, P, seed=P)
        bias = orc.randn_bf16((N,), 9, 0.02)
        want = orc.gemm_all_reduce(a, b, peers, bias)
        out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev), peers=peers.to(dev), bias=bias.to(dev))
        torch.testing.assert_close(out.cpu(), want, rtol=1e-3, atol=1e-3)
        outb = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev), peers=peers.to(dev), bias=bias.to(dev),
                                                    out_dtype=BF16)
        torch.testing.assert_close(outb.cpu(), want.to(BF16), **TOL)


@pytest.mark.parametrize("P", [1, 3, 7, 15])
def test_separate_peer_buffers_match_the_stacked_form(dev, tile, P):
    """Pointer-table entry point: the peers' partial sums as P separate allocations give the
    stacked form's bits, on whole-band 256-tiles (matrix-core path, 7-peer and generic epilogue
    paths) and on a ragged shape."""
    for (M, N, K) in [(512, 512, 192), (200, 136, 72)]:
        a, b, peers = mk(M, N, K, P, seed=P)
        bias = orc.randn_bf16((N,), 9, 0.02)
        pads, plist = [], [None] * P
        for j in reversed(range(P)):
            pads.append(torch.empty(1208 * (j % 3 + 1), dtype=BF16, device=dev))
            plist[j] = peers[j].to(dev)
        ad, bd, pd, biasd = a.to(dev), b.to(dev), peers.to(dev), bias.to(dev)
        for dt in (torch.float32, BF16):
            o1 = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd, out_dtype=dt)
            o2 = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=plist, bias=biasd, out_dtype=dt)
            assert torch.equal(o1, o2)
        torch.testing.assert_close(o2.cpu(), orc.gemm_all_reduce(a, b, peers, bias).to(BF16), **TOL)
    # reduce-scatter: band of rank 1 of W = P + 1, other bands to the scratch
    W = P + 1
    M, N, K = 256 * W, 256, 128
    a, b, _ = mk(M, N, K, 0)
    peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(P)])
    plist = [peers[j].to(dev) for j in range(P)]
    c1 = torch.zeros(M, N, dtype=BF16, device=dev)
    c2 = torch.zeros(M, N, dtype=BF16, device=dev)
    o1 = fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=peers.to(dev), rank=1, c_scratch=c1)
    o2 = fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=plist, rank=1, c_scratch=c2)
    assert torch.equal(o1, o2) and torch.equal(c1, c2)
    want, _ = orc.gemm_reduce_scatter(a, b, peers, 1, W)
    torch.testing.assert_close(o2.cpu(), want, **TOL)
    # the copy-engine variant takes a list as well
    o3 = fused.gemm_reduce_scatter_ce_persistent(a.to(dev), b.to(dev), peers=plist, rank=1, world_size=W)
    o4 = fused.gemm_reduce_scatter_ce_persistent(a.to(dev), b.to(dev), peers=peers.to(dev), rank=1, world_size=W)
    assert torch.equal(o3, o4)


@pytest.mark.parametrize("M,N,K", [(8, 512, 256), (512, 1024, 4096), (2048, 8192, 256)])   # bands together; one by one
@pytest.mark.parametrize("form", ["stack", "list", "strided", "overlap", "misaligned", "host"])
def test_ce_reduce_reads_the_bands_in_place(dev, M, N, K, form):
    """Where the peers and the destinations lie does not change a bit of the result, also where the reduce may not
    read them in place: peers that are overwritten by what is sent, that are not aligned, or in host memory."""
    W, rank, m = 4, 2, M // 4
    a, b, _ = mk(M, N, K, 0, True, seed=5)
    a, b = a.to(dev), b.to(dev)
    peers = torch.stack([orc.randn_bf16((m, N), 100 + j) for j in range(W - 1)])
    sent = torch.full((W, m, N), 7.0, dtype=BF16, device=dev)
    plain = torch.zeros_like(sent)
    c = torch.empty(M, N, dtype=BF16, device=dev)
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import gemm_producer_w_progress
    gemm_producer_w_progress(a, b, c, *(torch.zeros(W, dtype=torch.int32, device=dev) for _ in range(2)),
                             {"RANK": rank, "WORLD_SIZE": W})
    bands = list(peers)
    bands.insert(rank, c[rank * m:(rank + 1) * m].cpu())
    want = orc.reduce_rotated(torch.cat(bands, 0), W, rank, acc_bf16=True)
    if form == "stack":
        arg = peers.to(dev)
    elif form == "list":
        arg = [p.to(dev) for p in peers]
    elif form == "strided":
        arg = torch.zeros(W - 1, 2, m, N, dtype=BF16, device=dev)[:, 1]
        arg.copy_(peers)
        sent = torch.full((W, m, 2 * N), 7.0, dtype=BF16, device=dev)[:, :, :N]
    elif form == "overlap":
        arg = sent[:W - 1]
        arg.copy_(peers)
        sent[rank].copy_(peers[rank])
    elif form == "misaligned":
        arg = torch.empty((W - 1) * m * N + 1, dtype=BF16, device=dev)[1:].view(W - 1, m, N)
        arg.copy_(peers)
    else:
        arg = peers
    own = sent[rank].clone()
    out = fused.gemm_reduce_scatter_ce_persistent(a, b, peers=arg, rank=rank, sent=sent)
    for r in range(W):
        assert torch.equal(sent[r], own if r == rank else c[r * m:(r + 1) * m])
    assert torch.equal(out.cpu(), want)
    assert torch.equal(out, fused.gemm_reduce_scatter_ce_persistent(a, b, peers=peers.to(dev), rank=rank, sent=list(plain)))


# bands of whole tiles; of parts of one; of 1 row; K loop in parts; few rows; more than a round, bands inside a tile
@pytest.mark.parametrize("M,N,K,W", [(1024, 512, 256, 4), (600, 1048, 264, 4), (8, 1024, 512, 8), (504, 776, 4096, 8), (40, 2048, 1024, 2),
                                     (2320, 8192, 128, 8)])
@pytest.mark.parametrize("b_t", [False, True])
def test_ce_bands_stored_by_the_product(dev, M, N, K, W, b_t):
    """Destinations in one matrix: the product stores the bands there itself.  Integers up to 4 times integers up to 2
    are exact in every order of the sums (K * 8 < 2^24), so bands and result are those of the product rounded once."""
    g = torch.Generator().manual_seed(M)
    a = torch.randint(-4, 5, (M, K), generator=g).to(BF16)
    b = torch.randint(-2, 3, (K, N), generator=g).to(BF16)
    m = M // W
    ad, bd = a.to(dev), b.T.contiguous().to(dev).T if b_t else b.to(dev)
    c = (a.float() @ b.float()).to(BF16)
    for rank in (0, W - 1):
        peers = torch.stack([orc.randn_bf16((m, N), 100 + j, 30.0) for j in range(W - 1)])
        sent = torch.full((W, m, N), float("nan"), dtype=BF16, device=dev)
        version = sent._version
        out = fused.gemm_reduce_scatter_ce_persistent(ad, bd, peers=peers.to(dev), rank=rank, sent=sent)
        assert sent._version > version
        for r in range(W):
            assert torch.isnan(sent[r]).all() if r == rank else torch.equal(sent[r].cpu(), c[r * m:(r + 1) * m]), (rank, r)
        bands = list(peers)
        bands.insert(rank, c[rank * m:(rank + 1) * m])
        assert torch.equal(out.cpu(), orc.reduce_rotated(torch.cat(bands, 0), W, rank, acc_bf16=True))


def test_ce_bands_sent_over_an_operand(dev):
    """Destinations in the memory of the left operand (its rows are those of the product, N = K): not stored by the
    product, which still reads them, but copied behind it."""
    M, N, K, W, rank = 512, 256, 256, 4, 1
    a, b, peers = mk(M, N, K, W - 1, True, seed=4)
    a, b, peers = a.to(dev), b.to(dev), peers[:, :M // W].contiguous().to(dev)
    apart = torch.zeros(W, M // W, N, dtype=BF16, device=dev)
    want = fused.gemm_reduce_scatter_ce_persistent(a, b, peers=peers, rank=rank, sent=apart)
    out = fused.gemm_reduce_scatter_ce_persistent(a, b, peers=peers, rank=rank, sent=a.view(W, M // W, N))
    assert torch.equal(out, want)
    for r in range(W):
        assert r == rank or torch.equal(a.view(W, M // W, N)[r], apart[r])


@pytest.mark.parametrize("M,N,K", [(512, 1024, 256), (2048, 8192, 256)])   # bands together; one by one
@pytest.mark.parametrize("form", ["expanded", "list"])
def test_ce_bands_sent_into_one_scratch_band(dev, M, N, K, form):
    """Destinations that are one and the same memory, as a tensor expanded over the ranks or the same tensor W times:
    the bands are copied there in the order rank + 1, rank + 2, ..., so that of rank - 1 remains."""
    W, rank, m = 4, 2, M // 4
    a, b, peers = mk(M, N, K, W - 1, True, seed=9)
    a, b, peers = a.to(dev), b.to(dev), peers[:, :m].contiguous().to(dev)
    apart = torch.zeros(W, m, N, dtype=BF16, device=dev)
    want = fused.gemm_reduce_scatter_ce_persistent(a, b, peers=peers, rank=rank, sent=apart)
    scratch = torch.zeros(m, N, dtype=BF16, device=dev)
    sent = scratch.expand(W, m, N) if form == "expanded" else [scratch] * W
    out = fused.gemm_reduce_scatter_ce_persistent(a, b, peers=peers, rank=rank, sent=sent)
    assert torch.equal(scratch, apart[rank - 1])
    assert torch.equal(out, want)


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K", [(256, 256, 256), (512, 1024, 4096), (2304, 8192, 256)])   # one pass, split K loop, more than a round
def test_producer_takes_fp32_operands(dev, M, N, K, b_t):
    """gemm_producer_w_progress with fp32 operands, at shapes with and without a workspace: integers up to 2^8 times
    integers up to 8 are one bf16 value each, so every fp32 sum is exact and gemm_out the product rounded once."""
    from kraken_amd.fused.gemm_reduce_scatter_ce_persistent import gemm_producer_w_progress
    g = torch.Generator().manual_seed(K)
    a = torch.randint(-256, 257, (M, K), generator=g).float()
    b = torch.randint(-8, 9, (K, N), generator=g).float()
    assert K * 256 * 8 < 1 << 24
    ad, bd = a.to(dev), b.T.contiguous().to(dev).T if b_t else b.to(dev)
    W = 4
    c = torch.empty(M, N, dtype=BF16, device=dev)
    progress, signal_pad = (torch.zeros(W, dtype=torch.int32, device=dev) for _ in range(2))
    gemm_producer_w_progress(ad, bd, c, progress, signal_pad, {"RANK": 1, "WORLD_SIZE": W})
    assert torch.equal(c, (ad @ bd).to(BF16)), (c.float() - ad @ bd).abs().max()
    assert (signal_pad == 1).all()


@pytest.mark.parametrize("splits", [2, 3, 5, 16])
@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("ks", ["0", "1"])
def test_split_k_loop(dev, monkeypatch, splits, b_t, ks):
    """Few output tiles: several workgroups share a tile's K loop, their partial products meet
    in the workspace.  Parity with the oracle for every epilogue form and the same bits run to
    run (the parts are summed in a fixed order).  Both kernels with 128 x 128 tiles."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "128")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_KS", ks)
    monkeypatch.setenv("KRAKEN_AMD_GEMM_SPLITK", str(splits))
    for (M, N, K) in [(128, 384, 1024), (200, 136, 520), (256, 256, 64 * splits)]:
        a, b, peers = mk(M, N, K, 3, b_t, seed=splits)
        bias = orc.randn_bf16((N,), 42, 0.02)
        want = orc.gemm_all_reduce(a, b, peers, bias)
        ad, bd, pd, biasd = a.to(dev), b.to(dev), peers.to(dev), bias.to(dev)
        out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd)
        torch.testing.assert_close(out.cpu(), want, rtol=1e-3, atol=1e-3)
        for _ in range(3):
            again = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd)
            assert torch.equal(out, again)
        outb = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=[p for p in pd], bias=biasd, out_dtype=BF16)
        torch.testing.assert_close(outb.cpu(), want.to(BF16), **TOL)
        plain = fused.gemm_one_shot_all_reduce_fused(ad, bd)
        torch.testing.assert_close(plain.cpu(), orc.gemm_all_reduce(a, b), rtol=1e-3, atol=1e-3)
    # reduce-scatter: band with peers, other bands to the scratch
    M, N, K, W = 512, 256, 640, 4
    a, b, _ = mk(M, N, K, 0, b_t)
    peers = torch.stack([orc.randn_bf16((M // W, N), 100 + j) for j in range(W - 1)])
    want, c_want = orc.gemm_reduce_scatter(a, b, peers, 2, W)
    c_scratch = torch.zeros(M, N, dtype=BF16, device=dev)
    out = fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=peers.to(dev), rank=2, c_scratch=c_scratch)
    torch.testing.assert_close(out.cpu(), want, **TOL)
    rows = torch.ones(M, dtype=torch.bool)
    rows[2 * M // W:3 * M // W] = False
    torch.testing.assert_close(c_scratch.cpu()[rows], c_want[rows], **TOL)


@pytest.mark.parametrize("M,N,K,b_t,splits", [(1000, 6656, 1024, True, 1), (2048, 4096, 512, False, 1), (1990, 4104, 200, True, 1),
                                              (1100, 4096, 4168, True, 1), (300, 520, 8200, True, 13),
                                              (1272, 2312, 12296, True, 2)])
def test_register_staged_kernel_where_the_rule_takes_it(dev, M, N, K, b_t, splits):
    """More than 256 tiles of 128 x 128, and few tiles with a long K loop in parts (transposed B), nothing forced: whole
    and ragged tiles, a last k-step that is not full, seven peers and a bias.  Small integers: every fp32 sum is exact."""
    plan = _lib.gemm_plan(M, N, K, b_t, 7, M, True, workspace_bytes=_lib.load().kr_gemm_workspace_bytes(M, N, K))
    assert plan["kernel"] == "gemm_reduce_kernel" and plan["k_splits"] == splits
    g = torch.Generator().manual_seed(K)
    a = torch.randint(-4, 5, (M, K), generator=g).float().to(dev)
    b = torch.randint(-4, 5, (K, N), generator=g).float().to(dev)
    peers = torch.randint(-8, 9, (7, M, N), generator=g).to(BF16).to(dev)
    bias = torch.randint(-8, 9, (N,), generator=g).to(BF16).to(dev)
    b16 = b.T.contiguous().to(BF16).T if b_t else b.to(BF16)
    out = fused.gemm_one_shot_all_reduce_fused(a.to(BF16), b16, peers=peers, bias=bias)
    assert torch.equal(out, a @ b + peers.float().sum(0) + bias.float())


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("force", ["", "3"])
def test_tail_round_split(dev, monkeypatch, b_t, force):
    """272 tiles of 256 x 256 = one full round of 256 + 16: the 16 get several workgroups each
    (second launch) and a finishing pass; every epilogue form against the oracle, and the plain
    product against the one-launch result."""
    if force:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", force)
    M, N, K, W = 4352, 4096, 4096 if not force else 1024, 2
    assert _lib.load().kr_gemm_workspace_bytes(M, N, K) == 16 * (int(force) if force else 8) * 256 * 256 * 4
    a, b, _ = mk(M, N, K, 0, b_t, seed=5)
    ad, bd = a.to(dev), b.to(dev)
    prod = a.float() @ b.float()
    plain = fused.gemm_one_shot_all_reduce_fused(ad, bd)
    torch.testing.assert_close(plain.cpu(), prod, rtol=1e-3, atol=1e-3)
    assert torch.equal(plain, fused.gemm_one_shot_all_reduce_fused(ad, bd))          # reproducible
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", "0")
    one_launch = fused.gemm_one_shot_all_reduce_fused(ad, bd)
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", force) if force else monkeypatch.delenv("KRAKEN_AMD_GEMM_TAILSPLIT")
    torch.testing.assert_close(plain, one_launch, rtol=1e-4, atol=1e-4)
    assert not torch.equal(plain, one_launch) or K <= 64                              # the split did run
    # all-reduce form: peers and bias on every row, bf16 result
    peers = torch.stack([orc.randn_bf16((M, N), 100 + j) for j in range(2)])
    bias = orc.randn_bf16((N,), 9, 0.02)
    out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=peers.to(dev), bias=bias.to(dev), out_dtype=BF16)
    want = (prod + peers.float().sum(0) + bias.float()).to(BF16)
    torch.testing.assert_close(out.cpu(), want, **TOL)
    # reduce-scatter form: band of rank 1 (rows 2176.., it starts inside a tile), other rows to the scratch
    rank = 1
    bp = torch.stack([orc.randn_bf16((M // W, N), 200 + j) for j in range(W - 1)])
    c_scratch = torch.zeros(M, N, dtype=BF16, device=dev)
    out = fused.gemm_reduce_scatter(ad, bd, peers=[p.to(dev) for p in bp], rank=rank, world_size=W, c_scratch=c_scratch)
    band = slice(rank * (M // W), (rank + 1) * (M // W))
    torch.testing.assert_close(out.cpu(), (prod[band] + bp.float().sum(0)).to(BF16), **TOL)
    rows = torch.ones(M, dtype=torch.bool)
    rows[band] = False
    torch.testing.assert_close(c_scratch.cpu()[rows], prod[rows].to(BF16), **TOL)


@pytest.mark.parametrize("b_t", [False, True])
def test_whole_launch_split_for_few_rows(dev, monkeypatch, b_t):
    """24 tiles of 256 x 256 and a long K loop: no full round at all, every tile's K loop is
    shared by 8 workgroups of the large-tile kernel.  Chosen by default for row-major B; forced
    for transposed-contiguous B (which takes this path only with more work per tile)."""
    M, N, K, W = 512, 3072, 8192, 4
    lib = _lib.load()
    if b_t:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    assert lib.kr_gemm_workspace_bytes(M, N, K) == 24 * 8 * 256 * 256 * 4
    a, b, _ = mk(M, N, K, 0, b_t, seed=11)
    ad, bd = a.to(dev), b.to(dev)
    prod = a.float() @ b.float()
    plain = fused.gemm_one_shot_all_reduce_fused(ad, bd)
    torch.testing.assert_close(plain.cpu(), prod, rtol=1e-3, atol=2e-3)
    assert torch.equal(plain, fused.gemm_one_shot_all_reduce_fused(ad, bd))          # reproducible
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "128")
    other = fused.gemm_one_shot_all_reduce_fused(ad, bd)
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256") if b_t else monkeypatch.delenv("KRAKEN_AMD_GEMM_TILE")
    torch.testing.assert_close(plain, other, rtol=1e-4, atol=1e-4)
    assert not torch.equal(plain, other)                                              # another kernel did run
    peers = torch.stack([orc.randn_bf16((M, N), 100 + j) for j in range(2)])
    bias = orc.randn_bf16((N,), 9, 0.02)
    out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=peers.to(dev), bias=bias.to(dev), out_dtype=BF16)
    torch.testing.assert_close(out.cpu(), (prod + peers.float().sum(0) + bias.float()).to(BF16), **TOL)
    rank = 1                                     # band = rows 128..255, inside the first row of tiles
    bp = torch.stack([orc.randn_bf16((M // W, N), 200 + j) for j in range(W - 1)])
    c_scratch = torch.zeros(M, N, dtype=BF16, device=dev)
    out = fused.gemm_reduce_scatter(ad, bd, peers=bp.to(dev), rank=rank, world_size=W, c_scratch=c_scratch)
    band = slice(rank * (M // W), (rank + 1) * (M // W))
    torch.testing.assert_close(out.cpu(), (prod[band] + bp.float().sum(0)).to(BF16), **TOL)
    rows = torch.ones(M, dtype=torch.bool)
    rows[band] = False
    torch.testing.assert_close(c_scratch.cpu()[rows], prod[rows].to(BF16), **TOL)


@pytest.mark.parametrize("b_t", [False, True])
def test_ragged_shapes_on_the_large_tile(dev, monkeypatch, b_t):
    """M and N that 256 does not divide, on the 256 x 256 kernel: edge tiles read short operand
    panels and store through the bounds-checked epilogue; every epilogue form."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    for (M, N, K) in [(1000, 520, 192), (300, 264, 64), (513, 1032, 256), (768, 8, 128), (8, 768, 128)]:
        a, b, peers = mk(M, N, K, 2, b_t, seed=M)
        bias = orc.randn_bf16((N,), 42, 0.02)
        ad, bd, pd, biasd = a.to(dev), b.to(dev), peers.to(dev), bias.to(dev)
        want = orc.gemm_all_reduce(a, b, peers, bias)
        out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd)
        torch.testing.assert_close(out.cpu(), want, rtol=1e-3, atol=1e-3)
        outb = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd, out_dtype=BF16)
        torch.testing.assert_close(outb.cpu(), want.to(BF16), **TOL)
        plain = fused.gemm_one_shot_all_reduce_fused(ad, bd, out_dtype=BF16)
        torch.testing.assert_close(plain.cpu(), orc.gemm_all_reduce(a, b).to(BF16), **TOL)
    # reduce-scatter with a band that ends inside the ragged last tile; guard rows behind the outputs
    M, N, K, W = 1000, 520, 192, 4
    a, b, _ = mk(M, N, K, 0, b_t, seed=3)
    for rank in (0, 3):
        bp = torch.stack([orc.randn_bf16((M // W, N), 300 + j) for j in range(W - 1)])
        want, c_want = orc.gemm_reduce_scatter(a, b, bp, rank, W)
        c_scratch = torch.zeros(M + 8, N, dtype=BF16, device=dev)
        out = fused.gemm_reduce_scatter(a.to(dev), b.to(dev), peers=bp.to(dev), rank=rank, c_scratch=c_scratch[:M])
        torch.testing.assert_close(out.cpu(), want, **TOL)
        rows = torch.ones(M, dtype=torch.bool)
        rows[rank * (M // W):(rank + 1) * (M // W)] = False
        torch.testing.assert_close(c_scratch.cpu()[:M][rows], c_want[rows], **TOL)
        assert (c_scratch[M:] == 0).all()                     # nothing written past row M


def test_split_k_is_chosen_for_few_rows(dev):
    """The default heuristic: 128 x 6656 x 4096 (52 tiles) asks for a workspace, 4096 x 4096 does not."""
    lib = _lib.load()
    assert lib.kr_gemm_workspace_bytes(128, 6656, 4096) > 0
    assert lib.kr_gemm_workspace_bytes(4096, 4096, 4096) == 0
    assert lib.kr_gemm_workspace_bytes(128, 6656, 64) == 0          # one k-step: nothing to split
    a, b, _ = mk(128, 6656, 4096, 0, True)
    out = fused.gemm_one_shot_all_reduce_fused(a.to(dev), b.to(dev))
    torch.testing.assert_close(out.cpu(), orc.gemm_all_reduce(a, b), rtol=1e-3, atol=2e-3)


def test_gemm_paths_replay_from_a_graph(dev, monkeypatch):
    """The GEMM entry point enqueues kernels only (no allocation, no memset, no host sync), so a
    caller may capture it: three fused calls are captured once and replayed with eager work in
    between; every replay must reproduce the eager result bit for bit."""
    monkeypatch.delenv("KRAKEN_AMD_GEMM_TILE", raising=False)
    monkeypatch.delenv("KRAKEN_AMD_GEMM_PEERS", raising=False)
    M, N, K, W, rank = 1024, 512, 512, 4, 1
    a, b, peers_full = mk(M, N, K, W - 1)
    bias = orc.randn_bf16((N,), 3, 0.02)
    ad, bd, bias_d = a.to(dev), b.to(dev), bias.to(dev)
    bt = bd.T.contiguous().T               # all_gather_matmul wants b.T contiguous
    pf = peers_full.to(dev)
    pb = pf[:, :M // W].contiguous()
    eager = (fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pf, bias=bias_d, out_dtype=BF16),
             fused.gemm_reduce_scatter(ad, bd, peers=pb, rank=rank),
             fused.all_gather_matmul(ad.view(W, M // W, K), bt, rank=rank)[1])
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(g, stream=side):
            got = (fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pf, bias=bias_d, out_dtype=BF16),
                   fused.gemm_reduce_scatter(ad, bd, peers=pb, rank=rank),
                   fused.all_gather_matmul(ad.view(W, M // W, K), bt, rank=rank)[1])
    for rep in range(3):
        for t in got:
            t.zero_()                      # eager work between the replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        for e, r in zip(eager, got):
            assert torch.equal(e, r)


@pytest.mark.parametrize("peers_mode", ["epilogue", "mfma"])
@pytest.mark.parametrize("mfma", ["16", "32"])
def test_split_tiles_round_like_unsplit_tiles(dev, monkeypatch, peers_mode, mfma):
    """Tiles whose K loop is split (tail round, finished by a separate pass) and tiles of the main
    launch must round alike: with small-integer operands and peers and bias on a grid of 1/16
    every fp32 sum is exact whatever its order, so the split result has to equal the unsplit one
    bit for bit -- with peers and bias on a bf16 result, where rounding the product before or after
    the peers are added makes a visible difference."""
    M, N, K, P = 4352, 4096, 1024, 3          # 272 tiles of 256 x 256: 256 + 16 in the tail
    g = torch.Generator().manual_seed(5)
    a = torch.randint(-3, 4, (M, K), generator=g).to(BF16)
    b = torch.randint(-3, 4, (K, N), generator=g).to(BF16)
    peers = (torch.randint(-127, 128, (P, M, N), generator=g).float() / 16).to(BF16)
    bias = (torch.randint(-32, 33, (N,), generator=g).float() / 4).to(BF16)
    ad, bd, pd, biasd = a.to(dev), b.to(dev), peers.to(dev), bias.to(dev)
    monkeypatch.setenv("KRAKEN_AMD_GEMM_PEERS", peers_mode)
    monkeypatch.setenv("KRAKEN_AMD_GEMM_MFMA", mfma)
    res = {}
    for split in ("0", "3"):
        monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", split)
        res[split] = [
            fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd, out_dtype=BF16),
            fused.gemm_one_shot_all_reduce_fused(ad, bd, bias=biasd, out_dtype=BF16),
            fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=pd, bias=biasd),
            fused.gemm_reduce_scatter(ad, bd, peers=pd[:1, : M // 2].contiguous(), rank=1, world_size=2),
        ]
    for x, y in zip(res["0"], res["3"]):
        assert torch.equal(x, y)
    # the exact product is large enough for the two rounding orders to differ somewhere
    prod = a.float() @ b.float()
    once = (prod + peers.float().sum(0) + bias.float()).to(BF16)
    twice = (prod.to(BF16).float() + peers.float().sum(0) + bias.float()).to(BF16)
    assert not torch.equal(once, twice)


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (255, 272, 144), (257, 240, 1040), (300, 528, 2064), (2049, 4112, 272), (4096, 272, 1136)])
def test_fp8_kernel_ragged_shapes(dev, M, N, K, split):
    """kr_gemm_fp8_ws on sizes no tile divides: one row, one column block, a row or column more or less than a
    tile, every kind of last k-step (16, 32, 96, 112 of 128 k), one tile up to more than a round of them, with and
    without the split of the K loop.  Small integers and halves: every fp32 sum is exact, so all result types
    equal the exact product bit for bit; what lies between the rows (stride > K) must not be read."""
    fp8 = torch.float8_e4m3fn
    g = torch.Generator().manual_seed(M + N + K)
    lda, ldb = K + 16, K + 32
    a, b = torch.full((M, lda), 3.0).to(fp8), torch.full((N, ldb), 3.0).to(fp8)
    a[:, :K] = torch.randint(-2, 3, (M, K), generator=g).float().to(fp8)
    b[:, :K] = (torch.randint(-3, 4, (N, K), generator=g).float() * 0.5).to(fp8)
    ad, bd = a.to(dev), b.to(dev)
    exact = (ad[:, :K].float() @ bd[:, :K].float().T)          # small integers and halves: exact in fp32
    lib = _lib.load()
    stream = torch.cuda.current_stream(dev).cuda_stream
    need = lib.kr_gemm_fp8_workspace_bytes(M, N, K) if split else 0
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=dev)
    for kind, dtype in ((0, BF16), (1, torch.float32), (2, fp8)):
        out = torch.zeros(M + 1, N, dtype=torch.float32, device=dev).to(dtype)
        rc = lib.kr_gemm_fp8_ws(ad.data_ptr(), lda, bd.data_ptr(), ldb, M, N, K, out.data_ptr(), kind,
                                ws.data_ptr() if need else None, need, stream)
        assert rc == 0, _lib.strerror(rc)
        want = exact.clamp(-448.0, 448.0).to(fp8) if kind == 2 else exact.to(dtype)
        assert torch.equal(out[:M].float(), want.float()), (M, N, K, kind)
        assert (out[M].float() == 0).all()                     # nothing past the last row


# 256-column tiles; an odd number of k-steps; ragged K (last step 8 or 56 of 64) and N; 224-column tiles with an odd number
# of steps; one column panel, so that a tile copies all it reads
@pytest.mark.parametrize("W,m,N,K", [(8, 512, 4096, 256), (4, 1024, 4096, 320), (8, 512, 4104, 1032), (2, 2304, 4096, 696),
                                     (16, 256, 7168, 320), (8, 512, 7168, 384), (2, 16640, 256, 256)])
def test_gather_inside_the_product(dev, W, m, N, K):
    """kr_gather_matmul_bf16: the gathered matrix is the shards bit for bit, nothing is written behind it, and the product has
    the bits of the product of the gathered matrix and of the form with copies and flags; with shards in separate
    buffers, in one stack, and with a shard in its own place of the gathered matrix."""
    rank = W - 1
    g = torch.Generator().manual_seed(N + K)
    a = (torch.rand(W, m, K, generator=g) - 0.5).to(BF16).to(dev)
    bT = (torch.rand(N, K, generator=g) - 0.5).to(BF16).to(dev)
    assert _lib.load().kr_gather_matmul_direct(W, m, N, K) == 1
    full = a.reshape(W * m, K)
    _, want = fused.all_gather_matmul(a, bT.T, rank=rank, gather=False)
    torch.testing.assert_close(want[::97].float(), full[::97].float() @ bT.float().T, **TOL)
    shards = [t.clone() for t in a]
    mem = torch.full((W * m * K + 64,), 7.0, dtype=BF16, device=dev)
    a_out = mem[:W * m * K].view(W * m, K)
    progress = torch.full((W + 1,), 5, dtype=torch.int32, device=dev)
    got, c = fused.all_gather_matmul(shards, bT.T, a_out, progress, rank=rank)
    assert got is a_out and torch.equal(a_out, full) and (mem[W * m * K:] == 7.0).all()
    assert torch.equal(c, want) and progress.tolist() == [1] * W + [0]
    got, c = fused.all_gather_matmul(a, bT.T, rank=rank, gather=True)
    assert torch.equal(got, full) and torch.equal(c, want)
    got, c = fused.all_gather_matmul(shards, bT.T, rank=rank, copy_engine=True)       # copies and flags
    assert torch.equal(got, full) and torch.equal(c, want)
    a_out.zero_()
    a_out[rank * m:] = shards[rank]
    shards[rank] = a_out[rank * m:]
    got, c = fused.all_gather_matmul(shards, bT.T, a_out, rank=rank)
    assert torch.equal(got, full) and torch.equal(c, want)


@pytest.mark.parametrize("m,N,dtype", [(512, 4096, BF16), (5, 1024, BF16), (5, 1024, torch.float8_e4m3fn)])
def test_gathered_matrix_is_known_to_be_written(dev, m, N, dtype):
    """Autograd sees that the gathered matrix changed, whether the product or a launch in front of it gathers; shards
    that require a gradient take the side stream, whose copies are recorded, with that form's results."""
    W, K = 8, 256
    shards = [torch.randn(m, K, device=dev).to(dtype) for _ in range(W)]
    b = torch.randn(N, K, device=dev).to(dtype).T
    a_out = torch.zeros(W * m, K, device=dev).to(dtype)
    version = a_out._version
    fused.all_gather_matmul(shards, b, a_out)
    assert a_out._version > version
    if dtype == BF16:
        # (the product behind the flags; one behind a launch that gathers may add in another order)
        _, want = fused.all_gather_matmul(shards, b, copy_engine=True)
        followed = [t.clone().requires_grad_() for t in shards]
        got, c = fused.all_gather_matmul(followed, b)
        assert torch.equal(got, torch.cat(shards)) and torch.equal(c, want)


def test_gathers_of_any_form_are_known_to_autograd(dev):
    """Below the size up to which a gather is one launch: shards that require a gradient get it back from the gathered matrix, a
    matrix that is kept does not keep earlier gathers, and every other form marks it as written."""
    W, m, K, N = 4, 40, 256, 1024
    b = torch.randn(N, K, device=dev).to(BF16).T
    def shards(grad):
        return [torch.randn(m, K, device=dev).to(BF16).requires_grad_(grad) for _ in range(W)]
    calls = {"matmul": lambda s, out, **kw: fused.all_gather_matmul(s, b, out, **kw)[0], "gather": lambda s, out, **kw: comm.all_gather_w_progress(s, out, **kw)}
    for what, call in calls.items():
        kept, first, second = torch.empty(W * m, K, dtype=BF16, device=dev), shards(True), shards(True)
        for s in (first, second):
            got = call(s, kept)
            assert got is kept and torch.equal(got, torch.cat(s)) and got.grad_fn is not None, what
        weight = torch.randn(W * m, K, device=dev).to(BF16)
        kept.backward(weight)
        assert all(t.grad is None for t in first) and torch.equal(torch.cat([t.grad for t in second]), weight), what
        call(shards(False), kept)
        assert not kept.requires_grad, what
        with torch.no_grad():
            assert not call(shards(True), None).requires_grad, what
        # (a leaf takes no recorded copies)
        leaf = torch.empty(W * m, K, dtype=BF16, device=dev, requires_grad=True)
        version, s = leaf._version, shards(False)
        assert torch.equal(call(s, leaf), torch.cat(s)) and leaf._version > version, what
        out = torch.zeros(W * m, K, dtype=BF16, device=dev)
        for kw in ({}, {"copy_engine": True}):
            version, s = out._version, shards(False)
            assert torch.equal(call(s, out, **kw), torch.cat(s)) and out._version > version, (what, kw)


def test_gather_inside_the_product_is_for_shards_apart(dev):
    """A shard that lies in another one's place of the gathered matrix, and shards that are not 16-byte aligned, take the
    copies; shapes of few tiles, or whose shards are no whole tiles, as well."""
    from kraken_amd.fused.all_gather_matmul import _direct
    W, m, N, K = 8, 512, 4096, 256
    a_out, b = torch.zeros(W * m, K, dtype=BF16, device=dev), torch.zeros(N, K, dtype=BF16, device=dev).T
    size, base = m * K * 2, torch.zeros(W, m, K, dtype=BF16, device=dev).data_ptr()
    apart = [base + r * size for r in range(W)]
    assert _direct(apart, a_out, b, W, m, N, K)
    assert _direct([a_out.data_ptr()] + apart[1:], a_out, b, W, m, N, K)
    assert not _direct([a_out.data_ptr() + size] + apart[1:], a_out, b, W, m, N, K)
    assert not _direct([a_out.data_ptr() - 16] + apart[1:], a_out, b, W, m, N, K)
    assert not _direct([base + 8] + apart[1:], a_out, b, W, m, N, K)
    assert not _direct(apart, a_out, b, W, 500, N, K) and not _direct(apart, a_out, b, W, 256, 1024, K)


@pytest.mark.parametrize("m,N", [(40, 1024), (512, 4096)])
@pytest.mark.parametrize("grad", [False, True])
def test_gathers_hand_tangents_on(dev, monkeypatch, m, N, grad):
    """Forward mode: the gathered matrix has the shards' tangents, and none of an earlier gather, also where the product or one launch would gather."""
    import torch.autograd.forward_ad as fw
    W, K = 8, 256
    b = torch.randn(N, K, device=dev).to(BF16).T
    shards, tangents = ([torch.randn(m, K, device=dev).to(BF16) for _ in range(W)] for _ in range(2))
    calls = (lambda s, out: fused.all_gather_matmul(s, b, out)[0], comm.all_gather_w_progress)
    # (the tangent is memory of the caller's stream: no copy runs on another one)
    monkeypatch.setattr(importlib.import_module("kraken_amd.comm.copy_engine_all_gather"), "_get_backend_stream", lambda dev: 1 / 0)
    with fw.dual_level(), torch.set_grad_enabled(grad):
        duals = [fw.make_dual(s, t) if r != 2 else s for r, (s, t) in enumerate(zip(shards, tangents))]
        for call in calls:
            out = torch.zeros(W * m, K, dtype=BF16, device=dev)
            primal, tangent = fw.unpack_dual(call(duals, out))
            assert torch.equal(primal, torch.cat(shards))
            assert torch.equal(tangent, torch.cat([t if r != 2 else torch.zeros_like(t) for r, t in enumerate(tangents)]))
            assert not fw.unpack_dual(call(shards, out)).tangent.any()
        sent = fw.make_dual(torch.zeros(2, 8, N, dtype=BF16, device=dev), torch.ones(2, 8, N, dtype=BF16, device=dev))
        fused.gemm_reduce_scatter_ce_persistent(shards[0][:16], b, peers=torch.zeros(1, 8, N, dtype=BF16, device=dev), rank=1, sent=sent)
        assert not fw.unpack_dual(sent).tangent[0].any()


@pytest.mark.parametrize("m,N,K,dtype", [(40, 264, 256, BF16), (512, 4096, 256, BF16), (512, 1024, 128, torch.float8_e4m3fn), (6, 48, 48, torch.float8_e4m3fn)])
@pytest.mark.parametrize("copy_engine", [False, True])
def test_shards_in_each_others_places_are_gathered_whole(dev, m, N, K, dtype, copy_engine):
    """Shards that lie in the gathered matrix, rotated by one place, one of them across two: every row comes out as the shard
    held it at the call, and so does the product.  One shard in its own place, one outside."""
    W, rank = 4, 1
    b = torch.randn(N, K, device=dev).to(dtype).T
    rows = torch.randn(W * m, K, device=dev).to(dtype)
    for places in ((1, 2, 3, 0), (0, 2, 1.5, None), (2.5, 0.5, None, 3)):
        a_out = rows.clone()
        shards = [rows[:m].clone() if p is None else a_out[int(p * m):int(p * m) + m] for p in places]
        full = torch.cat([s.view(torch.uint8) for s in shards]).view(dtype)
        _, want = fused.all_gather_matmul(full.view(W, m, K), b, gather=False)
        got, c = fused.all_gather_matmul(shards, b, a_out, rank=rank, copy_engine=copy_engine)
        assert got is a_out and torch.equal(got.view(torch.uint8), full.view(torch.uint8)), places
        torch.testing.assert_close(c.float(), want.float(), rtol=2e-2 if dtype == BF16 else 0.13, atol=2e-2)
        if dtype == BF16:
            a_out.copy_(rows)
            assert torch.equal(comm.all_gather_w_progress(shards, a_out, rank=rank, copy_engine=copy_engine), full), places


@pytest.mark.parametrize("plan", [None, 0, 3, 4000, 5001, 6000, 7002])
@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (255, 272, 112), (257, 528, 1040), (300, 1040, 528), (513, 816, 384)])
def test_fp8_wide_kernel_shapes(dev, monkeypatch, M, N, K, plan):
    """kr_gemm_fp8_wide_ws on sizes no tile divides, by its own choice of tiles, with 256-column tiles only, with every K
    loop in three parts, and with narrow tiles of every width behind 0, 1 or 2 panels of 256 columns; odd and even
    numbers of k-steps, the last one full or not.  Small integers and halves: every fp32 sum is exact, the fp8 result is the
    rounded product (saturated where it is large, NaN in the row of a NaN); what lies between the rows is not read."""
    fp8 = torch.float8_e4m3fn
    g = torch.Generator().manual_seed(M + N + K)
    lda, ldb = K + 16, K + 32
    a, b = torch.full((M, lda), float("nan")).to(fp8), torch.full((N, ldb), float("nan")).to(fp8)
    a[:, :K] = torch.randint(-2, 3, (M, K), generator=g).float().to(fp8)
    b[:, :K] = (torch.randint(-3, 4, (N, K), generator=g).float() * 0.5).to(fp8)
    a[0, :K], b[0, :K] = 4.0, 16.0
    ad, bd = a.to(dev), b.to(dev)
    want = (ad[:, :K].float() @ bd[:, :K].float().T).clamp(-448.0, 448.0)
    if M > 1:
        ad[M - 1, K - 1] = float("nan")
        want[M - 1] = float("nan")
    if plan is not None:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_W8", str(plan))
    lib = _lib.load()
    ws = torch.empty(4 * -(-M // 256) * -(-N // 256) * 256 * 256 * 4, dtype=torch.uint8, device=dev)
    out = torch.zeros(M + 1, N, dtype=torch.float32, device=dev).to(fp8)
    rc = lib.kr_gemm_fp8_wide_ws(ad.data_ptr(), lda, bd.data_ptr(), ldb, M, N, K, out.data_ptr(), M // 2, ws.data_ptr(), ws.numel(),
                                 torch.cuda.current_stream(dev).cuda_stream)
    assert rc == 0, _lib.strerror(rc)
    assert torch.equal(torch.nan_to_num(out[:M].float(), nan=1000.0), torch.nan_to_num(want.to(fp8).float(), nan=1000.0))
    assert (out[M].float() == 0).all()                     # nothing past the last row


def test_fp8_wide_kernel_widens_every_code(dev):
    """Each of the 256 e4m3 codes on both sides of a product with 1.0: the conversion on the way to the matrix cores is
    exact, subnormals, both zeros and NaN included."""
    fp8 = torch.float8_e4m3fn
    codes = torch.arange(256, dtype=torch.uint8).repeat_interleave(1).view(256, 1)
    x = torch.zeros(256, 128, dtype=torch.uint8)
    x[torch.arange(256), torch.arange(256) % 128] = codes[:, 0]      # row r: code r at k = r % 128
    ones = torch.full((16, 128), 1.0).to(fp8)
    lib, stream = _lib.load(), torch.cuda.current_stream(dev).cuda_stream
    xd, od = x.to(dev).view(fp8), ones.to(dev)
    want = codes.view(fp8).float().expand(256, 16)
    for a, b, w in ((xd, od, want), (od, xd, want.T)):
        out = torch.empty(a.shape[0], b.shape[0], dtype=fp8, device=dev)
        assert lib.kr_gemm_fp8_wide_ws(a.data_ptr(), 128, b.data_ptr(), 128, a.shape[0], b.shape[0], 128, out.data_ptr(), 0, None, 0, stream) == 0
        assert torch.equal(torch.nan_to_num(out.cpu().float(), nan=1000.0), torch.nan_to_num(w, nan=1000.0))


@pytest.mark.parametrize("gather", [False, True])
@pytest.mark.parametrize("m,K,N", [(250, 144, 528), (33, 208, 4112), (256, 144, 512), (250, 128, 512)])
def test_all_gather_matmul_fp8_ragged_sums_keep_their_bits(dev, m, K, N, gather):
    """fp8 shapes that are no whole 256 x 256 x 128 tiles: the fp32 sums are exact, so the fp8 result is the rounded
    64-bit product in every element.  Operands N(0, 1) and N(0, 0.25) in e4m3 are multiples of 2^-9, their products
    of 2^-18, and with sum |a||b| below 2^6 every partial sum has at most 24 bits, whatever the order."""
    fp8 = torch.float8_e4m3fn
    W = 8
    g = torch.Generator().manual_seed(m + K + N)
    a = torch.randn(W, m, K, generator=g).to(fp8)
    bT = (torch.randn(N, K, generator=g) * 0.25).to(fp8)
    a2, b2 = a.reshape(W * m, K).double(), bT.double().T
    assert (a2.abs() @ b2.abs()).max() < 64.0
    want = (a2 @ b2).float().to(fp8)
    shards = [t.to(dev) for t in a] if gather else a.to(dev)
    a_out, c = fused.all_gather_matmul(shards, bT.to(dev).T, rank=2, gather=gather)
    assert torch.equal(a_out.cpu().view(torch.uint8), a.reshape(W * m, K).view(torch.uint8))
    assert torch.equal(c.cpu().float(), want.float()), int((c.cpu().float() != want.float()).sum())


@pytest.mark.parametrize("m,K,N,kwargs", [(256, 1024, 768, {"fp8_kernel": False}), (32, 64, 272, {}), (256, 112, 512, {})])
def test_all_gather_matmul_fp8_widened_behind_the_gather(dev, m, K, N, kwargs):
    """gather=True where the product is widened to bf16: whole tiles with fp8_kernel=False, and a K below one k-step.
    Small integers and halves: every fp32 sum is exact, the fp8 result is the rounded product."""
    fp8 = torch.float8_e4m3fn
    W = 8
    g = torch.Generator().manual_seed(m + K)
    a = torch.randint(-2, 3, (W, m, K), generator=g).float().to(fp8)
    bT = (torch.randint(-3, 4, (N, K), generator=g).float() * 0.5).to(fp8)
    want = (a.reshape(W * m, K).float() @ bT.float().T).clamp(-448.0, 448.0).to(fp8)
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    a_out, c = fused.all_gather_matmul(a.to(dev), bT.to(dev).T, None, progress, rank=3, gather=True, **kwargs)
    assert torch.equal(a_out.cpu().view(torch.uint8), a.reshape(W * m, K).view(torch.uint8))
    assert progress.tolist() == [1] * W
    assert torch.equal(c.cpu().float(), want.float())


@pytest.mark.parametrize("m,K,N", [(125, 144, 528), (64, 2064, 272), (256, 1136, 272)])
def test_all_gather_matmul_fp8_ragged_entry(dev, m, K, N):
    """kr_all_gather_matmul_fp8_ragged with chunks that have arrived (every flag is set before the launch) and the local
    shard in a buffer of its own: the bits of the exact product of small integers and halves."""
    fp8 = torch.float8_e4m3fn
    W, rank = 4, 1
    g = torch.Generator().manual_seed(K)
    a = torch.randint(-2, 3, (W * m, K), generator=g).float().to(fp8)
    bT = (torch.randint(-3, 4, (N, K), generator=g).float() * 0.5).to(fp8)
    want = a.float() @ bT.float().T
    ad, bd = a.to(dev), bT.to(dev)
    local = ad[rank * m:(rank + 1) * m].clone()
    if m % 256 == 0:
        ad[rank * m:(rank + 1) * m].zero_()    # (tiles that lie in the local shard read their rows from it)
    flags = torch.ones(W, dtype=torch.int32, device=dev)
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    out = torch.empty(W * m, N, dtype=torch.float32, device=dev)
    rc = _lib.load().kr_all_gather_matmul_fp8_ragged(
        ad.data_ptr(), K, local.data_ptr(), K, bd.data_ptr(), K, W * m, N, K, W, rank, 1, flags.data_ptr(), 0,
        status.data_ptr(), out.data_ptr(), 1, torch.cuda.current_stream(dev).cuda_stream)
    assert rc == 0, _lib.strerror(rc)
    assert torch.equal(out.cpu(), want) and status.item() == 0


@pytest.mark.parametrize("K", [128, 2048, 16384])
def test_fp8_kernel_precision_of_the_sums(dev, K):
    """The fp8 instruction keeps about 16 bits of a sum: against 64 bits the fp32 result is off by 1.1e-5 to 1.5e-5 in
    the 2-norm (measured, K = 128 .. 16384, N(0, 1) x N(0, 0.25)); the bound is twice that, 2^-15.  In one pass and
    with the K loop split."""
    fp8 = torch.float8_e4m3fn
    M, N = 512, 768
    g = torch.Generator().manual_seed(K)
    a = torch.randn(M, K, generator=g).to(fp8)
    bT = (torch.randn(N, K, generator=g) * 0.25).to(fp8)
    exact = a.double() @ bT.double().T
    ad, bd = a.to(dev), bT.to(dev)
    lib = _lib.load()
    need = lib.kr_gemm_fp8_workspace_bytes(M, N, K)
    assert (need > 0) == (K > 128)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device=dev)
    for nbytes in {0, need}:
        out = torch.empty(M, N, dtype=torch.float32, device=dev)
        rc = lib.kr_gemm_fp8_ws(ad.data_ptr(), K, bd.data_ptr(), K, M, N, K, out.data_ptr(), 1, ws.data_ptr() if nbytes else None,
                                nbytes, torch.cuda.current_stream(dev).cuda_stream)
        assert rc == 0, _lib.strerror(rc)
        err = ((out.cpu().double() - exact).norm() / exact.norm()).item()
        assert err <= 2.0 ** -15, (nbytes, err)


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K", [(256, 256, 72), (512, 264, 120), (264, 512, 328), (511, 520, 1016)])
def test_large_tile_kernel_last_k_step_not_full(dev, monkeypatch, M, N, K, b_t):
    """The 256 x 256 kernel with K no multiple of its k-step: the pieces past K of the last step are zeros whatever
    follows them in memory (here NaN: strides larger than the rows, and the next row otherwise)."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "256")
    g = torch.Generator().manual_seed(K)
    a = torch.full((M, K + 64), float("nan"))
    b = torch.full((N, K + 64) if b_t else (K + 64, N), float("nan"))
    a[:, :K] = torch.randn(M, K, generator=g)
    if b_t:
        b[:, :K] = torch.randn(N, K, generator=g) * 0.05
    else:
        b[:K] = torch.randn(K, N, generator=g) * 0.05
    ad, bd = a.to(BF16).to(dev)[:, :K], b.to(BF16).to(dev)
    bd = bd[:, :K].T if b_t else bd[:K]
    out = fused.gemm_one_shot_all_reduce_fused(ad, bd)
    torch.testing.assert_close(out.cpu(), ad.float().cpu() @ bd.float().cpu(), rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (1, 8, 72), (130, 136, 128), (129, 264, 320), (256, 128, 392), (131, 1032, 1000)])
def test_deep_ring_kernel_edges(dev, monkeypatch, M, N, K, b_t):
    """The 128 x 128 kernel with a five-stage ring (KRAKEN_AMD_GEMM_KS=1): one k-step, fewer steps than stages, one
    more, many; a last step that is not full; ragged rows and columns; a number of tiles 8 does not divide; one
    part and three.  Small integers: every fp32 sum is exact, so all of them equal the product bit for bit; what
    lies between the rows (NaN) is not read."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TILE", "128")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_KS", "1")
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.full((M, K + 8), float("nan"))
    b = torch.full((N, K + 8) if b_t else (K, N + 8), float("nan"))
    a[:, :K] = torch.randint(-4, 5, (M, K), generator=g).float()
    bk = torch.randint(-4, 5, (K, N), generator=g).float()
    if b_t:
        b[:, :K] = bk.T
    else:
        b[:, :N] = bk
    ad, bd = a.to(BF16).to(dev)[:, :K], b.to(BF16).to(dev)
    bd = bd[:, :K].T if b_t else bd[:, :N]
    want = a[:, :K] @ bk
    for splits in ("1", "3"):
        monkeypatch.setenv("KRAKEN_AMD_GEMM_SPLITK", splits)
        assert torch.equal(fused.gemm_one_shot_all_reduce_fused(ad, bd).cpu(), want), splits


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (1, 8, 8), (130, 136, 40), (129, 264, 96), (256, 128, 328), (131, 1032, 1000)])
def test_fp32_operands_split_in_registers(dev, monkeypatch, M, N, K, b_t):
    """kr_gemm_reduce_f32_ws: one k-step down to 8 k, last steps of every kind (a stage missing, half a stage), fewer
    steps than the ring has stages, ragged rows and columns, one part and three, with peers and bias.  Exact part:
    integers up to 2^11 times integers up to 8 -- hi and lo parts are exact, every partial sum is below 2^24 --
    equal the product bit for bit.  Random part: within 2^-15 of sum |a||b| of the double-precision product (the
    dropped a_lo b_lo is below 2^-18, the rounding of lo below 2^-18 twice, fp32 sums of K terms below K 2^-24)."""
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.full((M, K + 4), float("nan"))
    b = torch.full((N, K + 4) if b_t else (K, N + 4), float("nan"))

    def operands(av, bv):
        a[:, :K] = av
        if b_t:
            b[:, :K] = bv.T
        else:
            b[:, :N] = bv
        bd = b.to(dev)
        return a.to(dev)[:, :K], bd[:, :K].T if b_t else bd[:, :N]

    peers = torch.randint(-8, 9, (3, M, N), generator=g).to(BF16)
    bias = torch.randint(-8, 9, (N,), generator=g).to(BF16)
    av = torch.randint(-2047, 2048, (M, K), generator=g).float()
    bv = torch.randint(-8, 9, (K, N), generator=g).float()
    exact = av.double() @ bv.double() + peers.double().sum(0) + bias.double()
    assert K * 2047 * 8 < 1 << 24
    ar, br = torch.randn(M, K, generator=g), torch.randn(K, N, generator=g)
    for splits in ("1", "3"):
        monkeypatch.setenv("KRAKEN_AMD_GEMM_SPLITK", splits)
        ad, bd = operands(av, bv)
        out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=peers.to(dev), bias=bias.to(dev))
        assert torch.equal(out.cpu().double(), exact), splits
        ad, bd = operands(ar, br)
        out = fused.gemm_one_shot_all_reduce_fused(ad, bd).cpu().double()
        assert ((out - ar.double() @ br.double()).abs() <= 2.0 ** -15 * (ar.abs().double() @ br.abs().double())).all(), splits


@pytest.mark.parametrize("pairs", [None, "0"])
@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K", [(2304, 4096, 256), (2200, 4104, 72), (256, 4096, 260)])
def test_fp32_operands_split_in_a_pass(dev, monkeypatch, M, N, K, b_t, pairs):
    """More than 512 tiles of 128 x 128: the operands are split by a pass of their own, as pairs, and with KRAKEN_AMD_GEMM_PAIRS=0, and for a K
    that is no multiple of 8, into three blocks that are multiplied as a bf16 product of 3K.  Integers up to 2^11 (hi and lo
    parts exact) times integers up to 8, every sum below 2^24: exact."""
    from kraken_amd.fused import _gemm
    if pairs is not None:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_PAIRS", pairs)
    g = torch.Generator().manual_seed(K)
    a = torch.randint(-2047, 2048, (M, K), generator=g).float().to(dev)
    b = torch.randint(-8, 9, (K, N), generator=g).float().to(dev)
    assert K * 2047 * 8 < 1 << 24
    bd = b.T.contiguous().T if b_t else b
    assert not _gemm.fp32_direct(a, bd) and _gemm.fp32_pairs(a, bd) == (pairs is None and K % 8 == 0)
    assert torch.equal(fused.gemm_one_shot_all_reduce_fused(a, bd), a @ b)


@pytest.mark.parametrize("wide", ["a", "b", "b_t"])
def test_fp32_operands_with_very_wide_rows(dev, wide):
    """fp32 operands that are slices of matrices with rows of 4.2 million elements: 128 such rows reach past the 2 GiB that
    the kernel which splits in registers can address, so they take the split pass.  Small integers: the product is exact."""
    M, N, K, ld = 72, 136, 64, 4_200_000
    rows = {"a": M, "b": K, "b_t": N}[wide]
    big = torch.zeros(rows, ld, dtype=torch.float32, device=dev)     # 1.1 to 2.3 GB
    g = torch.Generator().manual_seed(ld)
    a = torch.randint(-8, 9, (M, K), generator=g).float().to(dev)
    b = torch.randint(-8, 9, (K, N), generator=g).float().to(dev)
    want = a @ b
    part = big[:, 16:16 + {"a": K, "b": N, "b_t": K}[wide]]
    part.copy_({"a": a, "b": b, "b_t": b.T}[wide])
    if wide == "a":
        a = part
    else:
        b = part if wide == "b" else part.T
    assert torch.equal(fused.gemm_one_shot_all_reduce_fused(a, b), want)


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (16, 32, 64), (17, 40, 72), (32, 264, 520), (33, 136, 1000), (64, 1032, 1096)])
def test_few_rows_kernel(dev, monkeypatch, M, N, K, b_t, fp32):
    """gemm_skinny_kernel: every number of columns per workgroup, one part and three, one row up to 64, fewer units of
    64 k than wavefronts and more than they keep in flight, a last unit that is not full, columns no width divides,
    eight or more peers than are requested early, a bias, a band that is part of the rows.  Small integers (fp32
    operands: up to 2^11, hi and lo parts exact): every fp32 sum is exact, results equal the product bit for bit; what
    lies between the rows (NaN) is not read."""
    g = torch.Generator().manual_seed(M + N + K)
    dt = torch.float32 if fp32 else BF16
    a = torch.full((M, K + 8), float("nan"))
    b = torch.full((N, K + 8) if b_t else (K, N + 8), float("nan"))
    big = 2047 if fp32 else 4
    a[:, :K] = torch.randint(-big, big + 1, (M, K), generator=g).float()
    bk = torch.randint(-4, 5, (K, N), generator=g).float()
    if b_t:
        b[:, :K] = bk.T
    else:
        b[:, :N] = bk
    ad, bd = a.to(dt).to(dev)[:, :K], b.to(dt).to(dev)
    bd = bd[:, :K].T if b_t else bd[:, :N]
    product = a[:, :K] @ bk
    peers = torch.randint(-8, 9, (9, M, N), generator=g).to(BF16)
    bias = torch.randint(-8, 9, (N,), generator=g).to(BF16)
    for cb in (1, 2) if fp32 else (1, 2, 4):
        for splits in (1, 5):
            monkeypatch.setenv("KRAKEN_AMD_GEMM_SKINNY", str(100 * cb + splits))
            _lib.reload_env()
            out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=peers.to(dev), bias=bias.to(dev))
            assert torch.equal(out.cpu(), product + peers.float().sum(0) + bias.float()), (cb, splits)
            if not fp32 and M % 2 == 0:
                c = torch.zeros(M, N, dtype=BF16, device=dev)
                half = M // 2
                out = fused.gemm_reduce_scatter(ad, bd, peers=peers[:1, :half].contiguous().to(dev), rank=1, c_scratch=c)
                want = product.to(BF16)
                assert torch.equal(out.cpu(), (want[half:].float() + peers[0, :half].float()).to(BF16)), (cb, splits)
                assert torch.equal(c.cpu()[:half], want[:half]), (cb, splits)
    plan = _lib.gemm_plan(M, N, K, b_t)
    assert fp32 or plan["kernel"] == "gemm_skinny_kernel"
    monkeypatch.delenv("KRAKEN_AMD_GEMM_SKINNY")
    _lib.reload_env()
    out = fused.gemm_one_shot_all_reduce_fused(ad, bd, peers=peers.to(dev), bias=bias.to(dev))
    assert torch.equal(out.cpu(), product + peers.float().sum(0) + bias.float())


@pytest.mark.parametrize("W,splits,rank,nbytes", [(1, 1, 0, 16), (2, 1, 1, 16384), (3, 2, 0, 16400), (8, 3, 5, 49136), (16, 1, 15, 1 << 20)])
def test_gather_chunks(dev, W, splits, rank, nbytes):
    """kr_gather_chunks: one vector, a piece exactly, a piece and one vector, a piece short of one, more pieces than
    workgroups; all bytes arrive, nothing behind them is written, and every flag reads 1."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(nbytes)
    src = [torch.randint(0, 256, (splits * nbytes + 64,), generator=g, dtype=torch.uint8).to(dev) for _ in range(W)]
    dst = torch.full((W * splits * nbytes + 64,), 7, dtype=torch.uint8, device=dev)
    flags = torch.zeros(W * splits + 1, dtype=torch.int32, device=dev)
    table = (ctypes.c_void_p * W)(*[t.data_ptr() for t in src])
    rc = lib.kr_gather_chunks(table, W, splits, rank, nbytes, dst.data_ptr(), flags.data_ptr(), torch.cuda.current_stream(dev).cuda_stream)
    assert rc == 0, _lib.strerror(rc)
    assert flags.tolist() == [1] * (W * splits) + [0]
    assert torch.equal(dst[:W * splits * nbytes], torch.cat([t[:splits * nbytes] for t in src]))
    assert (dst[W * splits * nbytes:] == 7).all()


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("shape", [(0, 64), (6, 0)])
def test_gather_of_empty_shards_sets_its_flags(dev, shape, splits):
    """Chunks without bytes have arrived as soon as the gather runs: every flag reads 1, the others stay."""
    W = 4
    for shards in (torch.empty(W, *shape, dtype=BF16, device=dev), [torch.empty(shape, dtype=BF16, device=dev) for _ in range(W)]):
        progress = torch.zeros(W * splits + 1, dtype=torch.int32, device=dev)
        out = torch.empty(W * shape[0], shape[1], dtype=BF16, device=dev)
        assert comm.all_gather_w_progress(shards, out, progress, splits_per_rank=splits, rank=1) is out
        assert progress.tolist() == [1] * (W * splits) + [0]


@pytest.mark.parametrize("rows", [8, 520])      # a run of one piece per chunk, several runs
def test_gather_over_the_flags_of_an_earlier_one(dev, rows):
    """The chunked copy with flags that are still 1 from the gather before: the new shards arrive and the flags end at 1."""
    from kraken_amd.comm.copy_engine_all_gather import _copy_engine_all_gather_w_progress
    W, K = 4, 1024
    progress = torch.zeros(W, dtype=torch.int32, device=dev)
    out = torch.empty(W * rows, K, dtype=BF16, device=dev)
    for seed in range(3):
        shards = orc.randn_bf16((W, rows, K), seed).to(dev)
        torch.cuda.current_stream(dev).wait_stream(_copy_engine_all_gather_w_progress(out, shards, progress, 1, rank=2))
        assert torch.equal(out, shards.view(W * rows, K))
        assert progress.tolist() == [1] * W


def _small_integers(shape, seed, density, dev):
    g = torch.Generator(device=dev).manual_seed(seed)
    v = torch.randint(-1, 2, shape, generator=g, device=dev).to(BF16)
    return v * (torch.rand(shape, generator=g, device=dev) < density)


@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K,W,rank", [
    (4136, 4104, 4104, 2, 1),      # 289 tiles, all edges ragged, a K that is no multiple of 64: the tiles beyond the first round in parts
    (4400, 4096, 4160, 8, 7),      # 288 tiles, ragged rows only
    (2312, 4104, 264, 8, 3),       # the band's tiles ahead of the others, both its edges inside a tile
    (2312, 4104, 264, 8, 7),       # ... the last band, which ends with the matrix
    (3000, 3000, 72, 4, 0), (6144, 3072, 128, 2, 1), (2560, 4096, 64, 2, 0),
    (4104, 4096, 3080, 4, 2), (5632, 4224, 8192, 8, 0),      # 272 tiles, 16 in four parts; 374 tiles, 118 in two
    (520, 2056, 4112, 8, 3), (736, 3608, 4144, 8, 7), (504, 6656, 4112, 8, 0), (944, 2960, 6944, 2, 1)])      # few tiles, all in parts, the last k-step not full
def test_reduce_scatter_of_many_tiles(dev, M, N, K, W, rank, b_t):
    """More than 128 tiles of 256 x 256, and fewer that are all in parts.  Operands of -1, 0, 1 (a sixth of b's are not zero, a twelfth with a
    K above 5000; two thirds of a's): every sum is an integer far below 256 (six standard deviations at K = 4160: 129, at
    K = 8192: 128; seven peers 7), so product, sum and rounding are exact."""
    a, b = _small_integers((M, K), 1, 1.0, dev), _small_integers((K, N), 2, 0.25 if K <= 5000 else 0.125, dev)
    peers = _small_integers((W - 1, M // W, N), 3, 1.0, dev)
    c = torch.full((M, N), float("nan"), dtype=BF16, device=dev)
    out = fused.gemm_reduce_scatter(a, b.T.contiguous().T if b_t else b, peers=peers, rank=rank, c_scratch=c)
    want = a.float() @ b.float()
    lo, hi = rank * (M // W), (rank + 1) * (M // W)
    assert torch.equal(out.float(), want[lo:hi] + peers.float().sum(0))
    assert torch.equal(c[:lo].float(), want[:lo]) and torch.equal(c[hi:].float(), want[hi:])
    assert bool(c[lo:hi].isnan().all())      # the band's own rows are not the scratch's


@pytest.mark.parametrize("P", [0, 1, 7])
@pytest.mark.parametrize("M,N,K", [(4136, 4104, 4096), (4352, 4096, 4096), (4360, 4096, 3072)])
def test_rounding_of_tiles_in_parts_behind_whole_rounds(dev, M, N, K, P):
    """289 and 272 tiles, the last ones in parts: with a workspace the bits are those without.  Integers, so every sum is exact, of
    nine bits and more, so rounding once and twice differ: tiles that are whole and in the band add peers and bias in fp32, the others
    round the product first."""
    g = torch.Generator(device=dev).manual_seed(M + P)
    rnd = lambda *s: torch.randint(-3, 4, s, generator=g, device=dev).to(BF16)      # noqa: E731
    a, b, bias, peers = rnd(M, K), rnd(K, N), rnd(N), rnd(max(P, 1), M, N)
    lib, stream = _lib.load(), _lib.current_stream(dev)
    need = lib.kr_gemm_workspace_bytes(M, N, K)
    assert _lib.gemm_plan(M, N, K, False, P, M, workspace_bytes=need)["tail_tiles"] == (33 if N == 4104 else 16 if K == 4096 else 32)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    outs = [torch.empty(M, N, dtype=BF16, device=dev) for _ in range(2)]
    args = [a.data_ptr(), K, 1, b.data_ptr(), N, 1, M, N, K, peers.data_ptr(), P, M * N, bias.data_ptr(), 0, M, None]
    assert lib.kr_gemm_reduce_bf16(*args, outs[0].data_ptr(), 0, 0, stream) == 0
    assert lib.kr_gemm_reduce_ws_bf16(*args, outs[1].data_ptr(), 0, 0, ws.data_ptr(), need, stream) == 0
    product, added = a.float() @ b.float(), peers[:P].float().sum(0) + bias.float()
    want = (product.to(BF16).float() + added).to(BF16)
    m, n = M // 256 * 256, N // 256 * 256
    want[:m, :n] = (product + added)[:m, :n].to(BF16)
    assert torch.equal(outs[0], want)
    assert torch.equal(outs[1], want)


@pytest.mark.parametrize("P", [1, 2, 3, 4, 7, 8])
@pytest.mark.parametrize("M,N,K", [(264, 264, 64), (520, 328, 136), (90, 8, 64), (383, 640, 72)])
def test_epilogue_at_the_edges(dev, tile, M, N, K, P):
    """Peers added in the epilogue, for waves that are in the band, partly in it and outside, at the edges of the matrix, with
    bf16 and fp32 results: integers as above, exact."""
    a, b, bias = _small_integers((M, K), 1, 1.0, dev), _small_integers((K, N), 2, 0.25, dev), _small_integers((N,), 4, 1.0, dev)
    peers = _small_integers((P, M, N), 3, 1.0, dev)
    want = a.float() @ b.float()
    for dtype in (BF16, torch.float32):
        out = fused.gemm_one_shot_all_reduce_fused(a, b, peers=peers, bias=bias, out_dtype=dtype)
        assert out.dtype == dtype and torch.equal(out.float(), want + peers.float().sum(0) + bias.float())
    W = P + 1
    rows = M // W
    a, want = a[:rows * W], want[:rows * W]
    for rank in (0, W // 2, W - 1):
        c = torch.full((rows * W, N), float("nan"), dtype=BF16, device=dev)
        out = fused.gemm_reduce_scatter(a, b, peers=peers[:, :rows].contiguous(), rank=rank, c_scratch=c)
        lo, hi = rank * rows, (rank + 1) * rows
        assert torch.equal(out.float(), want[lo:hi] + peers[:, :rows].float().sum(0))
        assert torch.equal(c[:lo].float(), want[:lo]) and torch.equal(c[hi:].float(), want[hi:]) and bool(c[lo:hi].isnan().all())


@pytest.mark.parametrize("P", [1, 2, 4, 5, 6])
@pytest.mark.parametrize("M,N", [(264, 328), (3, 8)])
def test_epilogue_of_peers_that_are_not_there(dev, tile, M, N, P):
    """Fewer peers than the epilogue's form has room for: what it reads in their place (values that are not finite here) is not added."""
    a, b, peers = _small_integers((M, 72), 1, 1.0, dev), _small_integers((72, N), 2, 0.25, dev), _small_integers((P, M, N), 3, 1.0, dev)
    peers[0, 0, :8] = torch.tensor([float("inf"), float("-inf"), 1, 2, 3, 4, 5, float("inf")])
    for dtype in (BF16, torch.float32):
        out = fused.gemm_one_shot_all_reduce_fused(a, b, peers=peers, out_dtype=dtype)
        assert torch.equal(out.float(), a.float() @ b.float() + peers.float().sum(0))


@pytest.mark.parametrize("parts", [0, 3])
@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("M,N,K,W,rank", [(65, 8, 8, 1, 0), (128, 264, 40, 2, 1), (256, 256, 64, 2, 0), (260, 520, 72, 4, 2), (520, 328, 1000, 8, 7)])
def test_fp32_operands_as_pairs(dev, monkeypatch, M, N, K, W, rank, b_t, parts):
    """kr_split_pairs_fp32 and kr_gemm_reduce_pairs_ws: a last group of 32 k that is not full (its zeros are written into a
    buffer of NaN), edges of the 64 x 64 blocks of the pass and of the tiles, K loops in one pass and in three parts, operands whose rows
    lie apart.  Integers up to 2^11 (hi and lo parts exact) times integers up to 8, every sum below 2^24: exact."""
    monkeypatch.setenv("KRAKEN_AMD_GEMM_PAIRS", "1")
    monkeypatch.setenv("KRAKEN_AMD_GEMM_TAILSPLIT", str(parts))
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.full((M, K + 4), float("nan"), device=dev)
    b = torch.full((N, K + 4) if b_t else (K, N + 4), float("nan"), device=dev)
    a[:, :K] = torch.randint(-2047, 2048, (M, K), generator=g).float()
    bv = torch.randint(-8, 9, (K, N), generator=g).float().to(dev)
    if b_t:
        b[:, :K] = bv.T
        b = b[:, :K].T
    else:
        b[:, :N] = bv
        b = b[:, :N]
    a = a[:, :K]
    assert K * 2047 * 8 < 1 << 24
    from kraken_amd.fused import _gemm
    assert _gemm.fp32_pairs(a, b)
    rows = M // W
    peers = torch.randint(-8, 9, (W - 1, M, N), generator=g).to(BF16).to(dev) if W > 1 else None
    bias = torch.randint(-8, 9, (N,), generator=g).to(BF16).to(dev)
    want = a.contiguous().double() @ bv.double()
    for poison in range(2):     # (the allocator hands the pass a buffer of the last call's values)
        out = fused.gemm_one_shot_all_reduce_fused(a, b, peers=peers, bias=bias)
        assert torch.equal(out.double(), want + (peers.double().sum(0) if W > 1 else 0) + bias.double())
        torch.full(((M + N) * (K // 32 + 1) * 32,), float("nan"), device=dev)
    if M % W == 0 and W > 1:
        c = torch.zeros((M, N), dtype=BF16, device=dev)
        mine = peers[:, :rows].contiguous()
        out = fused.gemm_reduce_scatter(a, b, peers=mine, rank=rank, c_scratch=c)
        lo, hi = rank * rows, (rank + 1) * rows
        assert out.dtype == torch.float32 and torch.equal(out.double(), want[lo:hi] + mine.double().sum(0))
        assert torch.equal(c[:lo], want[:lo].to(BF16)) and torch.equal(c[hi:], want[hi:].to(BF16))


@pytest.mark.parametrize("where", [None, "mfma", "first", "last", "epilogue"])
@pytest.mark.parametrize("M,N,K,W,rank", [
    (2304, 4096, 128, 2, 1),       # 144 whole tiles, the band starts inside a tile
    (2312, 4104, 192, 8, 3),       # ragged rows and columns
    (2304, 4096, 72, 3, 0),        # a K that is no multiple of 64: peers in the epilogue whatever is asked for
    (4136, 4104, 1024, 2, 0),      # 289 tiles, 33 of them in parts behind a whole round
    (4352, 4096, 1024, 8, 7)])     # 272, 16 in parts
def test_fp32_operands_as_pairs_in_whole_rounds(dev, monkeypatch, M, N, K, W, rank, where):
    """More than 512 tiles of 128 x 128, the route of such calls: peers on the matrix cores, ahead of the k loop and behind it, and in the
    epilogue.  Integers as above, exact."""
    from kraken_amd.fused import _gemm
    if where is not None:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_PEERS", where)
    g = torch.Generator(device=dev).manual_seed(M + K)
    rnd = lambda v, *s: torch.randint(-v, v + 1, s, generator=g, device=dev)      # noqa: E731
    a, b, bias = rnd(2047, M, K).float(), rnd(8, N, K).float(), rnd(8, N).to(BF16)
    peers = rnd(8, W - 1, M, N).to(BF16)
    assert K * 2047 * 8 + W * 8 < 1 << 24 and _gemm.fp32_pairs(a, b.T)
    assert (_lib.load().kr_gemm_pairs_workspace_bytes(M, N, K) > 0) == (K == 1024)
    want = a.double() @ b.double().T
    out = fused.gemm_one_shot_all_reduce_fused(a, b.T, peers=peers, bias=bias)
    assert out.dtype == torch.float32 and torch.equal(out.double(), want + peers.double().sum(0) + bias.double())
    mine, c = peers[:, :M // W].contiguous(), torch.full((M, N), float("nan"), dtype=BF16, device=dev)
    out = fused.gemm_reduce_scatter(a, b.T, peers=mine, rank=rank, c_scratch=c)
    lo, hi = rank * (M // W), (rank + 1) * (M // W)
    assert torch.equal(out.double(), want[lo:hi] + mine.double().sum(0))
    assert torch.equal(c[:lo], want[:lo].to(BF16)) and torch.equal(c[hi:], want[hi:].to(BF16)) and bool(c[lo:hi].isnan().all())


@pytest.mark.parametrize("fp8", [False, True])
def test_products_without_memory_for_their_workspace(dev, fp8):
    """A last round that runs in parts, and an fp8 product of few tiles in parts: in one pass where the parts have no room."""
    from kraken_amd.fused import _gemm
    lib, dt = _lib.load(), torch.float8_e4m3fn if fp8 else BF16
    M, N, K = (264, 4112, 8192) if fp8 else (4136, 4104, 4096)
    need = lib.kr_gemm_fp8_wide_workspace_bytes(M, N, K) if fp8 else lib.kr_gemm_workspace_bytes(M, N, K)
    a, b = _small_integers((M, K), 1, 1.0, dev), _small_integers((N, K), 2, 0.25, dev)
    want = (a.float() @ b.float().T).to(dt)
    a, b, out = a.cpu().to(dt), b.cpu().to(dt), M * N * a.element_size()
    kept = dict(_gemm._workspaces)
    try:
        for listed in (False, True):      # the native form and the general path
            _gemm._workspaces.clear()
            torch.cuda.empty_cache()
            ad, bd = a.to(dev), b.to(dev)
            room = torch.cuda.memory_reserved(dev) + out + need // 2
            torch.cuda.set_per_process_memory_fraction(room / torch.cuda.mem_get_info(dev)[1], dev)
            with pytest.raises(torch.OutOfMemoryError):
                torch.empty(need + out, dtype=torch.uint8, device=dev)
            if fp8:
                c = fused.all_gather_matmul(list(ad.view(1, M, K)) if listed else ad.view(1, M, K), bd.T)[1]
            else:
                c = fused.gemm_one_shot_all_reduce_fused(ad, bd.T, peers=[] if listed else None, out_dtype=BF16)
            torch.cuda.set_per_process_memory_fraction(1.0, dev)
            assert torch.equal(c.float(), want.float())
            del c, ad, bd
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
        _gemm._workspaces.update(kept)


@pytest.mark.parametrize("b_t", [False, True])
def test_fp32_operands_as_pairs_without_memory_for_them(dev, b_t):
    """A shape whose parts take 165 MB that are not to be had: it runs in registers.  Integers as above, exact."""
    from kraken_amd.fused import _gemm
    M, N, K = 1316, 3136, 9280
    a, b = _small_integers((M, K), 1, 1.0, dev).float(), _small_integers((K, N), 2, 1.0, dev).float()
    want = a @ b
    peers = _small_integers((1, M, N), 3, 1.0, dev)
    a, b = a.cpu(), (b.T.contiguous().T if b_t else b).cpu()
    torch.cuda.empty_cache()
    a, b = a.to(dev), b.to(dev)      # (in memory of their own: no cached rest of it holds the parts)
    assert _gemm.fp32_pairs(a, b)
    total = torch.cuda.mem_get_info(dev)[1]
    try:
        for given in (peers, list(peers)):      # the native form and the general path
            _gemm._workspaces.clear()
            torch.cuda.empty_cache()
            torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + (100 << 20)) / total, dev)
            with pytest.raises(torch.OutOfMemoryError):
                torch.empty(4 * (M + N) * K, dtype=torch.uint8, device=dev)
            out = fused.gemm_one_shot_all_reduce_fused(a, b, peers=given)
            torch.cuda.set_per_process_memory_fraction(1.0, dev)
            assert torch.equal(out, want + peers[0].float())
            del out
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)


def test_fp32_operands_and_a_peer_that_is_not_finite(dev):
    """More than 512 tiles of 128 x 128 and a K of 64: the infinity of one element of a peer stays in that element."""
    M, N, K = 2304, 4096, 64
    a, b = _small_integers((M, K), 1, 1.0, dev).float(), _small_integers((K, N), 2, 1.0, dev).float()
    peers = _small_integers((1, M, N), 3, 1.0, dev)
    peers[0, 300, 1029] = float("inf")
    want = a @ b + peers[0].float()
    for given in (peers, list(peers)):      # the native form and the general path
        assert torch.equal(fused.gemm_one_shot_all_reduce_fused(a, b, peers=given), want)


@pytest.mark.parametrize("form", [None, 101, 201, 401, 102, 203, 404])
@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (16, 48, 112), (17, 272, 128), (32, 80, 1040), (33, 1040, 144), (64, 304, 2064)])
def test_fp8_few_rows_kernel(dev, monkeypatch, M, N, K, form):
    """fp8 operands with at most 64 rows: units of k that are not full, columns past N, one part of K and several.  Operands of -1, 0,
    1: the sums are whole numbers below 2^24, so the result is their one rounding to fp8; poisoned beyond the sizes."""
    if form is not None:
        monkeypatch.setenv("KRAKEN_AMD_GEMM_SKINNY", str(form))
    fp8 = torch.float8_e4m3fn
    big = torch.full((M + N + 2, K + 32), float("nan"), device=dev).to(fp8)
    a, b = _small_integers((M, K), 1, 1.0, dev), _small_integers((N, K), 2, 1.0, dev)
    big[:M, :K], big[M + 1:-1, :K] = a.to(fp8), b.to(fp8)
    lib = _lib.load()
    out = torch.full((M + 1, N), float("nan"), device=dev).to(fp8)
    ws = torch.full((lib.kr_gemm_fp8_wide_workspace_bytes(M, N, K) + 4 * 4 * M * N,), 255, dtype=torch.uint8, device=dev)
    rc = lib.kr_gemm_fp8_wide_ws(big.data_ptr(), K + 32, big[M + 1:].data_ptr(), K + 32, M, N, K, out.data_ptr(), 0, ws.data_ptr(), ws.numel(),
                                 _lib.current_stream(torch.device("cuda", torch.cuda.current_device())))
    assert rc == 0
    want = (a.float() @ b.float().T).clamp(-448, 448).to(fp8)
    assert torch.equal(out[:M].view(torch.uint8), want.view(torch.uint8)) and bool(out[M:].float().isnan().all())
    whole = fused.all_gather_matmul(a.to(fp8).view(1, M, K), b.to(fp8).T)[1]
    assert torch.equal(whole.float(), want.float())      # (-0 and 0)
