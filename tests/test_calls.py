"""The native form of the common calls (csrc/calls.cpp) against the general path: the same results and the same errors,
whichever of the two takes a call."""
import itertools

import pytest
import torch

from kraken_amd import _lib, comm, fused
from oracle import oracle as orc

BF16 = torch.bfloat16
FUNCTIONS = {"all_reduce": 1, "all_reduce_bias": 5, "two_shot_share": 4, "two_shot_bias": 8, "reduce_rms_norm": 7, "rms_norm": 3, "gemm": 9}


_General = _lib._NoCalls      # stands in for the native module: takes no call


@pytest.mark.parametrize("fault", ["missing", "no library", "another torch"])
def test_without_the_native_form_every_call_takes_the_general_path(monkeypatch, tmp_path, fault):
    other = tmp_path / "_calls.so"
    if fault == "no library":
        other.write_bytes(b"\x7fELF")
    monkeypatch.setattr(_lib, "_calls", None)
    if fault == "another torch":
        monkeypatch.setattr(_lib.torch, "__version__", "0.0")
    else:
        monkeypatch.setattr(_lib, "CALLS_PATH", other)
    with pytest.warns(RuntimeWarning, match="not usable"):
        native = _lib.calls()
    assert native is _lib.calls() and all(getattr(native, name)(*[None] * n) is None for name, n in FUNCTIONS.items())
    with pytest.raises(RuntimeError, match="run on a HIP device only"):
        comm.one_shot_all_reduce(torch.zeros(2, 8, dtype=BF16))


@pytest.mark.parametrize("name", FUNCTIONS)
def test_what_is_not_of_the_common_form_is_left_to_the_general_path(name):
    fn, n = getattr(_lib.calls(), name), FUNCTIONS[name]
    host = torch.zeros(2, 8, dtype=BF16)
    sub = host.as_subclass(type("Sub", (torch.Tensor,), {}))
    for value in (host, sub, None, [host, host], 1, 1.0, "x", host.to_sparse(), host.to("meta")):
        for count in (n, n - 1, n + 1, 0):
            assert fn(*[value] * count) is None


def test_world_size_of_the_reduce_scatter_is_a_number_of_ranks(monkeypatch):
    """What the general path refuses is not taken by the native one: ``world_size`` absent or the number of ranks, nothing else."""
    class Takes:
        def gemm(self, *args):
            return args

    monkeypatch.setattr(_lib, "_calls", Takes())
    a, b, peers, c = (torch.zeros(*s, dtype=BF16) for s in ((8, 16), (16, 8), (3, 2, 8), (8, 8)))
    for kw, taken in (({}, True), ({"world_size": 4}, True), ({"world_size": None}, False), ({"world_size": 4.0}, False), ({"world_size": 2}, False)):
        try:
            out = fused.gemm_reduce_scatter(a, b, peers=peers, c_scratch=c, **kw)
        except Exception:        # noqa: BLE001 (the general path's)
            out = None
        assert isinstance(out, tuple) == taken, kw


def _both(monkeypatch, call):
    """``call()`` as it is and through the general path: two results, or two exceptions' types."""
    got = []
    for general in (False, True):
        with monkeypatch.context() as m:
            if general:
                _lib.calls()
                m.setattr(_lib, "_calls", _General())
            try:
                got.append(call())
            except Exception as e:        # noqa: BLE001 (the type is what is compared)
                got.append(type(e))
    return got


def _same(monkeypatch, call, what):
    one, two = _both(monkeypatch, call)
    if isinstance(one, type) or isinstance(two, type):
        assert one is two, (what, one, two)
        return False
    for x, y in zip(one, two, strict=True):
        assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype, what
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8)), what
    return True


def _stacks(dev, W, rows, D):
    """Forms a stack comes in: contiguous, with room behind each slice, strided, transposed, a list, of another type, misaligned."""
    g = torch.Generator(device=dev).manual_seed(W * rows + D)
    big = torch.randn(W, rows + 2, D, generator=g, device=dev).to(BF16)
    plain = big[:, :rows].contiguous()
    yield "plain", plain
    yield "roomy", big
    yield "strided", big[:, :rows]
    yield "transposed", plain.transpose(1, 2).contiguous().transpose(1, 2)
    yield "list", list(plain)
    yield "fp32", plain.float()
    yield "misaligned", torch.cat([torch.zeros(1, dtype=BF16, device=dev), plain.flatten()])[1:].view(W, rows, D)
    yield "flat", plain.view(W, rows * D)


@pytest.mark.gpu
def test_the_common_form_is_taken(dev, monkeypatch):
    """Every native function takes its call in the common form, with each of its options, and gives the general path's bits
    (that both paths agree, above and below, says nothing of which one ran)."""
    g = torch.Generator(device=dev).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(BF16)      # noqa: E731
    native, W, rows, D, rank = _lib.calls(), 8, 16, 8192, 3
    stack, x, full, vec, w = rnd(W, rows, D), rnd(rows, D), rnd(rows, D), rnd(D), rnd(D)
    reduced = orc.reduce(stack.cpu())

    def own(t):                     # the stack with one rank's slice replaced
        s = stack.clone()
        s[rank] = t
        return s

    assert torch.equal(native.all_reduce(stack).cpu(), reduced)
    for xv, bias in itertools.product((None, x), (None, full, vec)):
        source = (stack if xv is None else own(xv)).cpu()
        b32 = None if bias is None else bias.cpu()
        y = torch.zeros(rows, D, dtype=BF16, device=dev)
        assert native.all_reduce_bias(stack, xv, bias, y, rank) is True
        want = torch.zeros_like(y)
        fused.one_shot_all_reduce_bias(list(own(xv) if xv is not None else stack), None, bias, want)
        assert torch.equal(y, want) and (bias is not None or torch.equal(y.cpu(), orc.reduce(source)))
        assert native.reduce_rms_norm(stack, xv, bias, w, y, 1e-5, rank) is True
        zero = torch.zeros(D, dtype=BF16) if b32 is None else b32
        torch.testing.assert_close(y.cpu(), orc.reduce_bias_rms_norm(source, zero, w.cpu()), rtol=2e-2, atol=2e-2)
    assert torch.equal(native.two_shot_share(stack, rank, False, 2048).cpu(), reduced.view(W, rows // W, D)[rank])
    share = native.two_shot_share(stack, rank, True, 2048)
    blocks = reduced.view(-1, W, 2048)[:, rank].reshape(-1)
    assert torch.equal(share.cpu(), blocks)
    for xv, bias, striped in itertools.product((None, x), (None, full), (False, True)):
        out, want = torch.zeros(rows * D // W, dtype=BF16, device=dev), torch.zeros(rows * D // W, dtype=BF16, device=dev)
        assert native.two_shot_bias(stack, xv, bias, out, 2048, rank, striped, rows * D) is True
        fused.two_shot_all_reduce_bias(list(own(xv) if xv is not None else stack), None, bias, want, BLOCK_SIZE=2048, rank=rank,
                                       layout="striped" if striped else "rows", numel=rows * D)
        assert torch.equal(out, want)
    with monkeypatch.context() as m:
        m.setattr(_lib, "_calls", _General())
        normed = fused.rms_norm(x, w, 1e-5)
    assert torch.equal(native.rms_norm(x, w, 1e-5), normed)
    M, N, K = 64, 256, 512
    for b in (rnd(K, N), rnd(N, K).T):
        a, peers, c = rnd(M, K), rnd(3, M // 4, N), torch.zeros(M, N, dtype=BF16, device=dev)
        for fp32 in (False, True):
            out = native.gemm(a, b, None, vec[:N], None, 0, M, fp32, 0)
            assert out.dtype == (torch.float32 if fp32 else BF16)
            torch.testing.assert_close(out.float(), a.float() @ b.float() + vec[:N].float(), rtol=2e-2, atol=2e-2)
        out, want = native.gemm(a, b, peers, None, c, M // 4, M // 4, False, M // 4), torch.zeros_like(c)
        assert torch.equal(out, fused.gemm_reduce_scatter(a, b, peers=list(peers), rank=1, c_scratch=want)) and torch.equal(c, want)


@pytest.mark.gpu
@pytest.mark.parametrize("W,rows,D", [(1, 3, 64), (2, 8, 1024), (3, 6, 136), (8, 16, 8192), (8, 8, 512), (16, 4, 72), (17, 2, 64), (4, 5, 20), (2, 1, 4096)])
def test_row_calls_take_both_paths_alike(dev, monkeypatch, W, rows, D):
    g = torch.Generator(device=dev).manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(BF16)      # noqa: E731
    x, full, vec, w = rnd(rows, D), rnd(rows, D), rnd(D), rnd(D)
    xs = {"none": None, "own": x, "wide": rnd(rows, 2 * D)[:, :D], "off": rnd(rows * D + 1)[1:].view(rows, D), "fp32": x.float(), "short": x[:1],
          "column": rnd(D, rows).T}
    ok = 0
    for (form, stack), (xf, xv), (bf, bias), rank in itertools.product(
            _stacks(dev, W, rows, D), xs.items(), {"none": None, "full": full, "vec": vec, "bad": rnd(D + 8)}.items(), (0, W - 1, W)):
        if rank == W and (xf, bf) != ("none", "vec"):
            continue
        what = (form, xf, bf, rank)

        def rms():
            y = torch.empty(rows, D, dtype=BF16, device=dev)
            fused.one_shot_all_reduce_bias_rms_norm(stack, xv, bias, w, y, rank=rank)
            return [y]

        def one_shot():
            out = torch.empty(rows, D, dtype=BF16, device=dev)
            fused.one_shot_all_reduce_bias(stack, xv, bias, out, rank=rank)
            return [out]

        ok += _same(monkeypatch, rms, ("rms", what)) + _same(monkeypatch, one_shot, ("bias", what))
        for layout, block, numel in (("rows", 48 * W, None), ("striped", 48 * W, rows * D), ("striped", 8 * W, None), ("rows", 16, rows * D), ("other", 16, None)):
            sizes = {rows * D, rows * D // W, rows * D // W + 8}
            if layout == "striped" and rows * D % 8 == 0 and W <= 16 and rank < W:
                sizes.add(max(8, _lib.load().kr_striped_share_numel(rows * D, W, block, rank)))
            for size in sizes:
                def two_shot():
                    out = torch.zeros(size, dtype=BF16, device=dev)
                    return [fused.two_shot_all_reduce_bias(stack, xv, bias, out, BLOCK_SIZE=block, rank=rank, layout=layout, numel=numel)]

                _same(monkeypatch, two_shot, ("two-shot", what, layout, block, numel, size))
        if (xf, bf) == ("none", "none"):
            ok += _same(monkeypatch, lambda: [comm.one_shot_all_reduce(stack)], what)
            for layout, block in (("rows", 2048), ("striped", 8 * W), ("striped", 2048), ("other", 8 * W)):
                _same(monkeypatch, lambda: [comm.two_shot_all_reduce(stack, rank=rank, layout=layout, BLOCK_SIZE=block)], (what, layout, block))
    assert (ok > 0) == (W <= 16 and D % 8 == 0)
    for v in (x, xs["wide"], xs["off"], xs["column"], x.float(), x[:0]):
        for wv in (w, w[:-8], w.float(), rnd(2 * D)[::2]):
            _same(monkeypatch, lambda: [fused.rms_norm(v, wv)], ("rms_norm", v.shape, v.stride(), wv.shape))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,W", [(8, 256, 128, 4), (1, 64, 72, 2), (512, 264, 4096, 8), (40, 20, 64, 2), (24, 64, 60, 3), (32, 128, 64, 1)])
def test_products_take_both_paths_alike(dev, monkeypatch, M, N, K, W):
    g = torch.Generator(device=dev).manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(BF16)      # noqa: E731
    a, b = rnd(M, K), rnd(K, N)
    left = {"plain": a, "wide": rnd(M, 2 * K)[:, :K], "column": rnd(K, M).T, "off": rnd(M * K + 1)[1:].view(M, K), "fp32": a.float(), "odd": rnd(M, K + 1)[:, :K]}
    right = {"rows": b, "columns": rnd(N, K).T, "wide": rnd(K, 2 * N)[:, :N], "off": rnd(K * N + 1)[1:].view(K, N), "fp32": b.float(), "long": rnd(K + 8, N)}
    ok = 0
    for (af, av), (bf, bv) in itertools.product(left.items(), right.items()):
        for rows, fn in ((M, "ar"), (M // W, "rs")):
            whole = rnd(max(W - 1, 1), rows, N)
            for pf, pv in {"none": None, "stack": whole[:W - 1], "list": list(whole[:W - 1]), "gap": rnd(max(W - 1, 1), rows + 1, N)[:W - 1, :rows],
                           "fp32": whole.float(), "flat": whole.flatten(1)}.items():
                what = (af, bf, fn, pf)
                if fn == "ar":
                    for bias, dtype in ((None, BF16), (rnd(N), torch.float32), (rnd(N).float(), BF16), (rnd(1, N), BF16), (None, torch.float16)):
                        ok += _same(monkeypatch, lambda: [fused.gemm_one_shot_all_reduce_fused(av, bv, peers=pv, bias=bias, out_dtype=dtype)], (what, dtype))
                else:
                    for rank, kw in ((0, {}), (W - 1, {"world_size": W}), (W, {}), (0, {"world_size": W + 1})):
                        def rs():
                            c = torch.zeros(M, N, dtype=BF16, device=dev)
                            return [fused.gemm_reduce_scatter(av, bv, peers=pv, rank=rank, c_scratch=c, **kw), c]

                        ok += _same(monkeypatch, rs, (what, rank, kw))
    assert (ok > 0) == (N % 8 == 0)


@pytest.mark.gpu
def test_native_calls_run_on_the_current_stream_and_in_a_graph(dev):
    stack, w = orc.make_stack(8, (16, 8192)).to(dev), torch.ones(8192, dtype=BF16, device=dev)
    y = torch.empty(16, 8192, dtype=BF16, device=dev)
    want = orc.reduce_bias_rms_norm(stack.cpu(), torch.zeros(8192, dtype=BF16), w.cpu())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fused.one_shot_all_reduce_bias_rms_norm(stack, None, None, w, y)     # the stream's workspace, outside the capture
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            fused.one_shot_all_reduce_bias_rms_norm(stack, None, None, w, y)
            out = comm.one_shot_all_reduce(stack)
    for _ in range(3):
        y.zero_()
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        torch.testing.assert_close(y.cpu(), want, rtol=2e-2, atol=2e-2)
        assert torch.equal(out.cpu(), orc.reduce(stack.cpu()))


def test_workspace_that_is_not_to_be_had(monkeypatch):
    from kraken_amd.fused import _gemm

    def full(*args, **kwargs):
        raise torch.OutOfMemoryError("full")

    small = torch.zeros(8, dtype=torch.uint8)
    monkeypatch.setattr(_gemm, "_workspaces", {(0, 5): small})
    monkeypatch.setattr(torch, "empty", full)
    assert _gemm.stream_workspace(0, 16, 5) is small and _gemm.stream_workspace(0, 16, 7) is None
    assert _gemm._workspaces == {(0, 5): small}


@pytest.mark.parametrize("kw,native", [({}, True), ({"gather": True}, True), ({"gather": False}, False), ({"gather": None}, None), ({"gather": 1}, None)])
def test_gather_as_it_is_named(monkeypatch, kw, native):
    """A mode that is named is taken by the native form only as True or False; the default is its own."""
    from kraken_amd.fused.all_gather_matmul import _common_form
    seen = []
    monkeypatch.setattr(_lib, "calls", lambda: type("Calls", (), {"gather_matmul": staticmethod(lambda *args: seen.append(args[6]))}))
    assert _common_form([torch.zeros(2, 8)], torch.zeros(8, 8), None, None, **kw) is None
    assert seen == ([] if native is None else [native])


@pytest.mark.parametrize("name,n", [("reduce_scatter_sent", 6), ("gather_matmul", 7)])
def test_overlap_calls_that_are_not_of_the_common_form(name, n):
    fn = getattr(_lib.calls(), name)
    host = torch.zeros(2, 8, dtype=BF16)
    for value in (host, None, [host, host], [], 1, 1.0, "x", host.to_sparse(), host.to("meta")):
        for count in (n, n - 1, n + 1, 0):
            assert fn(*[value] * count) is None


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,W", [(8, 16, 8, 4), (96, 264, 72, 8), (512, 1032, 200, 2), (24, 64, 64, 3), (2304, 4096, 64, 4)])
def test_fp32_products_are_taken(dev, monkeypatch, M, N, K, W):
    """fp32 operands: one native step for each kernel that splits them (few rows, in registers, as pairs), the general path's bits."""
    g = torch.Generator(device=dev).manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)      # noqa: E731
    native, a, bias = _lib.calls(), rnd(M, K), rnd(N).to(BF16)
    for b in (rnd(K, N), rnd(N, K).T, rnd(K, N + 4)[:, :N], rnd(N, K + 4)[:, :K].T):
        peers, c = rnd(W - 1, M // W, N).to(BF16), torch.zeros(M, N, dtype=BF16, device=dev)
        assert native.gemm(a, b, None, bias, None, 0, M, True, 0).dtype == torch.float32
        assert native.gemm(a, b, peers, None, c, 0, M // W, True, 0) is not None
        for dtype in (BF16, torch.float32):
            assert _same(monkeypatch, lambda: [fused.gemm_one_shot_all_reduce_fused(a, b, bias=bias, out_dtype=dtype)], (b.stride(), dtype))
        assert _same(monkeypatch, lambda: [fused.gemm_reduce_scatter(a, b, peers=peers, rank=W - 1, c_scratch=c), c.clone()], b.stride())
    for odd in (a[:, ::2], rnd(K, M).T, rnd(M * K + 1)[1:].view(M, K), a[:1].expand(M, K), a.double(), a.to(BF16)):
        b = rnd(odd.shape[1], N)
        _same(monkeypatch, lambda: [fused.gemm_one_shot_all_reduce_fused(odd, b)], (odd.dtype, odd.stride()))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,W", [(16, 16, 8, 2), (96, 264, 72, 8), (512, 1032, 200, 4), (2304, 4096, 64, 4)])
def test_reduce_scatter_with_destinations_takes_both_paths_alike(dev, monkeypatch, M, N, K, W):
    g = torch.Generator(device=dev).manual_seed(2)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(BF16)      # noqa: E731
    m, a = M // W, rnd(M, K)
    room = rnd(2 * W, m, N)
    peers = rnd(W - 1, m, N)
    sents = {"own": lambda: torch.zeros(W, m, N, dtype=BF16, device=dev), "list": lambda: list(torch.zeros(W, m, N, dtype=BF16, device=dev)),
             "grad": lambda: torch.zeros(W, m, N, dtype=BF16, device=dev, requires_grad=True), "short": lambda: torch.zeros(W - 1, m, N, dtype=BF16, device=dev),
             "spaced": lambda: torch.zeros(W, m + 1, N, dtype=BF16, device=dev)[:, :m], "none": lambda: None,
             "over the peers": lambda: room[1:W + 1]}
    taken = _lib.calls().reduce_scatter_sent(a, rnd(K, N), peers, sents["own"](), 1, True)
    assert taken.shape == (m, N)
    for bf, b in (("rows", rnd(K, N)), ("columns", rnd(N, K).T)):
        for sf, make in sents.items():
            for rank, kw in ((0, {}), (W - 1, {"fp32_acc": True}), (1, {"world_size": W}), (W, {}), (0, {"world_size": None}), (0, {"reduce_op": "avg"})):
                def run():
                    room[:W - 1].copy_(peers)
                    sent = make()
                    mine = room[:W - 1] if sf == "over the peers" else peers
                    versions = getattr(sent, "_version", None)
                    out = fused.gemm_reduce_scatter_ce_persistent(a, b, peers=mine, rank=rank, sent=sent, **kw)
                    assert sf != "own" or sent._version > versions
                    others = [] if sent is None else [t.detach().contiguous() for r, t in enumerate(sent) if r != rank]
                    return [out, *others]

                _same(monkeypatch, run, (bf, sf, rank, kw))


@pytest.mark.gpu
@pytest.mark.parametrize("m,N,K,W", [(1, 16, 16, 2), (12, 272, 144, 8), (256, 512, 128, 2), (250, 1040, 272, 3), (512, 4096, 256, 5), (4, 16, 16, 17), (4, 20, 24, 2)])
def test_gathered_products_take_both_paths_alike(dev, monkeypatch, m, N, K, W):
    g = torch.Generator(device=dev).manual_seed(4)
    fp8 = torch.float8_e4m3fn
    for dtype in (BF16, fp8):
        rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(dtype)      # noqa: E731
        stack = rnd(W, m, K)
        room = rnd(W + 1, m, K)
        forms = {"stack": stack, "list": [t.clone() for t in stack.unbind()], "tuple": tuple(stack.unbind()),
                 "columns": stack.view(torch.uint8 if dtype == fp8 else BF16).transpose(1, 2).contiguous().view(dtype).transpose(1, 2), "in the result": list(room[1:].unbind())}
        ok = 0
        for (form, shards), (bf, b) in itertools.product(forms.items(), {"columns": rnd(N, K).T, "wide": rnd(N, 2 * K)[:, :K].T, "rows": rnd(K, N)}.items()):
            for kw in ({}, {"gather": True}, {"gather": False}, {"gather": True, "rank": W - 1, "splits_per_rank": 2}, {"gather": True, "splits_per_rank": 3},
                       {"gather": True, "rank": W}, {"gather": 1}, {"gather": 0}, {"gather": None}):
                for given in ("both", "neither", "flags", "many flags", "small"):
                    def run():
                        a_out = None if given in ("neither", "flags") else room[:W].reshape(W * m, K) if form == "in the result" else torch.zeros(W * m, K, device=dev).to(dtype)
                        flags = None if given == "neither" else torch.full(((W if given == "small" else 3 * W + 5),), 7, dtype=torch.int32, device=dev)
                        if given == "flags" or given == "both":
                            flags = flags[:W * kw.get("splits_per_rank", 1)]
                        if form == "in the result":
                            room[1:].view(torch.uint8).copy_(stack.view(torch.uint8))
                        before = None if a_out is None else a_out._version
                        gathered, c = fused.all_gather_matmul(shards, b, a_out=a_out, progress=flags, **kw)
                        torch.cuda.synchronize()
                        assert a_out is None or kw.get("gather") is not True or gathered._version > before
                        return [gathered.contiguous(), c] + ([] if flags is None else [flags])

                    ok += _same(monkeypatch, run, (dtype, form, bf, kw, given))
        assert ok > 0 or N % 16 != 0
        if W <= 16 and N % 16 == 0:
            a_out, flags = torch.zeros(W * m, K, device=dev).to(dtype), torch.zeros(W, dtype=torch.int32, device=dev)
            b = rnd(N, K).T
            assert _lib.calls().gather_matmul(forms["list"], b, a_out, flags, 0, 1, True) is not None
            assert _lib.calls().gather_matmul(stack, b, None, None, 0, 1, False) is not None
            if dtype == BF16:     # what autograd follows is left to it
                forms["list"][0].requires_grad_()
                assert _lib.calls().gather_matmul(forms["list"], b, a_out, flags, 0, 1, True) is None
                with torch.no_grad():
                    assert _lib.calls().gather_matmul(forms["list"], b, a_out, flags, 0, 1, True) is not None
