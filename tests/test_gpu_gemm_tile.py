"""The small-tile forms of the wide GEMM (gemm_tile.inl): edges of the 64 / 128 tiles, one K-tile up to more K-tiles than the LDS pipelines
hold, strided operands, every epilogue, plain and hi/lo rows, against float64 products of the same bf16 operands.  Tolerances: fp32 results
3e-5 of the largest value (fp32 accumulation of <= 4096 products), bf16 results one ulp (2^-8)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# (M, N, K): what the rule makes of them (64 x 64, 64 x 128 and two-per-CU 128 x 128 tiles; 128 x 128 of eight waves for SwiGLU only); test_every_form has the rest
SHAPES = [(1, 4, 64), (63, 60, 128), (64, 64, 192), (65, 68, 256), (65, 3072, 320), (129, 132, 576), (200, 1028, 1024), (300, 3076, 512),
          (520, 2736, 1024), (1025, 1024, 1024), (1025, 3072, 256), (1409, 3200, 128), (2048, 3072, 192), (2100, 2052, 2048), (33, 32004, 64)]


def rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).abs().max() / (b.abs().max() + 1e-30))


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_forms(M, N, K):
    from ming_univision_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x, b = rnd(M, K), rnd(2 * N).to(torch.bfloat16)
    w = (rnd(2 * N, K) * K ** -0.5).to(torch.bfloat16)
    w1, b1 = w[:N].contiguous(), b[:N].contiguous()
    a2, a1 = ops.split_hilo(x), x.to(torch.bfloat16)
    wide = torch.zeros(M, K + 64, dtype=torch.bfloat16, device="cuda")       # rows with a stride of their own
    wide[:, :K] = a1
    for a, xr, hilo in ((a2, a2.double().sum(0), True), (a1, a1.double(), False)):
        both = xr @ w.double().T + b.double()
        ref = both[:, :N]
        lin = (lambda e, out=None: ops.gemm256(a2, w1, b1, e, out=out)) if hilo else (lambda e, out=None: ops.gemm_bf16(wide[:, :K], w1, b1, e, out=out))
        assert rel(lin("f32"), ref) < 3e-5
        acc = rnd(M, N + 4)
        base = acc.double().clone()
        lin("f32_resid", acc[:, :N]) if not hilo else ops.linear_hilo(a2, w1, b1, out=acc[:, :N], resid=True)
        assert rel(acc[:, :N], base[:, :N] + ref) < 3e-5 and torch.equal(acc[:, N:].double(), base[:, N:])
        if not hilo:
            assert rel(lin("bf16"), ref) < 2 ** -8
            assert rel(lin("bf16_gelu"), F.gelu(ref)) < 2 ** -8
        act = F.silu(both[:, :N]) * both[:, N:]
        if hilo:
            y = ops.gemm256_swiglu_split(a2, w, b)
            assert rel(y.double().sum(0), act) < 3e-5
            if K >= 256:
                assert rel(ops.gemm256_splitk(a2, w1, b1, 2).double().sum(0), ref) < 3e-5
        else:
            assert rel(ops.gemm256_swiglu(a1, w, b), act) < 2 ** -8



@pytest.fixture
def dev_lib():
    """The same code with the switches of mingnative_dev.h, in the place of the product library."""
    import ctypes
    import os
    from ming_univision_amd import _lib
    shipped = _lib.lib()
    handle = ctypes.CDLL(os.path.join(os.path.dirname(_lib.LIB_PATH), "libmingnative_dev.so"))
    for name, (res, args) in _lib.SYMBOLS.items():
        fn = getattr(handle, name)
        fn.restype, fn.argtypes = res, args
    _lib._lib = handle
    yield handle
    handle.mn_gemm_tile_tune(-1)
    _lib._lib = shipped


@pytest.mark.parametrize("form", [0, 1, 2, 3, 4])
def test_every_form(dev_lib, form):
    """Each tile form in turn (0: 256 x 256) on rows and columns that end inside its tiles, one to five K-tiles and more than its pipeline holds, and the activations in
    the epilogues with a tail that begins and ends inside a tile.  (Hi / lo rows have no form 4: the 256-tile kernel takes them.)"""
    dev_lib.mn_gemm_tile_tune(form)
    for M, N, K in ((1, 4, 64), (63, 60, 128), (65, 68, 192), (129, 132, 256), (257, 260, 320), (300, 516, 64), (200, 1028, 1024)):
        test_forms(M, N, K)
    for M, width, ff in ((65, 64, 96), (130, 128, 516), (300, 64, 1028)):
        test_activations_in_the_products_epilogue(M, width, ff)


def test_activations_on_the_large_tiles():
    """A prompt wide enough for the 256 x 256 tiles under the rule."""
    test_activations_in_the_products_epilogue(2048, 2048, 4096)


@pytest.mark.parametrize("M,N,K", [(16380, 1020, 1024), (4100, 4100, 2048)])
def test_rule_picks_the_large_tiles(M, N, K):
    """A round of 256 x 256 tiles and more with ragged last rows and columns, every epilogue."""
    test_forms(M, N, K)


@pytest.mark.parametrize("M,width,ff", [(65, 64, 96), (130, 128, 516), (300, 64, 1028), (70, 128, 102)])
def test_activations_in_the_products_epilogue(M, width, ff):
    """Prompt rows whose hidden units leave the product activated (squared relu beside the mixers' projections; gelu(gate) x up), against the same
    layers in fp32 arithmetic, where every activation is a launch of its own; a hidden width that is no multiple of 4 keeps the launch."""
    from ming_univision_amd.configuration import DaberaxConfig, ZuzenexConfig
    from ming_univision_amd.daberax import DaberaxDecoder
    from ming_univision_amd.zuzenex import ZuzenexDecoder
    mlp = dict(kind="dense", ff=ff)
    zu = ZuzenexConfig(width=width, vocab=40, norm=dict(eps=1e-6), layers=[
        dict(type="attention", mixer=dict(heads=2, kv_heads=1, dim=20, vdim=32, scale=0.2), mlp=mlp),
        dict(type="lightning", mixer=dict(heads=2, dim=16, vdim=16, decay=[0.9, 0.99]), mlp=mlp)])
    da = DaberaxConfig(width=width, vocab=40, norm=dict(eps=1e-6), token_side=dict(dim=8), layers=[
        dict(type="attention", mixer=dict(heads=2, kv_heads=1, dim=16, vdim=32, scale=0.2), mlp=mlp)])
    ids = torch.arange(M, device="cuda") % 40
    for cls, cfg in ((ZuzenexDecoder, zu), (DaberaxDecoder, da)):
        out = [cls.synthetic(cfg, "cuda", t_max=M + 1, n_seq=1, arith=a).prefill(ids) for a in ("bf16", "f32")]
        assert rel(out[0], out[1]) < 3e-2                # two layers of products on bf16 operands (2^-9 each, some ten of them, of values up to 4 rms)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("M", [65, 130, 300])
def test_output_product_in_slabs(M, off):
    """A hybrid prompt pass whose joined output product comes as split-K slabs, summed by the next layer's norm, the final norm and the trace's sum: against the
    same layers in fp32 arithmetic; off: the caller's result and the norms' gains lie where no vector access may go."""
    from ming_univision_amd._lib import lib
    from ming_univision_amd.configuration import ZuzenexConfig
    from ming_univision_amd.sequences import rows_of_spans
    from ming_univision_amd.zuzenex import ZuzenexDecoder
    W, ff = 128, 448
    assert lib().mn_gemm256_plan_ksplit(M, W, 64 + ff, 0) > 1
    mlp = dict(kind="dense", ff=ff)
    cfg = ZuzenexConfig(width=W, vocab=40, norm=dict(eps=1e-6), layers=[
        dict(type="attention", mixer=dict(heads=2, kv_heads=1, dim=32, vdim=32, scale=0.2), mlp=mlp),
        dict(type="lightning", mixer=dict(heads=2, dim=32, vdim=32, decay=[0.9, 0.99]), mlp=mlp)])
    got = []
    for arith in ("bf16", "f32"):
        dec = ZuzenexDecoder.synthetic(cfg, "cuda", t_max=M, n_seq=1, arith=arith)
        x = dec.embed(torch.arange(M, device="cuda") % 40)
        tabs = {k: torch.from_numpy(v).cuda() for k, v in rows_of_spans([(0, M, 0)], dec.block_rows, dec.chunk_rows).items() if k != "max_len"}
        keep = []
        if off and arith == "bf16":
            for s, name in [(dec._layers[0], "norm1"), (dec._layers[1], "norm1"), (dec.struct, "final_w")]:
                src = next(t for t in dec._keep if t.data_ptr() == getattr(s, name))
                keep.append(torch.empty(W + 1, dtype=torch.bfloat16, device="cuda"))
                keep[-1][1:] = src
                setattr(s, name, keep[-1].data_ptr() + 2)
        buf = torch.full((M * W + 2,), 7.0, device="cuda")
        out, trace = buf[off:off + M * W].view(M, W), torch.empty(dec.n_trace, M, W, device="cuda")
        for tr in (None, trace):
            dec.step(x, tabs["row_seq"], tabs["row_slot"], tabs["row_back"], blk_tab=tabs["blk_tab"], max_len=M, out=out, trace=tr, chunk_tab=tabs["chunk_tab"])
            got.append(out.clone())
        got.append(trace)
        assert bool((buf[off + M * W:] == 7.0).all())
    assert rel(got[0], got[1]) < 1e-6                    # the trace takes the slabs in a launch of its own
    for a, b in zip(got[:3], got[3:]):
        assert rel(a, b) < 3e-2                          # (as above)


@pytest.mark.parametrize("M,n", [(1, 4), (3, 1020), (5, 1024), (2, 1028), (70, 2048), (4, 4100), (3, 8192), (2, 8196), (3, 33)])
def test_residual_and_rms_rows(M, n):
    """x += m y, RMS norm: rows in registers and the walking form (odd or very wide rows)."""
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    g = torch.Generator(device="cuda").manual_seed(M + n)
    x, y = torch.randn(M, n + 4, generator=g, device="cuda"), torch.randn(M, n + 8, generator=g, device="cuda")
    w = (1 + 0.1 * torch.randn(n, generator=g, device="cuda")).to(torch.bfloat16)
    o, o16 = torch.full((M, n + 4), 5.0, device="cuda"), torch.full((M, n + 4), 5.0, device="cuda").to(torch.bfloat16)
    for yy in (y, None):
        ref = x[:, :n].double() + (0.5 * y[:, :n].double() if yy is not None else 0)
        nrm = ref / torch.sqrt((ref * ref).mean(-1, keepdim=True) + 1e-5) * w.double()
        check(lib().mn_axpy_rms_rows(ptr(x), n + 4, ptr(yy), n + 8, 0.5, ptr(w), 1e-5, ptr(o), n + 4, ptr(o16), n + 4, M, n, current_stream()), "axpy")
        assert rel(x[:, :n], ref) < 1e-6 and rel(o[:, :n], nrm) < 2e-6 and rel(o16[:, :n], nrm) < 2 ** -8
        assert bool((o[:, n:] == 5).all()) and bool((o16[:, n:] == 5).all())


@pytest.mark.parametrize("T,H,d,e", [(65, 2, 16, 16), (100, 3, 20, 36), (1000, 2, 128, 128), (2100, 1, 64, 100), (70, 2, 6, 10)])
def test_lightning_scan(T, H, d, e):
    """The chunked recurrence around its batches of 16 chunks, two sequences in one pass (one continuing), vector and scalar staging, against the
    recurrence in float64."""
    import numpy as np
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    from ming_univision_amd.sequences import rows_of_spans
    L, g = lib(), torch.Generator().manual_seed(T + d)
    spans = [(1, T // 3, 0), (0, T - T // 3, 5)]
    tabs = rows_of_spans(spans, 4, L.mn_lightning_chunk_rows())
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in tabs.items() if k != "max_len"}
    qkv, S0 = torch.randn(T, H * (2 * d + e), generator=g), torch.randn(2, H, d, e, generator=g)
    decay = torch.tensor([0.5, 0.97, 0.999][:H])
    state, out = S0.cuda(), torch.empty(T, H * e, device="cuda")
    n_ch = dev["chunk_tab"].shape[0]
    ws = torch.empty(L.mn_lightning_scan_workspace_bytes(n_ch, H, d, e), dtype=torch.uint8, device="cuda")
    qd, dd = qkv.cuda(), decay.cuda()
    check(L.mn_lightning_rows_scan(ptr(qd), qkv.shape[1], T, H, d, e, ptr(dd), ptr(state), ptr(dev["row_seq"]), ptr(dev["row_slot"]), ptr(dev["row_back"]),
                                   ptr(dev["chunk_tab"]), n_ch, ptr(out), H * e, ptr(ws), ws.numel(), current_stream()), "scan")
    act = F.silu(qkv.double())
    r = 0
    for seq, n, past in spans:
        S = S0[seq].double() * (0 if past == 0 else 1)
        for t in range(r, r + n):
            q, k, v = act[t, :H * d].reshape(H, d), act[t, H * d:2 * H * d].reshape(H, d), act[t, 2 * H * d:].reshape(H, e)
            S = decay.double()[:, None, None] * S + k[:, :, None] * v[:, None, :]
            if t in (r, r + n // 2, r + n - 1):
                ref = torch.einsum("hde,hd->he", S, q).reshape(-1)
                # fp32 sums of up to 1 / (1 - decay) = 1000 terms: 1e-5 of the row's largest value
                assert float((out[t].double().cpu() - ref).abs().max() / ref.abs().max()) < 1e-5, t
        assert rel(state[seq], S) < 1e-5
        r += n


@pytest.mark.parametrize("M,lda", [(3, 0), (300, 0), (3, 1 << 23), (130, 1 << 24), (600, 1 << 22)])
def test_rows_far_apart(M, lda):
    """One row for all (stride 0), one token of each sequence of a long batch, rows of which fewer than M and than 256 fit under 4 GiB, chunks of 256 rows and more."""
    from ming_univision_amd import ops
    N, K = 132, 192
    g = torch.Generator(device="cuda").manual_seed(M)
    buf = torch.empty((M - 1) * lda + K, dtype=torch.bfloat16, device="cuda")
    a = buf.as_strided((M, K), (lda, 1))
    (a if lda else buf).copy_(torch.randn(*((M, K) if lda else (K,)), generator=g, device="cuda"))
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(torch.bfloat16)
    ref = a.double() @ w.double().T
    assert rel(ops.gemm_bf16(a, w, None, "f32"), ref) < 3e-5 and rel(ops.gemm_bf16(a, w, None, "bf16"), ref) < 2 ** -8


@pytest.mark.parametrize("H,d,e", [(2, 16, 16), (3, 20, 36), (16, 128, 128)])
@pytest.mark.parametrize("lens", [[2] * 64, [1, 33, 64, 1, 1, 700, 2] * 2, [1] * 300 + [40, 3] + [2] * 20, [8300]])
def test_lightning_scan_of_many_sequences(H, d, e, lens):
    """The walk over the chunks cut into parts: sequences of one chunk and of many, begun before and behind a part's end, new and continuing, more chunks than the
    256 of a table; the states carried, against the recurrence in float64."""
    import numpy as np
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    from ming_univision_amd.sequences import rows_of_spans
    if H == 16 and len(lens) > 100:
        return
    L, g = lib(), torch.Generator(device="cuda").manual_seed(H + len(lens))
    n = len(lens)
    order = [(7 * i + 3) % n if n % 7 else i for i in range(n)]
    spans = [(order[i], m, 5 * (i % 3)) for i, m in enumerate(lens)]
    tabs = rows_of_spans(spans, 4, L.mn_lightning_chunk_rows())
    dev = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in tabs.items() if k != "max_len"}
    T, n_ch = sum(lens), dev["chunk_tab"].shape[0]
    qkv, S0 = torch.randn(T, H * (2 * d + e), generator=g, device="cuda"), torch.randn(n, H, d, e, generator=g, device="cuda")
    decay = torch.tensor([0.5, 0.97, 0.999] * 6)[:H].cuda()
    state, out = S0.clone(), torch.empty(T, H * e, device="cuda")
    ws = torch.empty(L.mn_lightning_scan_workspace_bytes(n_ch, H, d, e), dtype=torch.uint8, device="cuda")
    check(L.mn_lightning_rows_scan(ptr(qkv), qkv.shape[1], T, H, d, e, ptr(decay), ptr(state), ptr(dev["row_seq"]), ptr(dev["row_slot"]), ptr(dev["row_back"]),
                                   ptr(dev["chunk_tab"]), n_ch, ptr(out), H * e, ptr(ws), ws.numel(), current_stream()), "scan")
    act, r = F.silu(qkv.double()), 0
    for seq, m, past in spans:
        S = S0[seq].double() * (past != 0)
        q, k, v = act[r:r + m, :H * d].reshape(m, H, d), act[r:r + m, H * d:2 * H * d].reshape(m, H, d), act[r:r + m, 2 * H * d:].reshape(m, H, e)
        pw = decay.double()[:, None] ** torch.arange(m - 1, -1, -1, device="cuda", dtype=torch.float64)[None]
        end = decay.double()[:, None, None] ** m * S + ((k * pw.T[..., None]).permute(1, 2, 0).contiguous() @ v.permute(1, 0, 2).contiguous())
        assert rel(state[seq], end) < 1e-5
        first = ((decay.double()[:, None, None] * S + k[0, :, :, None] * v[0, :, None, :]) * q[0, :, :, None]).sum(1).reshape(-1)
        assert float((out[r].double() - first).abs().max() / first.abs().max()) < 1e-5
        last = (end * q[m - 1, :, :, None]).sum(1).reshape(-1)
        assert float((out[r + m - 1].double() - last).abs().max() / last.abs().max()) < 1e-5
        r += m
