"""The dense products whose tiles are one round of the CUs: waves that split K inside a workgroup (rows_gemm.hip) for hi/lo rows, and for plain rows of prompts and pictures; plain rows
of the wide-row GEMM's own entry points keep one chain of K."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows, columns, K): one row, one fragment, columns and rows past the last tile, K of one k-step pair and no whole number of stages.  Hi/lo rows: forms of 16 x 32, 32 x 32, 32 x 64, 32 x 96, 16 x 64
# and 48 x 96; plain rows, which keep one chain of K at this entry point, the tiles beside them.
SHAPES = [(1, 4, 64), (15, 36, 192), (17, 100, 64), (33, 1024, 1024), (70, 1028, 320), (101, 2304, 768), (130, 1024, 4096), (250, 1020, 2752), (257, 2048, 576), (450, 1024, 1024), (600, 768, 2048),
          (1025, 1020, 1088), (1000, 2048, 8192)]


def rows(g, M, K, hilo, pad):
    """fp32 values of M rows and their bf16 operand: plain, or hi and lo rows with `pad` columns between the rows."""
    buf = torch.zeros(2, M, K + pad, dtype=torch.bfloat16, device="cuda")
    x = torch.randn(M, K, device="cuda", generator=g)
    buf[0, :, :K] = x
    if hilo:
        buf[1, :, :K] = x - buf[0, :, :K].float()
    return buf, buf[0, :, :K].double() + buf[1, :, :K].double()


# The forms that those leave: hi/lo 32 x 16, 32 x 64, 32 x 128 (whole and part tiles), 16 x 64, 48 x 64, 48 x 96, 64 x 64
HILO = [(450, 260, 1024), (1025, 100, 320), (65, 5372, 64), (257, 2752, 192), (200, 4092, 320), (47, 5372, 192), (144, 5372, 1088), (450, 2300, 768), (176, 5388, 1088)]
# plain rows whose K may be summed in parts: 32 x 16, 16 x 32, 32 x 32, 32 x 64, 64 x 32, 64 x 64, 64 x 128, in this order
PLAIN = [(1, 4, 64), (15, 36, 192), (33, 1024, 1024), (40, 2300, 320), (130, 1024, 4096), (250, 1020, 2752), (101, 2304, 768), (190, 2044, 320), (5400, 92, 320), (257, 2048, 576), (190, 4092, 1088),
         (257, 4092, 576), (450, 2300, 320), (1000, 2048, 8192)]


def dense_epilogues(product, M, N, K, hilo):
    from ming_univision_amd._lib import ptr
    g = torch.Generator(device="cuda").manual_seed(M + N + K + hilo)
    st = torch.cuda.current_stream().cuda_stream
    pad = 8 if M % 2 else 0
    A, a64 = rows(g, M, K, hilo, pad)
    W = torch.empty(N, K + pad, dtype=torch.bfloat16, device="cuda").normal_(0, K ** -0.5, generator=g)
    bias = torch.randn(N, device="cuda", generator=g).bfloat16() if M != 33 else None
    w64 = W[:, :K].double()
    prod = a64 @ w64.t() + (bias.double() if bias is not None else 0.0)
    sums = a64.abs() @ w64.abs().t() + (bias.double().abs() if bias is not None else 0.0)
    ldc = N + 4
    for epi in (2, 3, 0):                                # fp32, fp32 added to what is there, bf16
        C = torch.full((M + 1, ldc), 0.5, device="cuda", dtype=torch.bfloat16 if epi == 0 else torch.float32)
        rc = product(ptr(A), K + pad, A[0].numel() if hilo else 0, ptr(W), K + pad, ptr(bias) if bias is not None else None, ptr(C), ldc, M, N, K, epi, st)
        assert rc == 0
        ref = prod + (0.5 if epi == 3 else 0.0)
        # K products (twice for hi/lo) and the bias added in some order in fp32: 2^-24 of the sum of magnitudes each; one rounding to bf16: 2^-8
        bound = (2 * K + 16) * 2.0 ** -24 * (sums + 0.5) + (2.0 ** -8 * ref.abs() if epi == 0 else 0.0)
        assert bool(((C[:M, :N].double() - ref).abs() <= bound).all()), (epi, float((C[:M, :N].double() - ref).abs().max()))
        assert bool((C[M:] == 0.5).all()) and bool((C[:, N:] == 0.5).all())


@pytest.mark.parametrize("hilo", [0, 1])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_dense_epilogues(M, N, K, hilo):
    from ming_univision_amd import _lib
    dense_epilogues(_lib.lib().mn_gemm256, M, N, K, hilo)


@pytest.mark.parametrize("M,N,K", HILO)
def test_dense_epilogues_of_other_forms(M, N, K):
    from ming_univision_amd import _lib
    dense_epilogues(_lib.lib().mn_gemm256, M, N, K, 1)


@pytest.mark.parametrize("M,N,K", PLAIN)
def test_plain_rows_in_parts(M, N, K):
    """The entry that the sequence engines and the picture blocks call (mn_gemm_bf16_parts, by itself in the dev library alone)."""
    import ctypes
    import os
    from ming_univision_amd import _lib
    f = ctypes.CDLL(os.path.join(os.path.dirname(_lib.LIB_PATH), "libmingnative_dev.so")).mn_gemm_bf16_parts
    f.restype, f.argtypes = _lib.SYMBOLS["mn_gemm_bf16"]
    dense_epilogues(lambda a, lda, lo, *rest: f(a, lda, *rest), M, N, K, 0)


@pytest.mark.parametrize("width,lengths", [(256, (65, 70, 300)), (512, (130, 100, 90)), (1024, (66, 200, 450))])
def test_prompts_together_and_alone(width, lengths):
    """A row of a sequence model's prompt depends on the rows of its call up to the order of sums: a product's fp32 sums move by their own rounding, a bf16 rounding behind them by one unit (2^-8) for
    few of the values, and what each of the two layers' ten operands passes on is less than the 2^-9 that rounding costs it anyway."""
    from ming_univision_amd.configuration import DaberaxConfig
    from ming_univision_amd.daberax import DaberaxDecoder
    cfg = DaberaxConfig(width=width, vocab=40, norm=dict(eps=1e-6), token_side=dict(dim=8), layers=[
        dict(type="attention", mixer=dict(heads=4, kv_heads=2, dim=32, vdim=64, scale=0.2), mlp=dict(kind="dense", ff=2 * width + 64))] * 2)
    dec = DaberaxDecoder.synthetic(cfg, "cuda", t_max=max(lengths) + 1, n_seq=len(lengths), arith="bf16")
    g = torch.Generator().manual_seed(width)
    ids = [torch.randint(0, 40, (n,), generator=g).cuda() for n in lengths]
    alone = [dec.prefill(t, seq=i).double() for i, t in enumerate(ids)]
    both = torch.cat(ids)
    together = dec.forward_spans(dec.embed(both), [(i, n, 0) for i, n in enumerate(lengths)], tokens=both).double()
    for got, want in zip(together.split(lengths), alone):
        assert float((got - want).norm() / want.norm()) < 20 ** 0.5 * 2.0 ** -9


@pytest.mark.parametrize("M,width", [(65, 1024), (257, 1024), (450, 512), (700, 256)])
def test_plain_products_of_prompts(M, width):
    """Prompts whose plain bf16 products are one round, against the fp32 arithmetic of the same layers (two layers of products on bf16 operands, 2^-9 each of some ten of them)."""
    from ming_univision_amd.configuration import DaberaxConfig
    from ming_univision_amd.daberax import DaberaxDecoder
    cfg = DaberaxConfig(width=width, vocab=40, norm=dict(eps=1e-6), token_side=dict(dim=8), layers=[
        dict(type="attention", mixer=dict(heads=4, kv_heads=2, dim=32, vdim=64, scale=0.2), mlp=dict(kind="dense", ff=2 * width + 64))] * 2)
    ids = torch.arange(M, device="cuda") % 40
    got, want = (DaberaxDecoder.synthetic(cfg, "cuda", t_max=M + 1, n_seq=1, arith=a).prefill(ids).double() for a in ("bf16", "f32"))
    assert float((got - want).norm() / want.norm()) < 2e-2


# (K of 512 and more: 16 x 32, 32 x 32, 32 x 64, 32 x 96, 32 x 128, 64 x 64, 16 x 64, 48 x 64, 48 x 96, 48 x 64 past the caches)
@pytest.mark.parametrize("M,hidden,K", [(1, 4, 64), (17, 36, 192), (40, 2048, 768), (101, 2752, 1024), (128, 1028, 320), (256, 2048, 768), (47, 100, 576), (144, 1020, 576), (130, 2748, 576),
                                        (5400, 92, 768), (16, 5372, 1088), (65, 4092, 1024), (190, 3068, 576), (33, 8160, 2048)])
def test_gated_hilo(M, hidden, K):
    from ming_univision_amd import _lib
    from ming_univision_amd._lib import ptr
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(M + hidden + K)
    A, a64 = rows(g, M, K, 1, 0)
    W = torch.empty(2 * hidden, K, dtype=torch.bfloat16, device="cuda").normal_(0, K ** -0.5, generator=g)
    b = torch.randn(2 * hidden, device="cuda", generator=g).bfloat16()
    Y = torch.full((2, M + 1, hidden), 3.0, dtype=torch.bfloat16, device="cuda")
    rc = L.mn_gemm256_swiglu_split(ptr(A), K, A[0].numel(), ptr(W), K, ptr(b), ptr(Y), hidden, Y[0].numel(), M, hidden, K, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    w64 = W.double()
    z, s = a64 @ w64.t() + b.double(), a64.abs() @ w64.abs().t() + b.double().abs()
    gate, up = z[:, :hidden], z[:, hidden:]
    act = torch.nn.functional.silu(gate)
    # the sums' error through the gate (slope of silu below 1.1) and the product, the fp32 silu (8 ulp) and the pair's 2^-17
    dz = (2 * K + 16) * 2.0 ** -24 * s
    bound = 1.1 * dz[:, :hidden] * up.abs() + dz[:, hidden:] * act.abs() + dz[:, :hidden] * dz[:, hidden:] + (2.0 ** -20 + 2.0 ** -16.5) * (act * up).abs() + 1e-30
    got = Y[0, :M].double() + Y[1, :M].double()
    assert bool(((got - act * up).abs() <= bound).all()), float((got - act * up).abs().max())
    assert bool((Y[:, M:] == 3.0).all())
