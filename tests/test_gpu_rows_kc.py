"""A Linear of 2 .. 32 rows as one launch (rows_kc.inl) around its edges: one and two row tiles, columns that fill no tile, one and two tiles a workgroup, K that
ends inside a chunk or leaves waves without one, every prologue and epilogue it takes, rows in wider buffers, and calls it must leave to the three
launches (output over the input, LayerNorm, more rows).  The reference is float64; hi / lo rows (the three launches) carry 17 bits:
2^-16 of the summed magnitudes."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu
F = torch.nn.functional


def call(x, ldx, w, out, ldo, M, N, K, ws, **kw):
    from ming_univision_amd._lib import SkinnyArgs, check, current_stream, lib
    a = SkinnyArgs()
    a.x, a.ldx, a.w, a.ldw, a.out, a.ldo, a.M, a.N, a.K = x, ldx, w.data_ptr(), K, out, ldo, M, N, K
    if ws is not None:
        a.ws, a.ws_bytes = ws.data_ptr(), ws.numel()
    for k, v in kw.items():
        setattr(a, k, v.data_ptr() if torch.is_tensor(v) else v)
    check(lib().mn_skinny_gemm(C.byref(a), current_stream()), "skinny")


@pytest.mark.parametrize("M", [2, 3, 16, 17, 32, 33])
@pytest.mark.parametrize("N,K", [(1, 8), (66, 200), (16, 512), (250, 1032), (1024, 1024), (4097, 504), (4500, 1024), (2048, 2048)])
def test_forms(M, N, K):
    from ming_univision_amd._lib import lib
    g = torch.Generator().manual_seed(M + N + K)
    w = (torch.randn(2 * N, K, generator=g)).bfloat16().cuda()
    bias, gain = torch.randn(2 * N, generator=g).bfloat16().cuda(), (1 + 0.2 * torch.randn(K, generator=g)).bfloat16().cuda()
    beta = (0.2 * torch.randn(K, generator=g)).bfloat16().cuda()
    xb, pb = (torch.randn(M, K + 3, generator=g) + 0.3).cuda(), torch.randn(M, K + 5, generator=g).cuda()
    x, add = xb[:, 1:1 + K].double(), pb[:, 2:2 + K].double()
    res, gate = torch.randn(M, N + 1, generator=g).cuda(), torch.randn(M, N, generator=g).cuda()
    L = lib()
    L.mn_skinny_workspace_bytes.restype = C.c_size_t
    rows = {0: x, 1: F.silu(x), 2: F.silu(x + add), 3: x * torch.rsqrt((x * x).mean(1, keepdim=True) + 1e-6) * gain.double(),
            4: F.layer_norm(x, (K,), gain.double(), beta.double(), 1e-6)}
    for pro, epi, with_bias in ((0, 0, 0), (0, 0, 1), (1, 1, 1), (2, 2, 1), (3, 0, 0), (3, 3, 1), (0, 3, 0), (0, 4, 1), (0, 5, 1), (0, 6, 0), (4, 0, 1)):
        pair = epi in (3, 6)
        r, wd, bd = rows[pro], w[:2 * N if pair else N].double(), bias[:2 * N if pair else N].double() * with_bias
        y, mag = r @ wd.T + bd, r.abs() @ wd.abs().T + bd.abs()
        room = mag[:, :N].clone()
        if pair:
            up, act = y[:, N:], F.silu(y[:, :N]) if epi == 3 else F.gelu(y[:, :N], approximate="tanh")
            room = 1.2 * mag[:, :N] * up.abs() + mag[:, N:] * act.abs()      # both activations are 1.13-Lipschitz
            y = act * up
        elif epi in (1, 2):
            y, room = (F.silu(y) if epi == 1 else F.gelu(y)), 1.2 * room
        elif epi == 4:
            y, room = y + res[:, :N].double(), room + res[:, :N].double().abs()
        elif epi == 5:
            room = room * gate.double().abs() + res[:, :N].double().abs()
            y = res[:, :N].double() + gate.double() * y
        ws = torch.empty(L.mn_skinny_workspace_bytes(M, N, K, epi), dtype=torch.uint8, device="cuda")
        out = torch.full((M + 1, N + 2), 7.0, device="cuda")
        kw = dict(prologue=pro, epilogue=epi, eps=1e-6, ln_g=gain, ln_b=beta, pro_a=pb.data_ptr() + 8, ld_pro_a=K + 5, res=res, ldres=N + 1, gate=gate, ldgate=N)
        if with_bias:
            kw["bias"] = bias
        call(xb.data_ptr() + 4, K + 3, w, out.data_ptr(), N + 2, M, N, K, ws, **kw)
        assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())
        assert float(((out[:M, :N].double() - y).abs() / (room + 1e-3)).max()) < 2.0 ** -15, (pro, epi)


@pytest.mark.parametrize("M,with_ws", [(2, False), (5, False), (8, False), (5, True), (20, True)])
def test_small_steps_and_infinities(M, with_ws):
    """2 .. 8 rows without scratch are held to the fp32 kernel's error (2^-24 a step of sums of trees: 1e-7 of the summed magnitudes); an infinite value
    makes its row's outputs infinite with the weights' signs, two of opposite sign NaN, and no other row sees them."""
    from ming_univision_amd._lib import lib
    g = torch.Generator().manual_seed(M)
    for N, K in ((1024, 1024), (4096, 1032), (100, 520)):
        w = torch.randn(N, K, generator=g).bfloat16().cuda()
        x = torch.randn(M, K, generator=g).cuda()
        ws = torch.empty(lib().mn_skinny_workspace_bytes(M, N, K, 0), dtype=torch.uint8, device="cuda") if with_ws else None
        out = torch.empty(M, N, device="cuda")
        call(x.data_ptr(), K, w, out.data_ptr(), N, M, N, K, ws)
        assert float(((out.double() - x.double() @ w.double().T).abs() / (x.double().abs() @ w.double().abs().T)).max()) < 1e-7
        x[1, 7] = float("inf")
        x[0, 3], x[0, K - 1] = float("inf"), -float("inf")
        call(x.data_ptr(), K, w, out.data_ptr(), N, M, N, K, ws)
        want = x.double() @ w.double().T
        assert torch.equal(out[1].double(), want[1]) and bool((torch.isnan(out[0]) == torch.isnan(want[0])).all()) and bool(torch.isfinite(out[2:]).all())


@pytest.mark.parametrize("M,with_ws", [(2, False), (8, False), (5, True), (20, True)])
def test_range_of_fp32(M, with_ws):
    """Finite values that bf16 rounds to infinity, and tiny ones: products of all their bits (1e-7 of the summed magnitudes) from 2^-100 on."""
    from ming_univision_amd._lib import lib
    g = torch.Generator().manual_seed(M)
    N, K = 1024, 1024
    w = torch.randn(N, K, generator=g).bfloat16().cuda()
    x = torch.randn(M, K, generator=g)
    x[0], x[1] = 0.0, x[1] * 2.0 ** -98
    x[0, 3], x[0, K - 1] = 3.4e38, -3.3999e38
    x = x.cuda()
    w[:, K - 1] = (w[:, 3].float() * 0.5).bfloat16()              # (sums stay finite)
    w[:, 3] = w[:, 3].clamp(-0.75, 0.75)
    w[:, K - 1] = w[:, K - 1].clamp(-0.125, 0.125)
    ws = torch.empty(lib().mn_skinny_workspace_bytes(M, N, K, 0), dtype=torch.uint8, device="cuda") if with_ws else None
    out = torch.empty(M, N, device="cuda")
    call(x.data_ptr(), K, w, out.data_ptr(), N, M, N, K, ws)
    off = (out.double() - x.double() @ w.double().T).abs() / (x.double().abs() @ w.double().abs().T)
    assert float(off.max()) < 1e-7


def test_output_over_the_input():
    """The rows are all read before any is written: out = x, and out between the rows of x."""
    from ming_univision_amd._lib import lib
    g = torch.Generator().manual_seed(3)
    M, N = 12, 512
    w = (torch.randn(N, N, generator=g) * N ** -0.5).bfloat16().cuda()
    ws = torch.empty(lib().mn_skinny_workspace_bytes(M, N, N, 0), dtype=torch.uint8, device="cuda")
    for ld, at in ((N, 0), (2 * N, N), (N + 64, 32)):
        buf = torch.randn(M + 1, ld, generator=g).cuda()
        flat = buf.reshape(-1)
        x = torch.stack([flat[i * ld:i * ld + N] for i in range(M)]).double()
        call(buf.data_ptr(), ld, w, buf.data_ptr() + 4 * at, ld, M, N, N, ws)
        got = torch.stack([flat[i * ld + at:i * ld + at + N] for i in range(M)]).double()
        want = x @ w.double().T
        assert float((got - want).abs().max() / want.abs().max()) < 1e-5


@pytest.mark.parametrize("M", [9, 17, 57, 16, 65])
def test_logits_of_a_row_by_itself(M):
    """One row more than whole chunks of eight (up to 64 rows): that row's logits are fp32 products (1e-7 of the summed magnitudes, as above), the others hi / lo."""
    from ming_univision_amd import configuration as cfgs
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    cfg = cfgs.BailingMoeConfig(vocab_size=512, hidden_size=256, num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=2, head_dim=128, use_bias=False,
                                rope_theta=600000.0, num_experts=8, num_shared_experts=2, num_experts_per_tok=3, moe_intermediate_size=64, multi_gate=True,
                                num_image_tokens_for_gen=16, image_start_token=500)
    dec = BailingMoeDecoder.synthetic(cfg, "cuda", seed=1, t_max=16, n_seq=1)
    h = torch.randn(M, 256, generator=torch.Generator().manual_seed(M)).cuda()
    want, mag = h.double() @ dec.lm_head.double().T, h.double().abs() @ dec.lm_head.double().abs().T
    off = (dec.logits(h).double() - want).abs() / mag
    assert float(off.max()) < 2.0 ** -16 and (M % 8 != 1 or M > 64 or float(off[-1].max()) < 1e-7)
