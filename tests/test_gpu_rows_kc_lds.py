"""The one-launch Linear of test_gpu_rows_kc on aligned rows of 5 and more, which come through LDS: K that ends inside a piece or leaves waves without one, rows that
fill no tile, strides of their own, plain and silu rows, the epilogues.  Same reference and tolerance."""
import pytest
import torch

from tests.test_gpu_rows_kc import call

pytestmark = pytest.mark.gpu
F = torch.nn.functional


@pytest.mark.parametrize("M", [4, 5, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("N,K", [(1, 8), (66, 40), (16, 64), (250, 72), (66, 520), (250, 1032), (4097, 504), (4500, 1024), (2048, 2048), (300, 2600)])
def test_forms(M, N, K):
    from ming_univision_amd._lib import lib
    g = torch.Generator().manual_seed(M * 7 + N + K)
    w, bias = torch.randn(2 * N, K, generator=g).bfloat16().cuda(), torch.randn(2 * N, generator=g).bfloat16().cuda()
    ld = (K + 7) // 4 * 4
    xb = torch.full((M + 1, ld), float("nan"), device="cuda")       # what lies beside the rows is no operand
    xb[:M, :K] = torch.randn(M, K, generator=g).cuda()
    x, res = xb[:M, :K].double(), torch.randn(M, N, generator=g).cuda()
    for pro, epi in ((0, 0), (1, 0), (0, 3), (1, 6), (0, 4)):
        pair = epi in (3, 6)
        r, wd, bd = (F.silu(x) if pro else x), w[:2 * N if pair else N].double(), bias[:2 * N if pair else N].double()
        y, mag = r @ wd.T + bd, r.abs() @ wd.abs().T + bd.abs()
        room = mag[:, :N].clone()
        if pair:
            up, act = y[:, N:], F.silu(y[:, :N]) if epi == 3 else F.gelu(y[:, :N], approximate="tanh")
            room, y = 1.2 * mag[:, :N] * up.abs() + mag[:, N:] * act.abs(), act * up      # both activations are 1.13-Lipschitz
        elif epi == 4:
            y, room = y + res.double(), room + res.double().abs()
        ws = torch.empty(lib().mn_skinny_workspace_bytes(M, N, K, epi), dtype=torch.uint8, device="cuda")
        out = torch.full((M + 1, N + 2), 7.0, device="cuda")
        call(xb.data_ptr(), ld, w, out.data_ptr(), N + 2, M, N, K, ws, prologue=pro, epilogue=epi, eps=1e-6, bias=bias, res=res, ldres=N)
        assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())
        assert float(((out[:M, :N].double() - y).abs() / (room + 1e-3)).max()) < 2.0 ** -15, (pro, epi)
