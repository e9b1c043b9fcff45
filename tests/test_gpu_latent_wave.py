"""Latent attention whose waves take whole tiles of 16 keys (latents of 128, 256, 384 and 512 values) against float64: edges of tiles and of a workgroup's share, runs of
rows, heads that do not fill 16, splits, and a maximum that rises in the middle of the walk."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _call(q, arena, seq, lens, blk, ks):
    from ming_univision_amd._lib import check, current_stream, lib, ptr
    M, H, r = q.shape
    ws = torch.empty(max(16, lib().mn_latent_attn_workspace_bytes(M, H, r, ks)), dtype=torch.uint8, device="cuda")
    out = torch.full((M, H, r), float("nan"), device="cuda")
    check(lib().mn_latent_attn(ptr(q), ptr(arena), ptr(seq), ptr(lens), ptr(blk), blk.shape[0], M, H, r, arena.shape[1], int(lens.max()), ks, ptr(out), ptr(ws), ws.numel(),
                               current_stream()))
    return out


def _want(q, arena, seq, lens):
    out = torch.empty_like(q, dtype=torch.float64)
    for m in range(q.shape[0]):
        k = arena[seq[m], :lens[m]].double()
        out[m] = torch.softmax(q[m].double() @ k.T, -1) @ k
    return out


@pytest.mark.parametrize("r", [128, 256, 384, 512])
@pytest.mark.parametrize("H,ks,first", [(16, 1, 128), (16, 1, 143), (5, 1, 129), (17, 2, 257), (16, 3, 400), (32, 2, 1040)])
def test_runs_of_rows(r, H, ks, first):
    g = torch.Generator().manual_seed(r + H + first)
    runs = [1, 4, 3, 2]                                   # rows of a run: consecutive positions of one sequence
    M, t_max = sum(runs), first + 8
    arena = torch.randn(len(runs), t_max, r, generator=g).cuda()
    arena[:, first + 4:] = float("nan")                   # nothing behind a row's length is used
    q = (torch.randn(M, H, r, generator=g) * 2 * r ** -0.5).cuda()
    seq, lens, blk, row = [], [], [], 0
    for i, n in enumerate(runs):
        blk.append([row, n])
        seq += [i] * n
        lens += [first + j - 16 * (i == 2) for j in range(n)]      # (a sequence a tile shorter)
        row += n
    seq, lens, blk = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in (seq, lens, blk))
    out, want = _call(q, arena, seq, lens, blk, ks), _want(q, arena, seq.tolist(), lens.tolist())
    # scores are sums of r products in fp32 (8 chains), off by about 2^-24 sqrt(r / 8) of their deviation of 2; the weights by as much, relative
    assert float((out - want).norm() / want.norm()) < 1e-6


@pytest.mark.parametrize("r", [256, 512])
def test_maximum_that_rises(r):
    """Keys that a query points at, further and further into the walk: the sums so far are scaled down in the middle of it."""
    g = torch.Generator().manual_seed(r)
    n, H = 640, 16
    arena = torch.randn(2, n, r, generator=g)
    q = torch.randn(2, H, r, generator=g) * r ** -0.5
    for s in range(2):
        for j, key in enumerate((200, 300, 420, 639)):
            arena[s, key] = q[s, 3] / q[s, 3].norm() * (12.0 + 14.0 * j) / q[s, 3].norm()      # scores of query 3: 12, 26, 40, 54
    arena, q = arena.cuda(), q.cuda()
    seq, lens = torch.arange(2, dtype=torch.int32, device="cuda"), torch.tensor([n, 421], dtype=torch.int32, device="cuda")
    blk = torch.tensor([[0, 1], [1, 1]], dtype=torch.int32, device="cuda")
    for ks in (1, 3):
        out, want = _call(q, arena, seq, lens, blk, ks), _want(q, arena, [0, 1], lens.tolist())
        assert float(((out - want).norm(dim=-1) / want.norm(dim=-1)).max()) < 1e-5      # (scores of 54 are off by 2^-24 x 54 x a few)
