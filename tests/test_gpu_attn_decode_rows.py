"""Decode attention around the row counts from which one wave serves a key head's four query heads (40 pairs of row and key head, 48 with two), past the caches the one-launch form takes: rows of
1 .. t_max keys, splits that hold no key of a row, holes in the mask, fp32 and hi / lo outputs.  The reference is float64; fp32 sums of at most 1300 products: 1e-5
of the largest value."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 7, 8, 9, 33, 64, 65])
@pytest.mark.parametrize("n_kv,n_q,hd,t_max", [(4, 16, 128, 1300), (1, 4, 128, 1100), (2, 8, 128, 1030), (4, 16, 64, 1100), (3, 6, 128, 1100)])
@pytest.mark.parametrize("use_mask", [False, True])
def test_rows(M, n_kv, n_q, hd, t_max, use_mask):
    from ming_univision_amd import ops
    g = torch.Generator().manual_seed(M + n_q)
    n_seq = 5
    q = torch.randn(M, n_q, hd, generator=g) * hd ** -0.5
    kv = torch.randn(n_seq, 2, n_kv, t_max, hd, generator=g)
    seq = torch.randint(0, n_seq, (M,), generator=g, dtype=torch.int32)
    lens = torch.randint(1, t_max + 1, (M,), generator=g, dtype=torch.int32)
    lens[0], lens[-1] = t_max, 1
    mask = (torch.rand(M, t_max, generator=g) < 0.7).to(torch.uint8)
    mask[:, 0] = 1
    got = ops.attn_decode(q.cuda(), n_q, n_kv, hd, kv.cuda(), seq.cuda(), lens.cuda(), mask.cuda() if use_mask else None).cpu().double().reshape(M, n_q, hd)
    for m in range(M):
        n = int(lens[m])
        k, v = kv[seq[m], 0, :, :n].double(), kv[seq[m], 1, :, :n].double()
        s = torch.einsum("ghd,gnd->ghn", q[m].double().reshape(n_kv, n_q // n_kv, hd), k)
        s = s.masked_fill(mask[m, :n] == 0, -float("inf")) if use_mask else s
        ref = torch.einsum("ghn,gnd->ghd", torch.softmax(s, -1), v).reshape(n_q, hd)
        assert float((got[m] - ref).abs().max() / ref.abs().max()) < 1e-5, m
