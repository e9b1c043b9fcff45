"""A row of NaN in a decoder step leaves the other rows as they are: it has no top-k, and its slots name experts 0 .. top_k - 1, so that no expert's group holds more
pairs than there are rows (the grouped products pass over such a group, for all of its rows) and no index lies outside the experts."""
import pytest
import torch

from tests.test_gpu_chain_rows import decoder

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [2, 4, 6, 33, 64, 70, 130])
@pytest.mark.parametrize("experts, top, shared", [(64, 6, 2), (8, 2, 1), (64, 3, 0)])
def test_other_rows(rows, experts, top, shared):
    cfg, dec = decoder(experts, top, shared, 64, 24, rows)
    g = torch.Generator(device="cuda").manual_seed(rows + experts)
    x = torch.randn(rows, 256, generator=g, device="cuda")
    past = torch.randn(dec.kv_cache.shape, generator=g, device="cuda")
    seq = torch.arange(rows, dtype=torch.int32, device="cuda")
    slot = torch.full((rows,), 7, dtype=torch.int32, device="cuda")

    def step(v):
        dec.kv_cache.copy_(past)
        return dec.step(v, seq, slot, slot, slot + 1, distinct_sequences=True).clone()
    want = step(x)
    bad = rows // 2
    x[bad] = float("nan")
    got = step(x)
    others = [r for r in range(rows) if r != bad]
    assert bool(got[bad].isnan().all())
    # (the same products of the same rows; a row's place in its expert's tile may be another)
    assert float(((got - want)[others].norm(dim=1) / want[others].norm(dim=1)).max()) < 1e-6


@pytest.mark.parametrize("E, top", [(64, 6), (8, 3), (5, 5)])
@pytest.mark.parametrize("M", [1, 4, 5, 40])
def test_router(M, E, top):
    """The stand-alone router's slots of such a row, with and without norms of its weights."""
    from ming_univision_amd import ops
    g = torch.Generator(device="cuda").manual_seed(M + E)
    x = torch.randn(M, 128, generator=g, device="cuda")
    x[M - 1] = float("nan")
    ln, gate = torch.ones(128, dtype=torch.bfloat16, device="cuda"), torch.randn(E, 128, generator=g, device="cuda").to(torch.bfloat16)
    for norm in (True, False):
        _, idx, w = ops.moe_router(x, ln, 1e-6, gate, None, None, top, norm, 2)
        assert idx[M - 1].tolist() == list(range(top)) + [E, E + 1]
        assert bool(w[M - 1, :top].isnan().all()) and w[M - 1, top:].tolist() == [1.0, 1.0]
        assert all(sorted(set(r)) == sorted(r) and max(r) < E for r in idx[:M - 1, :top].tolist())
