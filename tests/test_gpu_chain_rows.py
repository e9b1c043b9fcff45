"""Decoder steps of up to 64 rows (one launch chain: router of a workgroup a row, pairs sorted 64 at a time) against the same rows one by one, which take
none of it: row counts at the edges of the sort's chunks, few and many experts, more pairs than chunks of one wave hold."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def decoder(experts, top, shared, inter, t_max, n_seq):
    from ming_univision_amd import configuration as C
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    from ming_univision_amd.synth import synth_state_dict
    cfg = C.BailingMoeConfig(vocab_size=64, hidden_size=256, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, num_experts=experts,
                             num_experts_per_tok=top, num_shared_experts=shared, moe_intermediate_size=inter, head_dim=128, use_bias=False,
                             image_patch_token=60, image_start_token=61)
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(C.llm_param_shapes(cfg), 5).items()}
    return cfg, BailingMoeDecoder.from_state_dict(cfg, sd, t_max=t_max, n_seq=n_seq)


@pytest.mark.parametrize("rows", [6, 8, 21, 32, 33, 43, 63, 64])
@pytest.mark.parametrize("experts, top, shared", [(64, 6, 2), (8, 2, 1), (64, 14, 2), (3, 3, 1), (14, 14, 2)])
def test_rows_together_and_alone(rows, experts, top, shared):
    """Every row that has the same experts in both is held to the products' error, in the output and in the second layer's keys and values; where not all experts are
    chosen, a few rows may differ in one (a tie within that error).  14 experts, all chosen, of 64 rows: 1024 pairs, every chunk of the sort full."""
    from ming_univision_amd._lib import check, lib, ptr
    cfg, dec = decoder(experts, top, shared, 64, 24, rows)
    g = torch.Generator(device="cuda").manual_seed(rows + experts)
    x = torch.randn(rows, 256, generator=g, device="cuda")
    past = torch.randn(dec.kv_cache.shape, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    slot = i32([5 + r % 11 for r in range(rows)])

    def step(rs):
        routes = torch.full((2, len(rs), top + shared), -7, dtype=torch.int32, device="cuda")
        check(lib().mn_llm_route_capture(ptr(routes)), "mn_llm_route_capture")
        try:
            at = slot[rs].contiguous()
            out = dec.step(x[rs].contiguous(), i32(rs), at, at, at + 1, distinct_sequences=True).clone()
        finally:
            check(lib().mn_llm_route_capture(None), "mn_llm_route_capture")
        return out, routes.sort(dim=2).values
    dec.kv_cache.copy_(past)
    together, routes = step(list(range(rows)))
    kv = dec.kv_cache.clone()
    dec.kv_cache.copy_(past)
    each = [step([r]) for r in range(rows)]
    alone, routes1 = torch.cat([o for o, _ in each]), torch.cat([r for _, r in each], dim=1)
    same = (routes == routes1).all(dim=2)                # [layer, row]
    assert int((~same.all(dim=0)).sum()) <= (0 if experts == top else 1 + rows // 32)
    # bf16 hi/lo operands against fp32 ones, two layers: 2^-17 each of a handful of products
    err = (together - alone).norm(dim=1) / alone.norm(dim=1)
    assert float(err[same.all(dim=0)].max()) < 1e-4, err
    off = (kv - dec.kv_cache).abs().amax(dim=(2, 3, 4, 5))          # [layer, row]
    assert float(off[0].max()) < 1e-3 * float(past.abs().max())
    assert float(off[1][same[0]].max()) < 1e-3 * float(past.abs().max()), off[1]
