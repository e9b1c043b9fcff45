"""Decoder steps of 2 .. 64 rows some of which take the image gate: the chain of launches of rows without one, its router reading each row's own gate, against the same rows one by
one.  bf16 hi / lo operands against fp32 ones, two layers: 2^-17 each of a handful of products, 1e-4 of a row's norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,experts,top,shared,weights", [(1024, 1408, 64, 6, 2, None), (256, 80, 5, 2, 1, None), (256, 128, 16, 4, 1, "int8")])
@pytest.mark.parametrize("rows", [2, 3, 17, 64])
def test_rows_together_and_alone(rows, hidden, inter, experts, top, shared, weights):
    from ming_univision_amd import configuration as C
    from ming_univision_amd._lib import check, lib, ptr
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    from ming_univision_amd.synth import synth_state_dict
    cfg = C.BailingMoeConfig(vocab_size=64, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, num_experts=experts,
                             num_experts_per_tok=top, num_shared_experts=shared, moe_intermediate_size=inter, head_dim=128, use_bias=False, multi_gate=True,
                             image_patch_token=60, image_start_token=61)
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(C.llm_param_shapes(cfg), 5, "cuda").items()}
    dec = BailingMoeDecoder.from_state_dict(cfg, sd, t_max=24, n_seq=rows, **({"weights": weights} if weights else {}))
    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g, device="cuda")
    past = torch.randn(dec.kv_cache.shape, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    slot, mask = i32([5 + r % 11 for r in range(rows)]), torch.tensor([r % 3 != 1 for r in range(rows)], dtype=torch.uint8, device="cuda")

    def step(rs, image):
        routes = torch.full((2, len(rs), top + shared), -7, dtype=torch.int32, device="cuda")
        check(lib().mn_llm_route_capture(ptr(routes)), "mn_llm_route_capture")
        try:
            at = slot[rs].contiguous()
            out = dec.step(x[rs].contiguous(), i32(rs), at, at, at + 1, image_mask=image[rs].contiguous(), distinct_sequences=True).clone()
        finally:
            check(lib().mn_llm_route_capture(None), "mn_llm_route_capture")
        return out, routes.sort(dim=2).values
    outs = []
    for image in (mask, torch.zeros_like(mask)):
        dec.kv_cache.copy_(past)
        together, routes = step(list(range(rows)), image)
        dec.kv_cache.copy_(past)
        each = [step([r], image) for r in range(rows)]
        alone, routes1 = torch.cat([o for o, _ in each]), torch.cat([r for _, r in each], dim=1)
        same = (routes == routes1).all(dim=2).all(dim=0)
        assert int((~same).sum()) <= 1 + rows // 32
        err = (together - alone).norm(dim=1) / alone.norm(dim=1)
        assert float(err[same].max()) < 1e-4, err
        outs.append(together)
    assert not torch.equal(outs[0][0], outs[1][0])       # (the image gate is another one)
