"""Expert products in row tiles of 32 and 64 (and of 128 beyond): row counts on both sides of the rules' lines, groups of no row, of one, of all and of one more than a tile,
widths of whole and of part column tiles, against the same rows a few at a time, which take the streaming kernels.  bf16 hi / lo operands against fp32 ones, two layers: 2^-17
each of a handful of products, 1e-4 of a row's norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,inter,experts,top,shared,counts", [
    (1024, 1408, 64, 6, 2, (65, 100, 266, 267)), (256, 192, 8, 2, 1, (65, 100, 101, 228, 229)), (512, 320, 12, 12, 1, (65, 80)), (256, 64, 16, 1, 0, (65, 129))])
def test_rows_together_and_in_parts(hidden, inter, experts, top, shared, counts):
    from ming_univision_amd import configuration as C
    from ming_univision_amd._lib import check, lib, ptr
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    from ming_univision_amd.synth import synth_state_dict
    cfg = C.BailingMoeConfig(vocab_size=64, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, num_experts=experts,
                             num_experts_per_tok=top, num_shared_experts=shared, moe_intermediate_size=inter, head_dim=128, use_bias=False,
                             image_patch_token=60, image_start_token=61)
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(C.llm_param_shapes(cfg), 5, "cuda").items()}
    dec = BailingMoeDecoder.from_state_dict(cfg, sd, t_max=24, n_seq=max(counts))
    g = torch.Generator(device="cuda").manual_seed(hidden + inter)
    past = torch.randn(dec.kv_cache.shape, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    for rows in counts:
        x = torch.randn(rows, hidden, generator=g, device="cuda")
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
        dec.kv_cache.copy_(past)
        next(ws for (r, _), ws in dec._ws.items() if r == rows).fill_(255)    # (NaN everywhere: what a step did not write it does not read)
        again, _ = step(list(range(rows)))
        assert torch.equal(together, again)
        dec.kv_cache.copy_(past)
        parts = [step(list(range(r, min(rows, r + 32)))) for r in range(0, rows, 32)]
        apart, routes1 = torch.cat([o for o, _ in parts]), torch.cat([r for _, r in parts], dim=1)
        same = (routes == routes1).all(dim=2).all(dim=0)
        assert int((~same).sum()) <= (0 if experts == top else 1 + rows // 32)
        err = (together - apart).norm(dim=1) / apart.norm(dim=1)
        assert float(err[same].max()) < 1e-4, (rows, err)
