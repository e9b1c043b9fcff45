"""Expert products of a decoder step that a resident set of workgroups shares in equal parts (3 rows and more; the down projection also above 32), against the same rows one by one,
which take none of it: row counts where the number of slabs changes, groups of one row and of all, blocks of 16 rows and one row more, widths of whole and of part chunks and
column tiles, fewer chunks than workgroups and many more.  bf16 hi / lo operands against fp32 ones, two layers: 2^-17 each of a handful of products, 1e-4 of a row's norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def decoder(hidden, inter, experts, top, shared, n_seq):
    from ming_univision_amd import configuration as C
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    from ming_univision_amd.synth import synth_state_dict
    cfg = C.BailingMoeConfig(vocab_size=64, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2, num_experts=experts,
                             num_experts_per_tok=top, num_shared_experts=shared, moe_intermediate_size=inter, head_dim=128, use_bias=False,
                             image_patch_token=60, image_start_token=61)
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(C.llm_param_shapes(cfg), 5, "cuda").items()}
    return BailingMoeDecoder.from_state_dict(cfg, sd, t_max=24, n_seq=n_seq)


@pytest.mark.parametrize("hidden,inter,experts,top,shared", [(1024, 1408, 64, 6, 2), (512, 200, 12, 12, 1), (256, 72, 4, 4, 2), (2048, 1408, 24, 3, 1)])
@pytest.mark.parametrize("rows", [3, 4, 5, 16, 17, 32, 33, 49, 64])
def test_rows_together_and_alone(rows, hidden, inter, experts, top, shared):
    from ming_univision_amd._lib import check, lib, ptr
    dec = decoder(hidden, inter, experts, top, shared, rows)
    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g, device="cuda")
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
    for ws in dec._ws.values():
        ws.fill_(127)                                    # what a slab does not hold is not read
    together, routes = step(list(range(rows)))
    dec.kv_cache.copy_(past)
    next(ws for (r, _), ws in dec._ws.items() if r == rows).fill_(255)        # (NaN everywhere)
    again, _ = step(list(range(rows)))
    assert torch.equal(together, again)
    dec.kv_cache.copy_(past)
    each = [step([r]) for r in range(rows)]
    alone, routes1 = torch.cat([o for o, _ in each]), torch.cat([r for _, r in each], dim=1)
    same = (routes == routes1).all(dim=2).all(dim=0)
    assert int((~same).sum()) <= (0 if experts == top else 1 + rows // 32)
    err = (together - alone).norm(dim=1) / alone.norm(dim=1)
    assert float(err[same].max()) < 1e-4, err
