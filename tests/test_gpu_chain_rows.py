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
@pytest.mark.parametrize("experts, top, shared", [(64, 6, 2), (8, 2, 1), (64, 14, 2), (3, 3, 1)])
def test_rows_together_and_alone(rows, experts, top, shared):
    cfg, dec = decoder(experts, top, shared, 64, 24, rows)
    g = torch.Generator(device="cuda").manual_seed(rows + experts)
    x = torch.randn(rows, 256, generator=g, device="cuda")
    past = torch.randn(dec.kv_cache.shape, generator=g, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    dec.kv_cache.copy_(past)
    slot = i32([5 + r % 11 for r in range(rows)])
    together = dec.step(x, i32(list(range(rows))), slot, slot, slot + 1, distinct_sequences=True).clone()
    kv = dec.kv_cache.clone()
    dec.kv_cache.copy_(past)
    alone = torch.cat([dec.step(x[r:r + 1].contiguous(), i32([r]), slot[r:r + 1].contiguous(), slot[r:r + 1].contiguous(), slot[r:r + 1] + 1,
                                distinct_sequences=True).clone() for r in range(rows)])
    # bf16 hi/lo operands against fp32 ones, two layers: 2^-17 each of a handful of products; a row whose k-th and next expert tie within that may differ in them
    err = (together - alone).norm(dim=1) / alone.norm(dim=1)
    assert int((err > 1e-4).sum()) <= (0 if experts == top else 1 + rows // 32), err.max()
    assert float((kv - dec.kv_cache)[0].abs().max()) < 1e-3 * float(past.abs().max())
