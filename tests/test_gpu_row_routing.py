"""The routing of a one-row step as partial sums of the launch before it (row_gemv.inl, moe_gate_up.hip): hidden sizes of 3 and 4 chunks, few and 64 experts, no and two shared experts, every
weight format, tied gate rows; against the step whose scratch ends before the partial sums, which routes in its expert launch.  A logit passes 8 + 32 + 8
rounded sums here and 32 + 6 there, each off by at most 2^-24 of its products' sizes, some 30 together with gate rows of 0.02: (48 + 38) 30 / 2^24 = 1.5e-4 at worst on a probability and so on an
expert's share of the row."""
import ctypes

import pytest
import torch

from ming_univision_amd import configuration as C
from tests.util import llm_sd, rel_err

pytestmark = pytest.mark.gpu


def decoder(hidden, experts, top_k, shared, inter, weights, tie):
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    d = C.BailingMoeConfig.ming_univision_16b_a3b().to_dict()
    d.pop("model_type", None)
    d.update(hidden_size=hidden, num_attention_heads=hidden // 128, num_key_value_heads=hidden // 512, head_dim=128, num_experts=experts, num_experts_per_tok=top_k, num_shared_experts=shared,
             moe_intermediate_size=inter, intermediate_size=inter * 2, vocab_size=512, num_hidden_layers=2, num_image_tokens_for_gen=3, image_start_token=500, pad_token_id=0)
    sd = llm_sd(d, dict(diffloss_w=64, diffloss_d=2, num_sampling_steps="4", gen_method="flow_matching_swiglu-4"), 31)
    if tie:
        for li in range(2):
            g = sd[f"model.layers.{li}.mlp.gate.weight"]
            g[experts // 2:] = g[:experts - experts // 2]                      # every expert's score twice: the lower id of a pair comes first, and the cut goes through pairs
    return BailingMoeDecoder.from_state_dict(C.BailingMoeConfig(**d), {k: v.to("cuda", torch.bfloat16).contiguous() for k, v in sd.items()}, t_max=8, n_seq=1, weights=weights)


@pytest.mark.parametrize("hidden,experts,top_k,shared,inter,weights,tie",
                         [(2048, 64, 6, 2, 136, "bf16", False), (2048, 64, 7, 1, 64, "bf16", True), (1536, 64, 8, 0, 72, "bf16", False), (1536, 5, 1, 1, 8, "bf16", False), (2048, 1, 1, 2, 64, "bf16", False),
                          (2048, 16, 3, 2, 64, "fp8", True), (1536, 33, 3, 2, 48, "int8", False), (2048, 64, 6, 2, 128, "int4", False)])
def test_partial_sums_route_like_the_expert_launch(hidden, experts, top_k, shared, inter, weights, tie):
    from ming_univision_amd._lib import lib
    dec = decoder(hidden, experts, top_k, shared, inter, weights, tie)
    i32 = dict(dtype=torch.int32, device="cuda")
    seq, slot = torch.zeros(1, **i32), torch.full((1,), 5, **i32)
    n, tail = lib().mn_llm_workspace_bytes(ctypes.byref(dec.struct), 1, dec.t_max), hidden // 8 * 65 * 4
    buf = torch.empty(n + 4096, dtype=torch.uint8, device="cuda")
    key = (1, torch.cuda.current_stream().cuda_stream)
    for seed in range(4):
        x = torch.randn(1, hidden, generator=torch.Generator().manual_seed(seed)).cuda() * 10.0 ** (seed - 2)
        out = []
        for size in (n, n - 1):
            buf.fill_(77)
            dec._ws[key] = buf[:size]
            dec.kv_cache.fill_(0.25)
            out.append(dec.step(x, seq, slot, slot, slot + 1, distinct_sequences=True).clone())
            assert bool((buf[n:] == 77).all())
            assert bool((buf[n - tail:n] == 77).all()) == (size < n)           # ... and the partial sums are there or not
        assert torch.isfinite(out[0]).all() and rel_err(out[0], out[1]) < 1.5e-4, (seed, rel_err(out[0], out[1]))


def test_captured_and_replayed():
    dec = decoder(2048, 64, 6, 2, 136, "bf16", False)
    i32 = dict(dtype=torch.int32, device="cuda")
    seq, slot = torch.zeros(1, **i32), torch.full((1,), 5, **i32)
    x, new = torch.empty(1, 2048, device="cuda"), slot + 1
    rows = [torch.randn(1, 2048, generator=torch.Generator().manual_seed(s)).cuda() for s in range(4)]

    def step():
        dec.kv_cache.fill_(0.25)
        return dec.step(x, seq, slot, slot, new, distinct_sequences=True)
    want = []
    for r in rows:
        x.copy_(r)
        want.append(step().clone())
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            y = step()
    torch.cuda.synchronize()
    for r, w in zip(rows, want):
        x.copy_(r)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, w)
