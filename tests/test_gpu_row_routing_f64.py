"""One-row decoder steps whose routing arrives as partial sums (row_gemv.inl, moe_gate_up.hip) against float64: the partial sums themselves, of a row that is known exactly as the attention's output
weights are zero, and the experts' result behind them."""
import ctypes

import pytest
import torch

from ming_univision_amd import configuration as C
from tests.util import llm_sd

pytestmark = pytest.mark.gpu


def mlp64(row, sd, p, cfg):
    """The decoder layer's sparse block in float64, its routing (ids by descending probability) and the smallest gap on the way to the last pick."""
    W = lambda name: sd[p + name].double()
    xn = row / torch.sqrt((row * row).mean() + cfg.rms_norm_eps) * W(".post_attention_layernorm.weight")
    prob = torch.softmax(W(".mlp.gate.weight") @ xn, 0)
    order = torch.sort(prob, descending=True)
    top = order.indices[:cfg.num_experts_per_tok]
    gap = float((order.values[:-1] - order.values[1:])[:cfg.num_experts_per_tok].min() / order.values[0])
    w = prob[top] / prob[top].sum() if cfg.norm_topk_prob else prob[top]
    ff = lambda q: W(q + ".down_proj.weight") @ (torch.nn.functional.silu(W(q + ".gate_proj.weight") @ xn) * (W(q + ".up_proj.weight") @ xn))
    y = sum(float(w[i]) * ff(f".mlp.experts.{int(e)}") for i, e in enumerate(top))
    return row + y + ff(".mlp.shared_experts"), gap


@pytest.mark.parametrize("hidden,experts,top_k,shared,inter", [(2048, 64, 6, 2, 136), (2048, 64, 7, 1, 64), (1536, 33, 4, 2, 72)])
def test_step_against_float64(hidden, experts, top_k, shared, inter):
    from ming_univision_amd._lib import lib
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    d = C.BailingMoeConfig.ming_univision_16b_a3b().to_dict()
    d.pop("model_type", None)
    d.update(hidden_size=hidden, num_attention_heads=hidden // 128, num_key_value_heads=hidden // 512, head_dim=128, num_experts=experts, num_experts_per_tok=top_k, num_shared_experts=shared,
             moe_intermediate_size=inter, intermediate_size=inter * 2, vocab_size=512, num_hidden_layers=1, num_image_tokens_for_gen=3, image_start_token=500, pad_token_id=0)
    cfg = C.BailingMoeConfig(**d)
    sd = {k: v.bfloat16() for k, v in llm_sd(d, dict(diffloss_w=64, diffloss_d=2, num_sampling_steps="4", gen_method="flow_matching_swiglu-4"), 17).items()}
    p = "model.layers.0"
    sd[p + ".attention.dense.weight"].zero_()
    for k in sd:
        if k.endswith("_proj.weight") or k.endswith("mlp.gate.weight"):
            sd[k] = (sd[k].float() * (sd[k].shape[1] ** -0.5 / sd[k].float().std())).bfloat16()      # (experts that weigh as much as the row)
    dec = BailingMoeDecoder.from_state_dict(cfg, {k: v.cuda().contiguous() for k, v in sd.items()}, t_max=8, n_seq=1)
    i32 = dict(dtype=torch.int32, device="cuda")
    seq, slot = torch.zeros(1, **i32), torch.full((1,), 5, **i32)
    n, tail = lib().mn_llm_workspace_bytes(ctypes.byref(dec.struct), 1, dec.t_max), hidden // 8 * 65 * 4
    buf = torch.empty(n, dtype=torch.uint8, device="cuda")
    dec._ws[(1, torch.cuda.current_stream().cuda_stream)] = buf
    done = 0
    for seed in range(12):
        x = torch.randn(1, hidden, generator=torch.Generator().manual_seed(seed)) * 2.0 ** (seed % 5 - 2)
        want, gap = mlp64(x[0].double(), sd, p, cfg)
        if gap < 1e-4:                                                                               # (a pick that rounding may turn)
            continue
        done += 1
        dec.kv_cache.fill_(0.25)
        got = dec.step(x.cuda(), seq, slot, slot, slot + 1, distinct_sequences=True).cpu()[0].double()
        part = buf[n - tail:].view(torch.float32).cpu()
        logits, sq = part[:hidden // 8 * 64].reshape(-1, 64)[:, :experts].double(), part[hidden // 8 * 64:].double()
        terms = (sd[p + ".mlp.gate.weight"].double() * sd[p + ".post_attention_layernorm.weight"].double() * x[0].double()).T.reshape(-1, 8, experts)
        assert bool(((logits - terms.sum(1)).abs() <= 8 * 2.0 ** -24 * terms.abs().sum(1)).all())
        squares = (x[0].double() ** 2).reshape(-1, 8).sum(1)
        assert bool(((sq - squares).abs() <= 8 * 2.0 ** -24 * squares).all())
        want = want / torch.sqrt((want * want).mean() + cfg.rms_norm_eps) * sd["model.norm.weight"].double()
        # sums of up to `hidden` products in 64 chains and a tree, some 40 roundings of the terms' root sum of squares in a chain of five products
        assert float((got - want).norm() / want.norm()) < 1e-6, seed
    assert done >= 6
