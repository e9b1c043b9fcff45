"""The calls whose speed users of this package see, each at the size and with the options of one real use.

A case is a dict of plain values.  `listed()` names the fixed ones, `draw(rng)` gives another of the same ranges, `prepare` makes what a
program holds before the call (weights, caches, inputs), `run` is the call, `exact` the same outputs in float64 from plain torch.

Kinds of cases
  recon      MingTok image -> latent -> semantic tokens -> image, in the bf16 regime: tokenizing and reconstructing image batches
  features   MingTok image -> semantic tokens, fp32-class: what feeds the language model in image understanding and editing
  prompt     a prompt (its middle an image, routed by the image gate) through the 28-layer 16B-A3B decoder, logits of its last token
  chat       one new token for every one of `rows` conversations: embedding, decoder step, logits
  image      one visual token for `images` images in lock-step: decoder step of the guidance rows, flow sampler, semantic decoder step.
             guidance 2: text to image; 3: editing
  pizitar, zuzenex, daberax: the other decoders' prompts and lock-step decode steps at the sizes their benchmark uses

The decoder's weights are random with two things as a trained model has them: the sublayers' outputs are small beside the residual stream
(output projections scaled by 1 / sqrt(2 layers)), and a token's experts are clear choices (its embedding has six directions of the
gates' rows in it), so that results do not hang on ties of a random router.
"""
import math

import torch

F64 = torch.float64
DEV = "cuda"

# ---- sizes -------------------------------------------------------------------------------------------------------------------------
# the 16B-A3B decoder, its flow head, the tokenizer
LLM = dict(hidden=2048, layers=28, n_q=16, n_kv=4, hd=128, experts=64, top=6, shared=2, inter=1408, vocab=126464, theta=600000.0, eps=1e-5)
RF = dict(w=3072, depth=12, hidden=8192, steps=16, target=32, text_cfg=3.0, image_cfg=1.1)
TOK = dict(enc_dim=768, enc_depth=12, patch=32, latent=32, sem_dim=1024, sem_depth=24, pix_dim=1024, pix_depth=24, pix_patch=16, grid=16,
           mean=1.46817409, scale=8.09449291)
# the sizes of the other decoders' benchmark (4 layers each)
LM = {1024: dict(heads=8, kv_rank=256, q_rank=384, ff=4096, vocab=32000), 2048: dict(heads=16, kv_rank=512, q_rank=768, ff=8192, vocab=32000)}


def listed():
    return [
        # one 256^2 picture through the tokenizer: the smallest call, some 200 short launches
        dict(name="recon_one_256", kind="recon", images=1, side=256),
        # a data-set pass: 64 pictures of 256^2
        dict(name="recon_batch_256", kind="recon", images=64, side=256),
        # a 1024^2 picture on its way into a question about it
        dict(name="features_one_1024", kind="features", images=1, height=1024, width=1024),
        # that question: 12 text tokens, the picture's 1026, 20 text tokens
        dict(name="prompt_picture", kind="prompt", tokens=1058, image_tokens=1024),
        # its answer, token by token, for one user
        dict(name="chat_one", kind="chat", rows=1, context=1100),
        # the same for 64 conversations in lock-step
        dict(name="chat_64", kind="chat", rows=64, context=1100),
        # text to image for one user (two guidance rows)
        dict(name="image_one", kind="image", images=1, guidance=2, prompt=40, made=40),
        # a dozen edits in lock-step (three guidance rows each, a prompt that holds a picture)
        dict(name="image_edit_12", kind="image", images=12, guidance=3, prompt=310, made=17),
        # offline generation: 768 images in lock-step
        dict(name="image_768", kind="image", images=768, guidance=2, prompt=40, made=40),
        # a long prompt of the hybrid decoder (softmax attention and decayed linear attention)
        dict(name="zuzenex_prompt_2048", kind="zuzenex", width=2048, phase="prompt", tokens=2048, sequences=1),
        # five prompts of unequal length in one pass of the post-norm decoder (latent attention, delta rule, windowed attention)
        dict(name="daberax_prompts_ragged", kind="daberax", width=1024, phase="prompt", tokens=1409, sequences=5),
        # 32 conversations of the latent-attention decoder, one new token each
        dict(name="pizitar_chat_32", kind="pizitar", width=2048, phase="chat", sequences=32, context=2048),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["recon", "features", "prompt", "chat", "chat", "image", "image", "zuzenex", "zuzenex", "daberax", "pizitar", "pizitar"])
    if kind == "recon":
        side = 32 * rng.choice([2, 4, 5, 7, 8, 11, 16])
        return dict(kind=kind, images=_log(rng, 1, max(1, 64 * 256 * 256 // (side * side))), side=side)
    if kind == "features":
        return dict(kind=kind, images=rng.choice([1, 1, 2, 3]), height=32 * rng.randint(7, 32), width=32 * rng.randint(7, 32))
    if kind == "prompt":
        t = _log(rng, 9, 1800)
        return dict(kind=kind, tokens=t, image_tokens=rng.choice([0, t // 2, max(0, t - 33)]))
    if kind == "chat":
        return dict(kind=kind, rows=_log(rng, 1, 64), context=_log(rng, 17, 1900))
    if kind == "image":
        n, g = _log(rng, 1, 600), rng.choice([2, 2, 3])
        n = min(n, 1200 // g)
        p = rng.randint(24, 60) if g == 2 or n > 60 else rng.randint(100, 330)
        return dict(kind=kind, images=n, guidance=g, prompt=p, made=rng.randint(0, 60))
    width = rng.choice([1024, 2048])
    if kind != "daberax" and rng.random() < 0.5:
        return dict(kind=kind, width=width, phase="chat", sequences=_log(rng, 1, 64), context=_log(rng, 33, 2048))
    t = _log(rng, 33, 2048)
    return dict(kind=kind, width=width, phase="prompt", tokens=t, sequences=rng.choice([1, 1, 2, 5]))


# ---- random tensors ------------------------------------------------------------------------------------------------------------------
class Source:
    """Normal tensors on the GPU, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def bf16(self, *shape, std=None, mean=0.0):
        std = shape[-1] ** -0.5 if std is None else std
        return torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(mean, std, generator=self.g)

    def f32(self, *shape, std=1.0):
        return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, std, generator=self.g)

    def ids(self, n, top):
        return torch.randint(0, top, (n,), device=DEV, generator=self.g)

    def perm(self, n):
        return torch.randperm(n, device=DEV, generator=self.g)

    def expert_sets(self, n):
        """[n, experts] with `top` ones in every row."""
        u = torch.rand(n, LLM["experts"], device=DEV, generator=self.g)
        return torch.zeros_like(u).scatter_(1, u.topk(LLM["top"], 1).indices, 1.0)


# ---- the 16B-A3B decoder -------------------------------------------------------------------------------------------------------------
CLEAR = 8.0          # length of a token's component along each of its experts' gate directions, in standard deviations of the rest


def decoder_tensors(src, vocab):
    c = LLM
    H, out = c["hidden"], (2.0 * c["layers"]) ** -0.5
    dirs = src.f32(c["experts"], H, std=1.0)
    dirs = dirs / dirs.norm(dim=1, keepdim=True)
    gate = lambda: (0.3 * dirs[src.perm(c["experts"])]).to(torch.bfloat16)  # noqa: E731
    layers = []
    for _ in range(c["layers"]):
        n = c["experts"] + c["shared"]
        layers.append(dict(
            ln1=src.bf16(H, std=0.02, mean=1.0), wqkv=src.bf16((c["n_q"] + 2 * c["n_kv"]) * c["hd"], H),
            wdense=src.bf16(H, c["n_q"] * c["hd"], std=out * H ** -0.5), ln2=src.bf16(H, std=0.02, mean=1.0), gate=gate(), image_gate=gate(),
            w_gate_up=src.bf16(n, 2 * c["inter"], H), w_down=src.bf16(n, H, c["inter"], std=out * c["inter"] ** -0.5)))
    t = dict(layers=layers, dirs=dirs, norm=src.bf16(H, std=0.02, mean=1.0))
    if vocab:
        t["embed"] = torch.cat([(src.f32(n, H) + CLEAR * src.expert_sets(n) @ dirs).to(torch.bfloat16) for n in (c["vocab"] // 2,) * 2])
        t["head"] = src.bf16(c["vocab"], H)
    return t


def token_rows(src, dirs, n):
    return (src.f32(n, LLM["hidden"]) + CLEAR * src.expert_sets(n) @ dirs).contiguous()


def make_decoder(t, t_max, n_seq):
    from ming_univision_amd.bailing_moe import BailingMoeDecoder
    from ming_univision_amd.configuration import BailingMoeConfig
    return BailingMoeDecoder(BailingMoeConfig.ming_univision_16b_a3b(), t["layers"], t["norm"], t.get("embed"), t.get("head"), t_max=t_max, n_seq=n_seq)


def lin(x, w, b=None):
    y = x @ w.to(F64).T
    return y if b is None else y + b.to(F64)


def rms(x, w, eps):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.to(F64)


def ln(x, w, b, eps=1e-6):
    c = x - x.mean(-1, keepdim=True)
    y = c / torch.sqrt((c * c).mean(-1, keepdim=True) + eps)
    y = y if w is None else y * w.to(F64)
    return y if b is None else y + b.to(F64)


def silu(x):
    return x * torch.sigmoid(x)


def gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x * 0.5 ** 0.5))


def gelu_tanh(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def turn_halves(x, pos, theta):
    """x [M, h, hd], pos [M]: rotary embedding over the two halves of a head."""
    hd = x.shape[-1]
    inv = 1.0 / (theta ** (torch.arange(0, hd, 2).float() / hd))                # fp32 tables, as the model defines them
    ang = torch.outer(torch.arange(int(pos.max()) + 1).float(), inv).to(x.device)[pos]
    c, s = ang.cos().to(F64)[:, None], ang.sin().to(F64)[:, None]
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def decoder_exact(t, x, pos, attend, image_rows=None):
    """The stack in float64: x [M, H], attend(layer, q [M, nq, hd], k, v [M, nkv, hd]) -> [M, nq, hd]."""
    c = LLM
    M = x.shape[0]
    for li, w in enumerate(t["layers"]):
        qkv = lin(rms(x, w["ln1"], c["eps"]), w["wqkv"]).reshape(M, c["n_q"] + 2 * c["n_kv"], c["hd"])
        q, k, v = qkv.split([c["n_q"], c["n_kv"], c["n_kv"]], 1)
        q, k = turn_halves(q, pos, c["theta"]) / math.sqrt(c["hd"]), turn_halves(k, pos, c["theta"])
        x = x + lin(attend(li, q, k, v).reshape(M, -1), w["wdense"])
        h = rms(x, w["ln2"], c["eps"])
        s = torch.softmax(lin(h, w["gate"]), -1)
        if image_rows is not None:
            s = torch.where(image_rows[:, None], torch.softmax(lin(h, w["image_gate"]), -1), s)
        wt, idx = s.topk(c["top"], -1)
        wt = wt / wt.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(c["experts"] + c["shared"]):
            if e < c["experts"]:
                r, j = (idx == e).nonzero(as_tuple=True)
                if not r.numel():
                    continue
                he, we = h[r], wt[r, j][:, None]
            else:
                r, he, we = torch.arange(M, device=x.device), h, 1.0
            gu = lin(he, w["w_gate_up"][e])
            y.index_add_(0, r, we * lin(silu(gu[:, :c["inter"]]) * gu[:, c["inter"]:], w["w_down"][e]))
        x = x + y
    return rms(x, t["norm"], c["eps"])


def grouped_softmax_sum(q, k, v, mask):
    """q [M, nq, hd] against k, v [M, T, nkv, hd], mask [M, T]."""
    M, nq, hd = q.shape
    g = k.shape[2]
    s = (q.reshape(M, g, nq // g, hd) @ k.permute(0, 2, 3, 1)).masked_fill(~mask[:, None, None], -math.inf)
    return (torch.softmax(s, -1) @ v.transpose(1, 2)).reshape(M, nq, hd)


def cached(kv, slots, mask):
    """attend() of decode rows: row r owns cache sequence r of kv [L, n_seq, 2, n_kv, t_max, hd], is slot slots and sees mask [M, slots + 1]."""
    def attend(li, q, k, v):
        out = []
        for r0 in range(0, q.shape[0], 256):
            r = slice(r0, min(q.shape[0], r0 + 256))
            n = r.stop - r.start
            old = kv[li, r, :, :, :slots].to(F64)
            ks = torch.cat([old[:, 0].transpose(1, 2), k[r].reshape(n, 1, -1, LLM["hd"])], 1)
            vs = torch.cat([old[:, 1].transpose(1, 2), v[r].reshape(n, 1, -1, LLM["hd"])], 1)
            out.append(grouped_softmax_sum(q[r], ks, vs, mask[r]))
        return torch.cat(out)
    return attend


# prompt
def prompt_inputs(case, seed):
    src = Source(seed)
    t = decoder_tensors(src, vocab=False)
    t["head"] = src.bf16(LLM["vocab"], LLM["hidden"])
    n, m = case["tokens"], case["image_tokens"]
    image = torch.zeros(n, dtype=torch.bool, device=DEV)
    lead = min(13, n - m)
    image[lead:lead + m] = True
    return t, token_rows(src, t["dirs"], n), (image if m else None)


def prepare_prompt(case, seed):
    t, x, image = prompt_inputs(case, seed)
    return dict(dec=make_decoder(t, case["tokens"] + 64, 1), x=x, image=image)


def run_prompt(s):
    # as the conversation class does: up to 64 tokens through the decode kernels, longer prompts as matrix products
    step = s["dec"].prefill if s["x"].shape[0] <= 64 else s["dec"].prefill_wide
    hidden = step(s["x"], seq=0, past=0, image_mask=s["image"])
    return dict(hidden=hidden, logits=s["dec"].logits(hidden[-1:].contiguous()))


def exact_prompt(case, seed):
    t, x, image = prompt_inputs(case, seed)
    n = x.shape[0]
    see = torch.ones(n, n, dtype=torch.bool, device=DEV).tril()

    def attend(li, q, k, v):
        rep = LLM["n_q"] // LLM["n_kv"]
        out = [torch.softmax((q[:, h] @ k[:, h // rep].T).masked_fill(~see, -math.inf), -1) @ v[:, h // rep] for h in range(LLM["n_q"])]
        return torch.stack(out, 1)
    hidden = decoder_exact(t, x.to(F64), torch.arange(n, device=DEV), attend, image)
    return dict(hidden=hidden, logits=lin(hidden[-1:], t["head"]))


# chat
def chat_inputs(case, seed):
    src = Source(seed)
    t = decoder_tensors(src, vocab=True)
    kv = src.f32(LLM["layers"], case["rows"], 2, LLM["n_kv"], case["context"] + 24, LLM["hd"])
    return t, kv, src.ids(case["rows"], LLM["vocab"])


def prepare_chat(case, seed):
    t, kv, ids = chat_inputs(case, seed)
    n = case["rows"]
    dec = make_decoder(t, kv.shape[4], n)
    dec.kv_cache.copy_(kv)
    slot = torch.full((n,), case["context"], dtype=torch.int32, device=DEV)
    return dict(dec=dec, ids=ids, seq=torch.arange(n, dtype=torch.int32, device=DEV), slot=slot, len=slot + 1)


def run_chat(s):
    dec = s["dec"]
    hidden = dec.step(dec.embed(s["ids"]), s["seq"], s["slot"], s["slot"], s["len"], distinct_sequences=True)
    return dict(hidden=hidden, logits=dec.logits(hidden))


def exact_chat(case, seed):
    t, kv, ids = chat_inputs(case, seed)
    n, c = case["rows"], case["context"]
    mask = torch.ones(n, c + 1, dtype=torch.bool, device=DEV)
    hidden = decoder_exact(t, t["embed"][ids].to(F64), torch.full((n,), c, device=DEV), cached(kv, c, mask))
    return dict(hidden=hidden, logits=lin(hidden, t["head"]))


# ---- one visual token ----------------------------------------------------------------------------------------------------------------
def flow_tensors(src):
    w, h, n = RF["w"], RF["hidden"], "diffloss.net."
    sd = {"vis_head.0.weight": src.bf16(w, LLM["hidden"]), "vis_head.0.bias": src.bf16(w, std=0.02),
          "vis_head.1.weight": src.bf16(w, std=0.02, mean=1.0), "vis_head.1.bias": src.bf16(w, std=0.02)}
    shapes = {"time_embed.mlp.0": (w, 256), "time_embed.mlp.2": (w, w), "cond_embed": (w, w), "input_proj": (w, RF["target"]),
              "final_layer.linear": (RF["target"], w), "final_layer.adaLN_modulation.1": (2 * w, w)}
    for i in range(RF["depth"]):
        b = f"res_blocks.{i}."
        shapes.update({b + "mlp.w12": (2 * h, w), b + "mlp.w3": (w, h), b + "adaLN_modulation.1": (3 * w, w)})
        sd[n + b + "in_ln.weight"], sd[n + b + "in_ln.bias"] = src.bf16(w, std=0.02, mean=1.0), src.bf16(w, std=0.02)
    for k, shp in shapes.items():
        sd[n + k + ".weight"], sd[n + k + ".bias"] = src.bf16(*shp), src.bf16(shp[0], std=0.02)
    return sd


def flow_exact(sd, hidden, noise, guidance):
    """hidden [images * guidance, H] -> latents [images, target]."""
    L = lambda x, k: lin(x, sd["diffloss.net." + k + ".weight"], sd["diffloss.net." + k + ".bias"])  # noqa: E731
    z = ln(lin(hidden, sd["vis_head.0.weight"], sd["vis_head.0.bias"]), sd["vis_head.1.weight"], sd["vis_head.1.bias"])
    cond = L(z, "cond_embed")
    x, B = noise.to(F64), noise.shape[0]
    ts = torch.linspace(1.0, 0.0, RF["steps"] + 1)[:-1] * 1000.0
    freqs = torch.exp(-math.log(10000.0) * torch.arange(0, 128, dtype=torch.float32) / 128)
    for t in ts:
        a = (t * freqs)[None]
        y = silu(L(silu(L(torch.cat([a.cos(), a.sin()], -1).to(DEV, F64), "time_embed.mlp.0")), "time_embed.mlp.2") + cond)
        h = L(x.repeat_interleave(guidance, 0), "input_proj")
        for i in range(RF["depth"]):
            b = f"res_blocks.{i}."
            shift, scale, gate = L(y, b + "adaLN_modulation.1").chunk(3, -1)
            u = ln(h, sd["diffloss.net." + b + "in_ln.weight"], sd["diffloss.net." + b + "in_ln.bias"]) * (1 + scale) + shift
            p, q = L(u, b + "mlp.w12").chunk(2, -1)
            h = h + gate * L(silu(p) * q, b + "mlp.w3")
        shift, scale = L(y, "final_layer.adaLN_modulation.1").chunk(2, -1)
        v = L(ln(h, None, None) * (1 + scale) + shift, "final_layer.linear").reshape(B, guidance, -1)
        if guidance == 3:
            v = v[:, 1] + RF["image_cfg"] * (v[:, 2] - v[:, 1]) + RF["text_cfg"] * (v[:, 0] - v[:, 2])
        else:
            v = v[:, 1] + RF["text_cfg"] * (v[:, 0] - v[:, 1])
        x = x + v / RF["steps"]
    return x


def image_masks(case):
    """[guidance, prompt + made + 1] of every image: the unconditional row does not see the prompt's text, the text-unconditional one not a part of it."""
    p, n = case["prompt"], case["prompt"] + case["made"] + 1
    m = torch.ones(case["guidance"], n, dtype=torch.long)
    m[1, 2:p - 2] = 0
    if case["guidance"] == 3:
        m[2, 2:8] = 0
    return m


def image_inputs(case, seed):
    src = Source(seed)
    t = decoder_tensors(src, vocab=False)
    B, rows = case["images"], case["images"] * case["guidance"]
    past = case["prompt"] + case["made"]
    kv = src.f32(LLM["layers"], rows, 2, LLM["n_kv"], past + 16, LLM["hd"])
    sem_kv = src.f32(TOK["sem_depth"], B, 2, TOK["sem_dim"] // 64, case["made"] + 8, 64)
    D, H = TOK["sem_dim"], LLM["hidden"]
    proj = [(src.bf16(H, D), src.bf16(H, std=0.02)), (src.bf16(H, H), src.bf16(H, std=0.02))]
    return dict(t=t, kv=kv, sem_kv=sem_kv, x=token_rows(src, t["dirs"], B), noise=src.f32(B, RF["target"]), flow=flow_tensors(src),
                tok=tokenizer_tensors(src), proj=proj)


def prepare_image(case, seed):
    from ming_univision_amd import MingTok, MingTokConfig
    from ming_univision_amd.bailing_moe import ImageGenState
    from ming_univision_amd.rf_head import RectifiedFlowHead
    i = image_inputs(case, seed)
    rows, past = case["images"] * case["guidance"], case["prompt"] + case["made"]
    dec = make_decoder(i["t"], i["kv"].shape[4], rows)
    dec.kv_cache.copy_(i.pop("kv"))
    st = ImageGenState(dec, [image_masks(case)] * case["images"], [past] * case["images"])
    tok = MingTok(MingTokConfig(), state_dict=i["tok"], linear_proj=i["proj"])
    sem = tok.new_decode_state(n_seq=case["images"], t_max=i["sem_kv"].shape[4])
    sem.kv.copy_(i.pop("sem_kv"))
    return dict(dec=dec, rf=RectifiedFlowHead(i["flow"], LLM["hidden"]), tok=tok, st=st, sem=sem, x=i["x"], noise=i["noise"], made=case["made"],
                images=case["images"], guidance=case["guidance"])


def run_image(s):
    dec, st, sem, n = s["dec"], s["st"], s["sem"], s["images"]
    sem.row_slot.fill_(s["made"])                       # the same token again: back to its slot
    sem.row_len.fill_(s["made"] + 1)
    sem.length = s["made"]
    hidden = dec.step(s["x"], st.row_seq, st.row_slot, st.row_pos, st.row_len, st.key_mask, rows=n * s["guidance"], x_row_div=s["guidance"],
                      distinct_sequences=True)
    latent = s["rf"].sample(hidden, s["noise"], text_cfg=RF["text_cfg"], image_cfg=RF["image_cfg"], n_images=n)
    embed = torch.empty(n, LLM["hidden"], dtype=torch.float32, device=DEV)
    tokens = s["tok"].decode_step(latent, sem, embed_out=embed)
    return dict(hidden=hidden, latent=latent, tokens=tokens, embed=embed)


def exact_image(case, seed):
    i = image_inputs(case, seed)
    B, g, past = case["images"], case["guidance"], case["prompt"] + case["made"]
    m = image_masks(case).to(DEV)
    pos = (m.cumsum(-1) - 1)[:, -1].repeat(B)
    hidden = decoder_exact(i["t"], i["x"].to(F64).repeat_interleave(g, 0), pos, cached(i["kv"], past, m.bool().repeat(B, 1)))
    del i["t"], i["kv"]
    latent = flow_exact(i["flow"], hidden, i["noise"], g)
    sd, made = i["tok"], case["made"]
    x = sem_input(latent * TOK["scale"] + TOK["mean"], sd)
    nh = TOK["sem_dim"] // 64
    for li in range(TOK["sem_depth"]):
        def attend(q, k, v):
            old = i["sem_kv"][li, :, :, :, :made].to(F64)
            ks = torch.cat([old[:, 0], k.reshape(B, nh, 1, 64)], 2)
            vs = torch.cat([old[:, 1], v.reshape(B, nh, 1, 64)], 2)
            return (torch.softmax(q.reshape(B, nh, 1, 64) @ ks.transpose(2, 3), -1) @ vs).reshape(B, -1)
        x = vit_block(x, sd, f"semantic_decoder.blocks.0.{li}", attend)
    tokens = ln(x, sd["semantic_decoder.norm.weight"], sd["semantic_decoder.norm.bias"])
    (w0, b0), (w1, b1) = i["proj"]
    return dict(hidden=hidden, latent=latent, tokens=tokens, embed=lin(gelu(lin(tokens, w0, b0)), w1, b1))


# ---- the tokenizer -------------------------------------------------------------------------------------------------------------------
def swiglu_width(d):
    return (int(4 * d * 2 / 3) + 7) // 8 * 8


def tokenizer_tensors(src):
    sd = {}

    def linear(name, n, k):
        sd[name + ".weight"], sd[name + ".bias"] = src.bf16(n, k), src.bf16(n, std=0.02)

    def norm(name, d):
        sd[name + ".weight"], sd[name + ".bias"] = src.bf16(d, std=0.02, mean=1.0), src.bf16(d, std=0.02)

    def blocks(stem, depth, d, swiglu):
        for i in range(depth):
            p = f"{stem}.blocks.0.{i}."
            norm(p + "norm1", d)
            linear(p + "attn.qkv", 3 * d, d)
            linear(p + "attn.proj", d, d)
            norm(p + "norm2", d)
            if swiglu:
                linear(p + "mlp.w12", 2 * swiglu_width(d), d)
                linear(p + "mlp.w3", d, swiglu_width(d))
            else:
                linear(p + "mlp.fc1", 4 * d, d)
                linear(p + "mlp.fc2", d, 4 * d)
    c = TOK
    De, Ds, Dp, P = c["enc_dim"], c["sem_dim"], c["pix_dim"], c["patch"]
    e = "low_level_encoder."
    sd[e + "cls_token"], sd[e + "pos_embed"] = src.bf16(1, 1, De, std=0.02), src.bf16(1, c["grid"] ** 2 + 1, De, std=0.02)
    sd[e + "patch_embed.proj.weight"] = src.bf16(De, 3, P, P, std=(3 * P * P) ** -0.5)
    sd[e + "patch_embed.proj.bias"] = src.bf16(De, std=0.02)
    blocks("low_level_encoder", c["enc_depth"], De, True)
    norm(e + "out_norm", De)
    linear(e + "out_proj", c["latent"], De)
    linear("semantic_decoder.in_proj", Ds, c["latent"])
    blocks("semantic_decoder", c["sem_depth"], Ds, True)
    norm("semantic_decoder.norm", Ds)
    blocks("pixel_decoder", c["pix_depth"], Dp, False)
    norm("pixel_decoder.norm", Dp)
    linear("pixel_decoder.head", c["pix_patch"] ** 2 * 3, Dp)
    linear("sem_to_pix", Dp * (P // c["pix_patch"]) ** 2, Ds)
    return sd


def pictures(src, n, h, w):
    """Smooth pictures with some grain, in [-1, 1]."""
    coarse = torch.nn.functional.interpolate(src.f32(n, 3, 8, 8, std=0.6), size=(h, w), mode="bilinear", align_corners=False)
    return (coarse + src.f32(n, 3, h, w, std=0.08)).clamp_(-1, 1).contiguous()


def tokenizer_inputs(case, seed):
    src = Source(seed)
    sd = tokenizer_tensors(src)
    h = case.get("height", case.get("side"))
    return sd, pictures(src, case["images"], h, case.get("width", h))


def prepare_tokenizer(case, seed):
    from ming_univision_amd import MingTok, MingTokConfig
    sd, px = tokenizer_inputs(case, seed)
    return dict(tok=MingTok(MingTokConfig(), state_dict=sd), px=px, kind=case["kind"])


def run_tokenizer(s):
    if s["kind"] == "recon":
        return s["tok"].forward_enc_dec(s["px"])
    return s["tok"].forward(s["px"], precision="fp32")


def vit_block(x, sd, p, attend):
    """x [rows, D]; attend(q, k, v) of [rows, D] each, q scaled."""
    w = lambda k: (sd[f"{p}.{k}.weight"], sd[f"{p}.{k}.bias"])  # noqa: E731
    q, k, v = lin(ln(x, *w("norm1")), *w("attn.qkv")).chunk(3, -1)
    x = x + lin(attend(q * 0.125, k, v), *w("attn.proj"))
    h = ln(x, *w("norm2"))
    if p + ".mlp.w12.weight" in sd:
        a, b = lin(h, *w("mlp.w12")).chunk(2, -1)
        return x + lin(silu(a) * b, *w("mlp.w3"))
    return x + lin(gelu(lin(h, *w("mlp.fc1"))), *w("mlp.fc2"))


def whole(B, T, D, causal):
    see = torch.ones(T, T, dtype=torch.bool, device=DEV).tril() if causal else None

    def attend(q, k, v):
        q, k, v = (a.reshape(B, T, D // 64, 64) for a in (q, k, v))
        out = torch.empty(B, T, D // 64, 64, dtype=F64, device=DEV)
        for b in range(B):
            s = q[b].transpose(0, 1) @ k[b].permute(1, 2, 0)
            s = s if see is None else s.masked_fill(~see, -math.inf)
            out[b] = (torch.softmax(s, -1) @ v[b].transpose(0, 1)).transpose(0, 1)
        return out.reshape(B * T, D)
    return attend


def sem_input(latent, sd):
    return lin(latent, sd["semantic_decoder.in_proj.weight"], sd["semantic_decoder.in_proj.bias"]) + latent.repeat_interleave(TOK["sem_dim"] // TOK["latent"], -1)


def exact_tokenizer(case, seed):
    sd, px = tokenizer_inputs(case, seed)
    c, e = TOK, "low_level_encoder."
    B, _, h, w = px.shape
    P, De, Ds, Dp = c["patch"], c["enc_dim"], c["sem_dim"], c["pix_dim"]
    gh, gw = h // P, w // P
    cols = px.to(F64).reshape(B, 3, gh, P, gw, P).permute(0, 2, 4, 1, 3, 5).reshape(B, gh * gw, 3 * P * P)
    x = lin(cols, sd[e + "patch_embed.proj.weight"].reshape(De, -1), sd[e + "patch_embed.proj.bias"])
    pe = sd[e + "pos_embed"].float()
    if (gh, gw) != (c["grid"], c["grid"]):
        grid = pe[:, :-1].reshape(1, c["grid"], c["grid"], De).permute(0, 3, 1, 2).to(F64)
        grid = torch.nn.functional.interpolate(grid, mode="bicubic", scale_factor=((gh + 0.1) / c["grid"], (gw + 0.1) / c["grid"]))
        pe = torch.cat([grid.permute(0, 2, 3, 1).reshape(1, -1, De), pe[:, -1:].to(F64)], 1)
    T = gh * gw + 1
    x = (torch.cat([x, sd[e + "cls_token"].to(F64).expand(B, 1, De)], 1) + pe.to(F64)).reshape(B * T, De)
    for i in range(c["enc_depth"]):
        x = vit_block(x, sd, f"{e}blocks.0.{i}", whole(B, T, De, False))
    latent = x.reshape(B * T, c["latent"], -1).mean(-1) + lin(gelu(ln(x, sd[e + "out_norm.weight"], sd[e + "out_norm.bias"])),
                                                               sd[e + "out_proj.weight"], sd[e + "out_proj.bias"])
    x = sem_input(latent, sd)
    for i in range(c["sem_depth"]):
        x = vit_block(x, sd, f"semantic_decoder.blocks.0.{i}", whole(B, T, Ds, True))
    sem = ln(x, sd["semantic_decoder.norm.weight"], sd["semantic_decoder.norm.bias"]).reshape(B, T, Ds)[:, :-1]
    if case["kind"] == "features":
        return {"x_norm_patchtokens": sem, "latent": ((latent - c["mean"]) / c["scale"]).reshape(B, T, -1)}
    r, n = P // c["pix_patch"], (T - 1) * (P // c["pix_patch"]) ** 2
    x = lin(sem, sd["sem_to_pix.weight"], sd["sem_to_pix.bias"]).reshape(B, gh, gw, r, r, Dp).permute(0, 1, 3, 2, 4, 5).reshape(B * n, Dp)
    for i in range(c["pix_depth"]):
        x = vit_block(x, sd, f"pixel_decoder.blocks.0.{i}", whole(B, n, Dp, False))
    x = lin(ln(x, sd["pixel_decoder.norm.weight"], sd["pixel_decoder.norm.bias"]), sd["pixel_decoder.head.weight"], sd["pixel_decoder.head.bias"])
    p = c["pix_patch"]
    return x.reshape(B, gh * r, gw * r, p, p, 3).permute(0, 5, 1, 3, 2, 4).reshape(B, 3, h, w).clamp(-1, 1)


# ---- the other decoders ----------------------------------------------------------------------------------------------------------------
WINDOW = 1024


def lm_layers(case):
    c = LM[case["width"]]
    H, ff, W = c["heads"], c["ff"], case["width"]
    s = 128 ** -0.5
    if case["kind"] == "pizitar":
        mlp = dict(kind="dense", ff=ff)
        a = dict(type="latent_attention", mixer=dict(heads=H, dim=128, vdim=128, kv_rank=c["kv_rank"], q_rank=c["q_rank"], scale=s), mlp=mlp)
        b = dict(type="latent_attention_2", mixer=dict(heads=H, dim=128, vdim=128, kv_rank=c["kv_rank"], scale=s), mlp=mlp)
        return dict(width=W, vocab=c["vocab"], layers=[a, b, a, b], canon=dict(taps=4), norm=dict(eps=1e-6), logit_softcap=30.0)
    if case["kind"] == "zuzenex":
        mlp = dict(kind="dense", ff=ff * 3 // 2)
        a = dict(type="attention", mixer=dict(heads=H, kv_heads=H // 4, dim=128, vdim=128, scale=s, q_temp=dict(coef=0.1, every=1024)), mlp=mlp)
        b = dict(type="lightning", mixer=dict(heads=H, dim=128, vdim=128, decay=[1.0 - 2.0 ** (-5 - 4 * h / H) for h in range(H)]), mlp=mlp)
        return dict(width=W, vocab=c["vocab"], layers=[a, b, b, a], norm=dict(eps=1e-6))
    mlp = dict(kind="dense", ff=ff)
    a = dict(type="attention", mixer=dict(heads=H, kv_heads=H // 4, dim=128, vdim=128, scale=s, softcap=50.0, mask=dict(size=WINDOW),
                                          rot=dict(base=1000000.0, dims=128, scaling=dict(factor=8.0, low=1.0, high=4.0, original=8192))), mlp=mlp)
    b = dict(type="latent_attention", mixer=dict(heads=H, dim=128, rot_dim=64, vdim=128, kv_rank=c["kv_rank"], scale=192 ** -0.5,
                                                 mask=dict(size=WINDOW), rot=dict(base=10000.0, dims=64)), mlp=mlp)
    d = dict(type="delta", mixer=dict(heads=H, kv_heads=H // 2, dim=128, vdim=128, conv=4), mlp=mlp)
    return dict(width=W, vocab=c["vocab"], layers=[b, d, d, a], norm=dict(eps=1e-6), token_side=dict(dim=64), logit_scale=0.5)


def lm_shapes(kind, cfg):
    """{tensor name: shape} of a checkpoint."""
    W, V = cfg["width"], cfg["vocab"]
    s = {"embed": (V, W), "final.norm": (W,), "head": (V, W)}
    if kind == "pizitar":
        s["final.norm.b"] = (W,)
    if kind == "daberax":
        s["side.embed"] = (V, 64 * len(cfg["layers"]))
    for i, ly in enumerate(cfg["layers"]):
        m, ff, t = ly["mixer"], ly["mlp"]["ff"], ly["type"]
        H, d, e = m["heads"], m["dim"], m["vdim"]
        n = {"norm1": (W,), "mix.o": (W, H * e), "mlp.up": (ff, W), "mlp.down": (W, ff)}
        if kind == "pizitar":
            r = m["kv_rank"]
            n.update({"norm1.b": (W,), "norm1b": (W,), "norm1b.b": (W,), "norm2": (W,), "norm2.b": (W,), "norm2b": (W,), "norm2b.b": (W,), "mlp.act": (4,),
                      "rg1": (W, W), "rg1.b": (W,), "rg2": (W, W), "rg2.b": (W,), "canon1": (W, 4), "mix.dkv": (r, W), "mix.dkv.norm": (r,),
                      "mix.uk": (H * d, r), "mix.uv": (H * e, r)})
            n.update({"mix.dq": (m["q_rank"], W), "mix.dq.norm": (m["q_rank"],), "mix.uq": (H * d, m["q_rank"])} if t == "latent_attention" else
                     {"mix.q": (H * d, W), "mix.g": (H * e, W)})
        elif t == "latent_attention":
            r, R = m["rot_dim"], m["kv_rank"]
            n.update({"mix.q": (H * (d + r), W), "mix.dkv": (R + r, W), "mix.dkv.norm": (R,), "mix.uk": (H * d, R), "mix.uv": (H * e, R)})
        else:
            G = m.get("kv_heads", H)
            n.update({"mix.q": ((G if t == "delta" else H) * d, W), "mix.k": (G * d, W), "mix.v": ((H if t == "delta" else G) * e, W)})
        if kind == "daberax":
            n.update({"norm2": (W,), "mlp.gate": (ff, W), "side.gate": (64, W), "side.proj": (W, 64), "side.norm": (W,)})
            if t == "attention":
                n.update({"mix.q.b": (H * d,), "mix.k.b": (G * d,), "mix.v.b": (G * e,), "mix.o.b": (W,), "mix.q.norm": (H * d,), "mix.k.norm": (G * d,),
                          "mix.g": (H, W)})
            elif t == "delta":
                n.update({"mix.q.conv": (G * d, 4), "mix.k.conv": (G * d, 4), "mix.v.conv": (H * e, 4), "mix.b": (H, W), "mix.a": (H, W),
                          "mix.A_log": (H,), "mix.dt_bias": (H,), "mix.norm": (e,), "mix.g": (H * e, W)})
        elif kind == "zuzenex":
            n.update({"mix.q.norm": (d,), "mix.k.norm": (d,), "mix.sink": (H,)} if t == "attention" else {"mix.g": (H * e, W), "mix.norm": (H * e,)})
        s.update({f"l{i}.{k}": v for k, v in n.items()})
    return s


def lm_tensors(src, kind, cfg):
    sd = {}
    for k, shp in lm_shapes(kind, cfg).items():
        last = k.split(".")[-1]
        if k in ("embed", "side.embed"):
            sd[k] = src.bf16(*shp, std=1.0)
        elif last == "act":
            sd[k] = torch.tensor([0.6, 0.3, 0.2, 0.05], device=DEV, dtype=torch.bfloat16)
        elif last == "A_log":
            sd[k] = src.bf16(*shp, std=0.5, mean=-1.0)
        elif last in ("dt_bias", "sink"):
            sd[k] = src.bf16(*shp, std=1.0)
        elif last in ("conv", "canon1"):
            sd[k] = src.bf16(*shp, std=0.4)
        elif last == "b" and len(shp) == 1:
            sd[k] = src.bf16(*shp, std=0.05)
        elif len(shp) == 1:
            sd[k] = src.bf16(*shp, std=0.05, mean=1.0)
        else:
            sd[k] = src.bf16(*shp)
    return sd


def lm_lengths(case):
    """Unequal lengths that add up to `tokens`."""
    n, t = case["sequences"], case["tokens"]
    part = [1 + (i * 7 + 3) % 5 for i in range(n)]
    cut = [0]
    for i in range(n):
        cut.append(t * sum(part[:i + 1]) // sum(part))
    return [b - a for a, b in zip(cut, cut[1:])]


def lm_inputs(case, seed):
    src = Source(seed)
    cfg = lm_layers(case)
    sd = lm_tensors(src, case["kind"], cfg)
    if case["phase"] == "prompt":
        return cfg, sd, src.ids(case["tokens"], cfg["vocab"]), None
    n, c = case["sequences"], case["context"]
    ids = src.ids(n, cfg["vocab"])
    past = []
    for ly in cfg["layers"]:
        m = ly["mixer"]
        if ly["type"].startswith("latent"):
            past.append(dict(c=src.f32(n, c, m["kv_rank"]), taps=src.f32(n, 3, case["width"])))
        elif ly["type"] == "attention":
            past.append(dict(k=src.f32(n, c, m["kv_heads"] * 128), v=src.f32(n, c, m["kv_heads"] * 128)))
        else:
            past.append(dict(s=src.f32(n, m["heads"], 128, 128)))
    return cfg, sd, ids, past


def prepare_lm(case, seed):
    cfg, sd, ids, past = lm_inputs(case, seed)
    if case["kind"] == "pizitar":
        from ming_univision_amd.pizitar import PizitarConfig as Config, PizitarDecoder as Decoder
    elif case["kind"] == "zuzenex":
        from ming_univision_amd.zuzenex import ZuzenexConfig as Config, ZuzenexDecoder as Decoder
    else:
        from ming_univision_amd.daberax import DaberaxConfig as Config, DaberaxDecoder as Decoder
    n = case["sequences"]
    longest = case["context"] + 64 if past else case["tokens"] + 64
    dec = Decoder(Config(**cfg), sd, t_max=longest, n_seq=n, arith="bf16")
    if not past:
        lens = lm_lengths(case)
        last = torch.tensor(lens, device=DEV).cumsum(0) - 1
        return dict(dec=dec, ids=ids, spans=[(i, k, 0) for i, k in enumerate(lens) if k], last=last[torch.tensor(lens, device=DEV) > 0])
    c = case["context"]
    for i, p in enumerate(past):
        if "c" in p:
            dec.latent[i][:, :c] = p["c"]
            dec.taps_state[i] = p["taps"]
        elif "k" in p:
            dec.state_t[i]["k"][:, :c], dec.state_t[i]["v"][:, :c] = p["k"], p["v"]
        else:
            dec.state_t[i]["lin"].copy_(p["s"])
    slot = torch.full((n,), c, dtype=torch.int32, device=DEV)
    ln_ = slot + 1
    graph = dec.decode_graph(torch.arange(n, dtype=torch.int32, device=DEV), slot, ln_)
    return dict(dec=dec, ids=ids, graph=graph, slot=slot, len=ln_, context=c)


def run_lm(s):
    dec = s["dec"]
    if "spans" in s:
        hidden = dec.forward_spans(dec.embed(s["ids"]), s["spans"], tokens=s["ids"])
        return dict(hidden=hidden, logits=dec.logits(hidden[s["last"]]))
    s["slot"].fill_(s["context"])                       # the step advances its rows: back to the token after the context
    s["len"].fill_(s["context"] + 1)
    hidden = s["graph"].run(dec.embed(s["ids"]), s["context"] + 1, tokens=s["ids"])
    return dict(hidden=hidden, logits=dec.logits(hidden))


def turn_pairs(x, rot, pos):
    """x [T, h, n]: pairs (2i, 2i + 1) of the last axis by position times frequency i."""
    dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
    fr = []
    for i in range(dims // 2):
        f = base ** (-2.0 * i / dims)
        if sc:
            wave = 2.0 * math.pi / f
            u = min(1.0, max(0.0, (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])))
            f = (1.0 - u) * f / sc["factor"] + u * f
        fr.append(f)
    ang = pos.to(F64)[:, None] * torch.tensor(fr, dtype=F64, device=DEV)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., 0:dims:2], x[..., 1:dims:2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)


def seen(q, k, v, first, scale, window=None, softcap=None, sink=None):
    """q [T, H, d] at positions first .., k, v [first + T, G, .] from position 0."""
    T, H, _ = q.shape
    rep = H // k.shape[1]
    i, j = torch.arange(first, first + T, device=DEV)[:, None], torch.arange(k.shape[0], device=DEV)[None]
    see = (j <= i) if not window else (j <= i) & (i - j < window)
    out = []
    for h in range(H):
        s = (q[:, h] @ k[:, h // rep].T) * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        s = s.masked_fill(~see, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].to(F64).expand(T, 1)], 1)
        out.append(torch.softmax(s, -1)[:, :k.shape[0]] @ v[:, h // rep])
    return torch.stack(out, 1)


def filtered(x, w, before=None):
    """Causal filter of x [T, C] with w [C, taps]; before [taps - 1, C]: the rows ahead of it, newest first."""
    taps = w.shape[1]
    pad = torch.cat([torch.zeros(taps - 1, x.shape[1], dtype=F64, device=DEV) if before is None else before.to(F64).flip(0), x])
    return sum(pad[j:j + x.shape[0]] * w[:, j].to(F64) for j in range(taps))


def pizitar_layer(x, p, ly, past, eps, first, tokens):
    m, T = ly["mixer"], x.shape[0]
    H, d, e = m["heads"], m["dim"], m["vdim"]
    n = ln(x, p["norm1"], p["norm1.b"], eps)
    h = n + filtered(n, p["canon1"], past and past["taps"])
    q = lin(rms(lin(h, p["mix.dq"]), p["mix.dq.norm"], eps), p["mix.uq"]) if "q_rank" in m else lin(h, p["mix.q"])
    c = rms(lin(h, p["mix.dkv"]), p["mix.dkv.norm"], eps)
    c = torch.cat([past["c"].to(F64), c]) if past else c
    o = seen(q.reshape(T, H, d), lin(c, p["mix.uk"]).reshape(-1, H, d), lin(c, p["mix.uv"]).reshape(-1, H, e), first, m["scale"]).reshape(T, H * e)
    if "q_rank" not in m:
        o = o * torch.sigmoid(lin(h, p["mix.g"]))
    x = x + ln(torch.sigmoid(lin(n, p["rg1"], p["rg1.b"])) * lin(o, p["mix.o"]), p["norm1b"], p["norm1b.b"], eps)
    n = ln(x, p["norm2"], p["norm2.b"], eps)
    z, a = lin(n, p["mlp.up"]), p["mlp.act"].to(F64)
    y = lin(a[0] * rms(z, None, eps) + a[1] * rms(z * z, None, eps) + a[2] * rms(z ** 3, None, eps) + a[3], p["mlp.down"])
    return x + ln(torch.sigmoid(lin(n, p["rg2"], p["rg2.b"])) * y, p["norm2b"], p["norm2b.b"], eps)


def zuzenex_layer(x, p, ly, past, eps, first, tokens):
    m, T = ly["mixer"], x.shape[0]
    H, G, d = m["heads"], m.get("kv_heads", m["heads"]), m["dim"]
    h = rms(x, p["norm1"], eps)
    q, k, v = (lin(h, p["mix." + n]).reshape(T, -1, 128) for n in "qkv")
    if ly["type"] == "attention":
        pos = torch.arange(first, first + T, device=DEV)
        temp = 1.0 + m["q_temp"]["coef"] * torch.log(torch.div(pos + 1, m["q_temp"]["every"], rounding_mode="floor").to(F64) + 1.0)
        q, k = rms(q, p["mix.q.norm"], eps) * temp[:, None, None], rms(k, p["mix.k.norm"], eps)
        if past:
            k, v = (torch.cat([past[n].to(F64).reshape(-1, G, d), new]) for n, new in (("k", k), ("v", v)))
        o = seen(q, k, v, first, m["scale"], sink=p["mix.sink"]).reshape(T, -1)
    else:
        q, k, v = silu(q), silu(k), silu(v)
        dec = torch.tensor(m["decay"], dtype=torch.float32).to(DEV, F64)                  # the decays are fp32 numbers of the model
        i = torch.arange(T, device=DEV)
        gap = (i[:, None] - i[None]).clamp(min=0).to(F64)
        o = torch.empty(T, H, d, dtype=F64, device=DEV)
        for n in range(H):
            o[:, n] = ((q[:, n] @ k[:, n].T) * torch.where(i[:, None] >= i[None], dec[n] ** gap, 0.0)) @ v[:, n]
            if past:
                o[:, n] += (dec[n] ** (i + 1).to(F64))[:, None] * (q[:, n] @ past["s"][n].to(F64))
        o = rms(o.reshape(T, -1), p["mix.norm"], eps) * torch.sigmoid(lin(h, p["mix.g"]))
    return x + lin(o, p["mix.o"]) + lin(torch.relu(lin(h, p["mlp.up"])) ** 2, p["mlp.down"])


def delta_recurrence(q, k, v, beta, g):
    T, H, d = q.shape
    S = torch.zeros(H, d, v.shape[2], dtype=F64, device=DEV)
    out = torch.empty_like(v)
    for t in range(T):
        S = S * g[t, :, None, None]
        u = beta[t, :, None] * (v[t] - torch.matmul(k[t, :, None], S)[:, 0])
        S = torch.baddbmm(S, k[t, :, :, None], u[:, None])
        out[t] = torch.matmul(q[t, :, None], S)[:, 0]
    return out


def daberax_layer(x, p, ly, past, eps, first, tokens):
    m, T, t = ly["mixer"], x.shape[0], ly["type"]
    H, d, e = m["heads"], m["dim"], m["vdim"]
    pos = torch.arange(first, first + T, device=DEV)
    if t == "attention":
        q, k = (rms(lin(x, p["mix." + n], p[f"mix.{n}.b"]), p[f"mix.{n}.norm"], eps).reshape(T, -1, d) for n in "qk")
        v = lin(x, p["mix.v"], p["mix.v.b"]).reshape(T, -1, e)
        o = seen(turn_pairs(q, m["rot"], pos), turn_pairs(k, m["rot"], pos), v, 0, m["scale"], m["mask"]["size"], m["softcap"])
        y = lin((o * torch.sigmoid(lin(x, p["mix.g"]))[:, :, None]).reshape(T, -1), p["mix.o"], p["mix.o.b"])
    elif t == "latent_attention":
        R = m["kv_rank"]
        q, kv = lin(x, p["mix.q"]).reshape(T, H, -1), lin(x, p["mix.dkv"])
        c = rms(kv[:, :R], p["mix.dkv.norm"], eps)
        q = torch.cat([q[..., :d], turn_pairs(q[..., d:], m["rot"], pos)], -1)
        k = torch.cat([lin(c, p["mix.uk"]).reshape(T, H, d), turn_pairs(kv[:, None, R:], m["rot"], pos).expand(T, H, -1)], -1)
        y = lin(seen(q, k, lin(c, p["mix.uv"]).reshape(T, H, e), 0, m["scale"], m["mask"]["size"]).reshape(T, -1), p["mix.o"])
    else:
        q, k, v = (silu(filtered(lin(x, p["mix." + n]), p[f"mix.{n}.conv"])).reshape(T, -1, 128) for n in "qkv")
        q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5
        k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        rep = H // m["kv_heads"]
        g = torch.exp(-torch.exp(p["mix.A_log"].to(F64)) * torch.nn.functional.softplus(lin(x, p["mix.a"]) + p["mix.dt_bias"].to(F64)))
        o = delta_recurrence(q.repeat_interleave(rep, 1), k.repeat_interleave(rep, 1), v, torch.sigmoid(lin(x, p["mix.b"])), g)
        y = lin((rms(o, p["mix.norm"], eps) * silu(lin(x, p["mix.g"])).reshape(T, H, e)).reshape(T, -1), p["mix.o"])
    x = x + rms(y, p["norm1"], eps)
    x = x + rms(lin(gelu_tanh(lin(x, p["mlp.gate"])) * lin(x, p["mlp.up"]), p["mlp.down"]), p["norm2"], eps)
    return x + rms(lin(gelu_tanh(lin(x, p["side.gate"])) * p["side"][tokens].to(F64), p["side.proj"]), p["side.norm"], eps)


def exact_lm(case, seed):
    cfg, sd, ids, past = lm_inputs(case, seed)
    layer = dict(pizitar=pizitar_layer, zuzenex=zuzenex_layer, daberax=daberax_layer)[case["kind"]]
    eps, n = cfg["norm"]["eps"], case["sequences"]
    lens = lm_lengths(case) if past is None else [1] * n
    x = sd["embed"][ids].to(F64)
    for i, ly in enumerate(cfg["layers"]):
        p = {k[len(f"l{i}."):]: w for k, w in sd.items() if k.startswith(f"l{i}.")}
        if "side.embed" in sd:
            p["side"] = sd["side.embed"][:, 64 * i:64 * (i + 1)]
        rows, r = [], 0
        for b, k in enumerate(lens):
            if k:
                old = None if past is None else {key: w[b] for key, w in past[i].items()}
                rows.append(layer(x[r:r + k], p, ly, old, eps, 0 if past is None else case["context"], ids[r:r + k]))
            r += k
        x = torch.cat(rows)
    hidden = ln(x, sd["final.norm"], sd["final.norm.b"], eps) if "final.norm.b" in sd else rms(x, sd["final.norm"], eps)
    last = hidden if past is not None else hidden[[sum(lens[:i + 1]) - 1 for i in range(n) if lens[i]]]
    logits = lin(last, sd["head"]) * cfg.get("logit_scale", 1.0)
    cap = cfg.get("logit_softcap")
    return dict(hidden=hidden, logits=cap * torch.tanh(logits / cap) if cap else logits)


# ---- the interface ---------------------------------------------------------------------------------------------------------------------
KINDS = dict(recon=(prepare_tokenizer, run_tokenizer, exact_tokenizer), features=(prepare_tokenizer, run_tokenizer, exact_tokenizer),
             prompt=(prepare_prompt, run_prompt, exact_prompt), chat=(prepare_chat, run_chat, exact_chat),
             image=(prepare_image, run_image, exact_image), pizitar=(prepare_lm, run_lm, exact_lm), zuzenex=(prepare_lm, run_lm, exact_lm),
             daberax=(prepare_lm, run_lm, exact_lm))


def prepare(case, seed):
    with torch.no_grad():
        return dict(KINDS[case["kind"]][0](case, seed), call=KINDS[case["kind"]][1])


def run(state):
    return state["call"](state)


def exact(case, seed):
    with torch.no_grad():
        return KINDS[case["kind"]][2](case, seed)


def tolerance(case):
    """About four times the distance of the calls from `exact`: 60 blocks on bf16 activations (recon 0.010), products on bf16 operands (the other
    decoders 0.0048), operands of 16 or more bits (features 8e-6, prompt and chat 3.5e-6, image 2.9e-5: the sampler's guidance amplifies)."""
    return {"rel": dict(recon=0.03, features=4e-5, prompt=2e-5, chat=2e-5, image=1.2e-4).get(case["kind"], 0.02)}


# ---- what a call cannot do without -------------------------------------------------------------------------------------------------------
def decoder_work(rows, pairs_rows, context, vocab_rows):
    """rows through the stack, `pairs_rows` of them with experts of their own choice; context: keys a row reads from the cache (0: a prompt
    that attends itself)."""
    c = LLM
    H, I, L = c["hidden"], c["inter"], c["layers"]
    attn = (c["n_q"] + 2 * c["n_kv"]) * c["hd"] * H + H * c["n_q"] * c["hd"] + c["experts"] * H
    distinct = c["experts"] * (1.0 - (1.0 - c["top"] / c["experts"]) ** pairs_rows) + c["shared"]
    keys = context if context else (rows + 1) / 2
    line = 2 * c["n_kv"] * c["hd"] * 4
    n_bytes = L * (2 * (attn + distinct * 3 * H * I) + rows * line * (1 + (context or 0)))
    flops = L * rows * (2 * attn + 2 * (c["top"] + c["shared"]) * 3 * H * I + 4 * c["n_q"] * c["hd"] * keys)
    n_bytes += 2 * rows * H * 4
    if vocab_rows:
        n_bytes += 2 * c["vocab"] * H + 4 * c["vocab"] * vocab_rows
        flops += 2 * c["vocab"] * H * vocab_rows
    return n_bytes, flops


def vit_work(n_images, tokens, depth, d, swiglu, causal):
    p = 4 * d * d + (3 * d * swiglu_width(d) if swiglu else 8 * d * d)
    return 2 * depth * p, n_images * depth * (2 * tokens * p + 4 * tokens * tokens * d * (0.5 if causal else 1.0))


def lm_work(case):
    cfg, n, W = lm_layers(case), case["sequences"], case["width"]
    rows = case["tokens"] if case["phase"] == "prompt" else n
    lens = lm_lengths(case) if case["phase"] == "prompt" else []
    n_bytes, flops = 0.0, 0.0
    for k, shp in lm_shapes(case["kind"], cfg).items():
        if len(shp) == 2 and k not in ("embed", "side.embed", "head"):
            n_bytes += 2 * shp[0] * shp[1]
            flops += 2 * shp[0] * shp[1] * rows
    n_bytes += 2 * cfg["vocab"] * W + 4 * cfg["vocab"] * n + 8 * rows * W
    flops += 2 * cfg["vocab"] * W * n
    for ly in cfg["layers"]:
        m = ly["mixer"]
        H = m["heads"]
        if ly["type"] in ("lightning", "delta"):
            n_bytes += 4 * n * H * 128 * 128 * (1 if lens else 2)
            flops += (4 if ly["type"] == "lightning" else 6) * rows * H * 128 * 128
            continue
        win = (m.get("mask") or {}).get("size", 1 << 30)
        pairs = sum(sum(min(i + 1, win) for i in range(k)) for k in lens) if lens else n * min(win, case["context"] + 1)
        line = 4 * (m["kv_rank"] + m.get("rot_dim", 0) if "kv_rank" in m else 2 * m["kv_heads"] * 128)
        n_bytes += line * (rows if lens else pairs)
        flops += 2 * pairs * H * (m["dim"] + m.get("rot_dim", 0) + m["vdim"])
    return n_bytes, flops


def work(case):
    k = case["kind"]
    if k in ("recon", "features"):
        B, h = case["images"], case.get("height", case.get("side"))
        w = case.get("width", h)
        T = h * w // TOK["patch"] ** 2 + 1
        parts = [vit_work(B, T, TOK["enc_depth"], TOK["enc_dim"], True, False), vit_work(B, T, TOK["sem_depth"], TOK["sem_dim"], True, True)]
        edge = TOK["enc_dim"] * 3 * TOK["patch"] ** 2
        px = 4 * B * 3 * h * w
        io = px + 4 * B * T * (TOK["sem_dim"] + TOK["latent"])
        if k == "recon":
            n = 4 * (T - 1)
            parts.append(vit_work(B, n, TOK["pix_depth"], TOK["pix_dim"], False, False))
            edge += 4 * TOK["pix_dim"] * TOK["sem_dim"] + 4 * 3 * TOK["pix_patch"] ** 2 * TOK["pix_dim"]
            io = 2 * px
        return {"bytes": sum(p[0] for p in parts) + 2 * edge + io, "flops": sum(p[1] for p in parts) + 2 * B * T * edge}
    if k == "prompt":
        b, f = decoder_work(case["tokens"], case["tokens"], 0, 1)
    elif k == "chat":
        b, f = decoder_work(case["rows"], case["rows"], case["context"], case["rows"])
    elif k == "image":
        B, rows = case["images"], case["images"] * case["guidance"]
        b, f = decoder_work(rows, B, case["prompt"] + case["made"], 0)
        blocks = RF["depth"] * 3 * RF["hidden"] * RF["w"]
        once = (RF["depth"] * 3 + 2) * RF["w"] ** 2
        # the blocks do not fit any cache: every step of the sampler reads them again
        b += RF["steps"] * 2 * blocks + 2 * once + 2 * RF["w"] * (RF["w"] + LLM["hidden"])
        f += 2 * rows * (RF["steps"] * (blocks + once) + RF["w"] * (RF["w"] + LLM["hidden"]))
        D = TOK["sem_dim"]
        sem = 4 * D * D + 3 * D * swiglu_width(D)
        proj = LLM["hidden"] * (D + LLM["hidden"])
        b += 2 * (TOK["sem_depth"] * sem + proj) + 4 * B * TOK["sem_depth"] * 2 * D * (case["made"] + 1)
        f += 2 * B * (TOK["sem_depth"] * (sem + 2 * D * (case["made"] + 1)) + proj)
    else:
        b, f = lm_work(case)
    return {"bytes": b, "flops": f}
