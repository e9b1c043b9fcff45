"""Lock-step rows of latent-cache models whose products read hi/lo rows the row kernels left (9 .. 64 rows in bf16 arithmetic).

test_steps: against the same steps operator by operator (a traced pass), where the products behind the norms split their rows themselves.  The rows' sums run over other
lanes in the two forms and nothing else differs: fp32 sums of at most 1000 values, 2e-5 of the largest value over two steps of two layers.  (The product behind the
polynomial takes split rows in both.)
test_against_the_oracle: all of them, the one behind the polynomial too (512 .. 8192 units), against float64.  Rows of hi/lo pairs are off by 2^-17 a value, seven products
one behind another: 1e-4 of the largest value; rows without their lo part, or with another row's, by 2^-9."""
import pytest
import torch

from tests import test_gpu_pizitar as P

pytestmark = pytest.mark.gpu

LA = dict(type="latent_attention", heads=2, dim=24, vdim=16, kv_rank=40, q_rank=24)
LB = dict(type="latent_attention_2", heads=2, dim=16, vdim=24, kv_rank=72)


@pytest.mark.parametrize("rows", [9, 32, 33, 64])
@pytest.mark.parametrize("width,ff,taps", [(64, 512, 3), (64, 72, 1), (520, 1000, 4), (48, 8192, 8), (48, 8200, 2), (44, 600, 2), (64, 510, 2)])
def test_steps(rows, width, ff, taps, monkeypatch):
    monkeypatch.setitem(P.MODELS, "split", dict(layers=[dict(LA, ff=ff), dict(LB, ff=ff)], width=width, vocab=40, taps=taps))
    cfg, _, fused = P.make("split", arith="bf16", t_max=8, n_seq=rows)
    _, _, plain = P.make("split", arith="bf16", t_max=8, n_seq=rows)
    for t in range(2):
        ids = torch.tensor(P.toks(cfg, rows, t), device="cuda")
        spans = [(rows - 1 - i, 1, t) for i in range(rows)]
        got, want = fused.forward_spans(fused.embed(ids), spans), plain.forward_spans(plain.embed(ids), spans, trace=True)[0]
        assert P.err(got, want.cpu()) < 2e-5, t


@pytest.mark.parametrize("rows", [33, 64])
@pytest.mark.parametrize("width,ff,taps", [(64, 512, 3), (520, 1000, 4), (48, 8192, 8)])
def test_against_the_oracle(rows, width, ff, taps, monkeypatch):
    monkeypatch.setitem(P.MODELS, "split", dict(layers=[dict(LA, ff=ff), dict(LB, ff=ff)], width=width, vocab=40, taps=taps))
    cfg, sd, dec = P.make("split", arith="bf16", t_max=8, n_seq=rows)
    ids = [P.toks(cfg, rows, t) for t in range(2)]
    for t in range(2):
        got = dec.forward_spans(dec.embed(torch.tensor(ids[t], device="cuda")), [(rows - 1 - i, 1, t) for i in range(rows)])
        want = []
        for i in range(rows):
            x, d = P.O.run_layers(cfg, sd, [ids[u][i] for u in range(t + 1)])
            want.append(P.O.affine_layer_norm(x[-1], d["final.norm"], d["final.norm.b"], cfg["norm"]["eps"]))
        want = torch.stack(want)
        off = (got.double().cpu() - want).abs().amax(1) / want.abs().max()
        assert float(off.max()) < 1e-4, (t, off)
