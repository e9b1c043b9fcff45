"""Hi/lo products of up to 128 rows (tiles of 32, 48 and 64 rows, 64 and 128 columns): edges of the tiles in rows and columns, one K-tile up to more than
the LDS pipelines hold, every epilogue; and the flow sampler on both sides of the row counts its routes change at.  Tolerances as in test_gpu_gemm_tile."""
import pytest
import torch

from tests import test_gpu_gemm_tile as G

pytestmark = pytest.mark.gpu
dev_lib = G.dev_lib


@pytest.mark.parametrize("M", [1, 16, 31, 32, 33, 47, 48, 49, 63, 64, 65, 128, 129])
def test_rule(M):
    for N, K in ((4, 64), (60, 128), (132, 448), (1028, 1024), (8196, 320)):
        G.test_forms(M, N, K)


@pytest.mark.parametrize("M", [1, 32, 33, 65, 127, 128])
def test_rule_of_many_columns(M):
    """More workgroups than a round of the few-row tiles: 64 x 128, and from 65 rows 128 x 128 (32004 columns) and 256 x 256 ones (65532)."""
    for N, K in ((32004, 128), (65532, 512)):
        G.test_forms(M, N, K)


@pytest.mark.parametrize("form", [5, 6, 7])
def test_forms_in_turn(dev_lib, form):
    dev_lib.mn_gemm_tile_tune(form)
    for M, N, K in ((1, 4, 64), (31, 28, 128), (33, 36, 192), (48, 60, 256), (49, 68, 320), (65, 132, 384), (97, 516, 1024)):
        G.test_forms(M, N, K)


@pytest.mark.parametrize("rows, images", [(5, 5), (6, 3), (6, 2), (23, 23), (32, 16), (33, 11), (64, 32), (128, 64), (129, 43)])
def test_sampler(rows, images):
    """A flow head of whole tiles: the batch's rows against the same rows two images at a time."""
    from ming_univision_amd import configuration as C
    from ming_univision_amd.rf_head import RectifiedFlowHead
    from ming_univision_amd.synth import synth_state_dict
    w = 384                                          # six K-tiles a row: the rows of w12's operand lie seven apart
    shapes = {"vis_head.0.weight": (w, 128), "vis_head.0.bias": (w,), "vis_head.1.weight": (w,), "vis_head.1.bias": (w,)}
    shapes.update(C.rf_param_shapes(w, 2, w))
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(shapes, 3).items()}
    head = RectifiedFlowHead(sd, 128, dict(diffloss_w=w, diffloss_d=2, num_sampling_steps="4", gen_method="flow_matching_swiglu-4", vis_head_arch="linear2-norm"))
    g = torch.Generator(device="cuda").manual_seed(rows)
    per = rows // images
    hid, noise = torch.randn(rows, 128, generator=g, device="cuda"), torch.randn(images, 32, generator=g, device="cuda")
    whole = head.sample(hid, noise, text_cfg=3.0, image_cfg=1.1, n_images=images)
    for i in range(images):
        one = head.sample(hid[i * per:(i + 1) * per].contiguous(), noise[i:i + 1].contiguous(), text_cfg=3.0, image_cfg=1.1, n_images=1)
        assert float((whole[i] - one[0]).norm() / one.norm()) < 1e-4


@pytest.mark.parametrize("w, hidden, steps", [(384, 128, 4), (64, 1024, 1), (128, 256, 2), (384, 1024, 1), (960, 128, 1)])
@pytest.mark.parametrize("images", [3, 8, 11, 16])
def test_condition(images, w, hidden, steps):
    """The product before the blocks as one launch on fp32 rows, whose scratch is the modulations' memory, and on hi/lo rows where heads of one block and one step leave it
    too small (384 behind 1024 values; of 960 behind 128 it holds this product's scratch and not the next one's; widths of 64 and 128 have no whole tiles and take the
    streaming kernels): two rows an image against each image alone."""
    from ming_univision_amd import configuration as C
    from ming_univision_amd.rf_head import RectifiedFlowHead
    from ming_univision_amd.synth import synth_state_dict
    shapes = {"vis_head.0.weight": (w, hidden), "vis_head.0.bias": (w,), "vis_head.1.weight": (w,), "vis_head.1.bias": (w,)}
    shapes.update(C.rf_param_shapes(w, 1, w))
    sd = {k: v.to("cuda", torch.bfloat16) for k, v in synth_state_dict(shapes, 5).items()}
    head = RectifiedFlowHead(sd, hidden, dict(diffloss_w=w, diffloss_d=1, num_sampling_steps=str(steps), gen_method="flow_matching_swiglu-4", vis_head_arch="linear2-norm"))
    g = torch.Generator(device="cuda").manual_seed(images)
    hid, noise = torch.randn(2 * images, hidden, generator=g, device="cuda"), torch.randn(images, 32, generator=g, device="cuda")
    whole = head.sample(hid, noise, text_cfg=3.0, image_cfg=1.1, n_images=images)
    for i in range(images):
        one = head.sample(hid[2 * i:2 * i + 2].contiguous(), noise[i:i + 1].contiguous(), text_cfg=3.0, image_cfg=1.1, n_images=1)
        assert float((whole[i] - one[0]).norm() / one.norm()) < 1e-4


@pytest.mark.parametrize("M, N, K", [(16, 256, 8192), (32, 68, 4096), (23, 512, 3072), (96, 16384, 3072)])
def test_sums_in_two_chains(M, N, K):
    """Positive operands, whose partial sums grow: a sum over all of K in one chain of fp32 additions (eight products at a time, as the matrix instruction rounds) is off
    by twice what two chains of half the length are.  The tiles that took the flow head's few rows over from K-slices may not fall back to one."""
    from ming_univision_amd import ops
    g = torch.Generator().manual_seed(3)
    x, w = ((0.5 + 0.5 * torch.rand(r, K, generator=g)).to(torch.bfloat16) for r in (M, N))
    got = ops.gemm256(torch.stack([x, torch.zeros_like(x)]).cuda(), w.cuda(), None, "f32").cpu()
    off = lambda v, ref: float(((v.double() - ref) / ref).pow(2).mean().sqrt())  # noqa: E731
    few = min(N, 64)
    parts = torch.einsum("mbk,nbk->bmn", x.double().reshape(M, -1, 8), w[:few].double().reshape(few, -1, 8)).float()
    chain = torch.zeros(M, few)
    for p in parts:
        chain = chain + p
    assert off(got, x.double() @ w.double().T) < 0.75 * off(chain, x.double() @ w[:few].double().T)


def test_modulations_beyond_four_gib():
    """A head of so many blocks that the stacked modulation weights (230 x 3072 rows of 3072) pass 32-bit byte offsets: three images together against each alone."""
    from ming_univision_amd import configuration as C
    from ming_univision_amd.rf_head import RectifiedFlowHead
    w, g = 3072, torch.Generator(device="cuda").manual_seed(1)
    shapes = {"vis_head.0.weight": (w, 64), "vis_head.0.bias": (w,), "vis_head.1.weight": (w,), "vis_head.1.bias": (w,)}
    shapes.update(C.rf_param_shapes(w, 76, w, mlp_mult=1))
    gain = ("in_ln.weight", "vis_head.1.weight")
    sd = {k: torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(1.0 if k.endswith(gain) else 0.0, s[-1] ** -0.5 if len(s) > 1 else 0.02, generator=g)
          for k, s in shapes.items()}
    head = RectifiedFlowHead(sd, 64, dict(diffloss_w=w, diffloss_d=76, num_sampling_steps="1", gen_method="flow_matching_swiglu-1", vis_head_arch="linear2-norm"))
    assert 2 * head.t["ada_w"].numel() > 1 << 32
    hid, noise = torch.randn(6, 64, generator=g, device="cuda"), torch.randn(3, 32, generator=g, device="cuda")
    whole = head.sample(hid, noise, n_images=3)
    for i in range(3):
        one = head.sample(hid[2 * i:2 * i + 2].contiguous(), noise[i:i + 1].contiguous(), n_images=1)
        assert float((whole[i] - one[0]).norm() / one.norm()) < 1e-4
