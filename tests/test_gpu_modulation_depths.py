"""The panels of the bf16 modulation projections at every kind of depth: slices of K shorter than, as long as and longer than the groups of 16 rows that
are requested together."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd.config import DiTConfig
from sd3_c_amd.params import block_param_shapes, dit_param_shapes

pytestmark = pytest.mark.gpu


# slices of 2, 14, 16, 18, 24, 30, 32, 34, 76, 96 and 128 rows; the last two are as deep as eight rows of y and as the kernel allow
@pytest.mark.parametrize("C", [64, 448, 512, 576, 768, 960, 1024, 1088, 2432, 3072, 4096])
@pytest.mark.parametrize("B", [1, 2, 3, 9])
def test_gates_of_any_depth(C, B):
    """With zero residual streams, zero output weights and one bias of ones the block's outputs are gates, i.e. columns of y @ W + b: against float64 on the
    weights' bf16 values, within the bound of a sum of C products and a bias in fp32 in any order."""
    g = torch.Generator(device="cuda").manual_seed(C + B)
    shapes = block_param_shapes(C, 1, True, True, False, 64)
    W = {s: torch.randn(shapes[f"{s}_ada_lnorm.linear.weight"], device="cuda", generator=g) for s in ("context", "latent")}
    b = {s: torch.randn(shapes[f"{s}_ada_lnorm.linear.bias"], device="cuda", generator=g) for s in ("context", "latent")}
    y = torch.randn((B, C), device="cuda", generator=g)
    for ones, chunk in (("{}_attn_Wout.bias", 2), ("{}_mlp.lin2.bias", 5), ("{}_dual_attn_Wout.bias", 8)):
        P = {n: torch.zeros(s, device="cuda") for n, s in shapes.items()}
        for s in ("context", "latent"):
            P[f"{s}_ada_lnorm.linear.weight"], P[f"{s}_ada_lnorm.linear.bias"] = W[s], b[s]
            if ones.format(s) in P:
                P[ones.format(s)].fill_(1.0)
        c, x = torch.zeros((B, 1, C), device="cuda"), torch.zeros((B, 3, C), device="cuda")
        out = dict(zip(("context", "latent"), M.Dit_block(y, c, x, P, B, 1, 3, C, C // 64, 1, True, True, False, precision="bf16")))
        for s in ("context", "latent"):
            if ones.format(s) not in P:
                continue
            w, bias = W[s][:, chunk * C:(chunk + 1) * C].bfloat16().double(), b[s][chunk * C:(chunk + 1) * C].double()
            bound = (C + 2) * 2.0 ** -24 * (y.double().abs() @ w.abs() + bias.abs())
            assert ((out[s].double() - (y.double() @ w + bias)[:, None]).abs() <= bound[:, None]).all(), (s, chunk)


@pytest.mark.parametrize("C,B,Tc,h,w", [(768, 4, 77, 16, 16), (768, 3, 5, 18, 18), (256, 2, 20, 24, 25), (1536, 4, 154, 16, 16)])
def test_forwards_whose_launches_leave_little_room(C, B, Tc, h, w):
    """Launches that fill the device take few panels along; the blocks' remaining modulation vectors are then computed together. Batch elements have the
    bits that they have in a batch too large to take any along."""
    cfg = DiTConfig(num_layers=5, dual_attention_layers=(0, 3), emb_dim=C, attn_heads=C // 64, pooled_dim=64, captions_dim=64, pos_embed_max_size=64, base_height=32)
    g = torch.Generator(device="cuda").manual_seed(C + Tc)
    P = {n: (1 if "rmsnorm" in n else 0) + 0.05 * torch.randn(s, device="cuda", generator=g) for n, s in dit_param_shapes(cfg).items()}
    a = [torch.randn(s, device="cuda", generator=g) for s in ((B + 5, 64), (B + 5, Tc, 64), (B + 5, 16, 2 * h, 2 * w))] + [1000 * torch.rand(B + 5, device="cuda", generator=g)]
    den = M.Denoiser(P, cfg, "bf16")
    try:
        whole = den(*a).clone()
        part = [t[2:2 + B].contiguous() for t in a]
        for _ in range(2):
            assert torch.equal(den(*part), whole[2:2 + B])
    finally:
        den.ctx.close()
