"""The modulation projections of the bf16 path: in a launch of their own (larger batches) or taken along by the GEMM launches of the block before."""
import pytest
import torch

from gpu_util import BF16_REL_L2, M
from sd3_c_amd import lib as L
from sd3_c_amd.config import DiTConfig
from sd3_c_amd.params import block_param_shapes, dit_param_shapes

pytestmark = pytest.mark.gpu


def _weights(cfg):
    g = torch.Generator(device="cuda").manual_seed(11)
    return {n: (1 if "rmsnorm" in n else 0) + 0.05 * torch.randn(s, device="cuda", generator=g) for n, s in dit_param_shapes(cfg).items()}


# widths whose slices of K are 2, 6, 10, 48 and 68 deep (16 rows are in flight at a time); from one patch row to where tiles fill most compute units
@pytest.mark.parametrize("C,Tc,h,w", [(64, 1, 2, 3), (192, 9, 4, 5), (320, 77, 16, 16), (1536, 77, 16, 17), (1536, 154, 32, 32), (2176, 5, 16, 16)])
def test_modulation_of_a_batch_element_in_any_batch(C, Tc, h, w):
    """One to four batch elements have their modulation vectors computed by the launches of the block before, six by a launch of their own:
    every element has the same bits either way, whatever the tiles of those launches."""
    cfg = DiTConfig(num_layers=4, dual_attention_layers=(0, 2), emb_dim=C, attn_heads=C // 64, pooled_dim=64, captions_dim=64, pos_embed_max_size=64, base_height=32)
    P = _weights(cfg)
    g = torch.Generator(device="cuda").manual_seed(C + Tc)
    a = [torch.randn(s, device="cuda", generator=g) for s in ((6, 64), (6, Tc, 64), (6, 16, 2 * h, 2 * w))] + [1000 * torch.rand(6, device="cuda", generator=g)]
    den = M.Denoiser(P, cfg, "bf16")
    try:
        whole = den(*a).clone()
        exact = M.Denoiser(P, cfg, "fp32")
        want = exact(*a)
        assert float((whole - want).norm()) <= BF16_REL_L2 * float(want.norm())
        exact.ctx.close()
        for first, n in ((0, 1), (5, 1), (1, 2), (0, 3), (2, 4)):
            part = [t[first:first + n].contiguous() for t in a]
            for tile in (0, 64064, 256) if n == 1 else (0,):
                L.call("sd3_gemm_bf16_force_tile", tile)
                got = [den(*part).clone() for _ in range(2)]
                L.call("sd3_gemm_bf16_force_tile", 0)
                assert torch.equal(got[0], whole[first:first + n]) and torch.equal(got[1], got[0]), (first, n, tile)
    finally:
        L.call("sd3_gemm_bf16_force_tile", 0)
        den.ctx.close()


def test_modulation_weights_at_any_float():
    """A weight bound one float after a 16-byte boundary gives the bits of an aligned one."""
    B, Tc, Tx, C = 2, 3, 20, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    P = {k: 0.1 * torch.randn(s, device="cuda", generator=g) for k, s in block_param_shapes(C, 2, True, True, False, 64).items()}
    y, c, x = (torch.randn(s, device="cuda", generator=g) for s in ((B, C), (B, Tc, C), (B, Tx, C)))
    Q = dict(P)
    for k in P:
        if "ada_lnorm" in k:
            Q[k] = torch.empty(P[k].numel() + 1, device="cuda")[1:].view(P[k].shape).copy_(P[k])
    want, got = (M.Dit_block(y, c.clone(), x.clone(), p, B, Tc, Tx, C, 2, 2, True, True, False, precision="bf16") for p in (P, Q))
    assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])
