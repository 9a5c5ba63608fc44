"""Joint attention in bf16 beyond the short sequences: workgroups of 4 or 8 wavefronts with 32 queries each, and of 4 with 64."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd import lib as L
from sd3_c_amd.config import DiTConfig
from sd3_c_amd.params import dit_param_shapes

pytestmark = pytest.mark.gpu


def _attention(bufs, T0, T1, NH):
    B, C = bufs[1].shape[0], NH * 64
    out = [torch.zeros((B, t, C), device="cuda", dtype=torch.bfloat16) for t in (max(T0, 1), T1)]
    L.call("sd3_flash_attention_bf16", bufs[0].data_ptr() if T0 else None, bufs[1].data_ptr(), out[0].data_ptr() if T0 else None, out[1].data_ptr(), None, None,
           None, None, B, T0, T1, NH, 64, None)
    torch.cuda.synchronize()
    return torch.cat([out[0][:, :T0], out[1]], 1)


# Heads and batches on either side of one 128-query workgroup per compute unit, one of 256 queries per unit, and two of 128.
@pytest.mark.parametrize("B,T0,T1,NH,kind", [(12, 0, 417, 32, "plain"), (6, 1, 447, 48, "plain"), (6, 0, 448, 48, "plain"), (7, 65, 448, 24, "plain"),
                                             (5, 77, 544, 24, "plain"), (3, 154, 1024, 24, "plain"), (5, 77, 544, 24, "growing"), (5, 77, 544, 24, "low"),
                                             (5, 77, 544, 24, "loud"), (3, 154, 1024, 24, "loud"), (3, 0, 1088, 24, "growing")])
def test_attention_bf16_of_a_batch_element_alone(B, T0, T1, NH, kind):
    """A batch element has the bits it has alone or beside one other, which other kernels take: sequences of whole 64-key tiles, one key past them and
    one short of them. Keys that grow along the sequence (by 30), scores around -60 and single queries of 40 times the size start items
    again with the moving reference; the queries beside those keep theirs. Against fp32 softmax on the bf16 inputs: the bf16 rounding (2^-9) of the
    scaled queries, the probabilities and the output; a rounded query moves the scores of the other kinds by more."""
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + T1)
    bufs = [torch.randn((B, t, 3, NH, 64), device="cuda", generator=g) for t in (max(T0, 1), T1)]
    if kind == "growing":
        bufs[1][:, :, 1] *= torch.linspace(1.0, 30.0, T1, device="cuda").view(1, -1, 1, 1)
    if kind == "low":
        for t in bufs:
            t[:, :, 0, :, 0] = 16.0
            t[:, :, 1, :, 0] = -30.0
    if kind == "loud":
        bufs[1][:, 100, 0] *= 40.0
        bufs[1][:, T1 - 1, 0] *= 40.0
    bufs = [t.bfloat16() for t in bufs]
    got = _attention(bufs, T0, T1, NH)
    for e in (0, B - 1):
        assert torch.equal(_attention([t[e:e + 1].contiguous() for t in bufs], T0, T1, NH)[0], got[e]), e
    assert torch.equal(_attention([t[:2].contiguous() for t in bufs], T0, T1, NH), got[:2])
    x = torch.cat([bufs[0][:, :T0], bufs[1]], 1).float()
    q, k, v = (t.transpose(1, 2).contiguous() for t in x.unbind(2))
    want = (torch.softmax(q @ k.transpose(2, 3).contiguous() / 8, -1) @ v).transpose(1, 2).reshape(B, T0 + T1, NH * 64)
    assert torch.isfinite(got).all()
    assert float((got.float() - want).norm() / want.norm()) <= (1e-2 if kind == "plain" else 3e-2)


@pytest.mark.parametrize("C,Tc,h,w", [(64, 1, 20, 21), (192, 9, 32, 33), (320, 77, 20, 18), (1536, 154, 32, 34)])
def test_modulation_taken_along_by_attention(C, Tc, h, w):
    """One or two batch elements have modulation vectors of the next block computed in the attention launch's free compute units, six by a
    launch of their own: every element has the same bits either way."""
    cfg = DiTConfig(num_layers=3, dual_attention_layers=(0, 2), emb_dim=C, attn_heads=C // 64, pooled_dim=64, captions_dim=64, pos_embed_max_size=64, base_height=32)
    g = torch.Generator(device="cuda").manual_seed(C + Tc)
    P = {n: (1 if "rmsnorm" in n else 0) + 0.05 * torch.randn(s, device="cuda", generator=g) for n, s in dit_param_shapes(cfg).items()}
    a = [torch.randn(s, device="cuda", generator=g) for s in ((6, 64), (6, Tc, 64), (6, 16, 2 * h, 2 * w))] + [1000 * torch.rand(6, device="cuda", generator=g)]
    den = M.Denoiser(P, cfg, "bf16")
    try:
        whole = den(*a).clone()
        for first, n in ((0, 1), (5, 1), (2, 2)):
            part = [t[first:first + n].contiguous() for t in a]
            got = [den(*part).clone() for _ in range(2)]
            assert torch.equal(got[0], whole[first:first + n]) and torch.equal(got[1], got[0]), (first, n)
    finally:
        den.ctx.close()
