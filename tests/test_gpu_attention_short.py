"""Joint attention over short sequences in bf16 (no fused norm): the kernels that take the keys in runs."""
import pytest
import torch

from gpu_util import M  # noqa: F401  (loads the package)
from sd3_c_amd import lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T0,T1,NH,spread", [(1, 0, 1, 1, 1.0), (2, 1, 31, 2, 1.0), (1, 32, 33, 3, 1.0), (2, 77, 256, 4, 1.0), (1, 160, 256, 2, 1.0),
                                               (1, 33, 383, 2, 1.0), (2, 20, 100, 2, 30.0)])
def test_short_attention_bf16(B, T0, T1, NH, spread):
    """One key, one query, wavefronts without keys, partly empty 32-key tiles of either segment, the longest sequence of the kernel, and keys
    that grow along the sequence so that the reference of the softmax has to move (spread). Against fp32 softmax on the bf16 inputs: bf16
    rounding (2^-9) of the scaled queries, the probabilities and the output; a rounded query moves a score by at most 2^-9 |q||k| / 8,
    i.e. the result by twice the largest such shift (1 for spread 1: |q||k| stays below 200, hence 2 * 2^-9 * 25 in the worst element)."""
    g = torch.Generator(device="cuda").manual_seed(T0 * 7 + T1)
    C = NH * 64
    bufs = [torch.randn((B, t, 3, NH, 64), device="cuda", generator=g) for t in (max(T0, 1), T1)]
    bufs[1][:, :, 1] *= torch.linspace(1.0, spread, T1, device="cuda").view(1, -1, 1, 1)
    bufs = [t.bfloat16() for t in bufs]
    out = [torch.zeros((B, t, C), device="cuda", dtype=torch.bfloat16) for t in (max(T0, 1), T1)]
    L.call("sd3_flash_attention_bf16", bufs[0].data_ptr() if T0 else None, bufs[1].data_ptr(), out[0].data_ptr() if T0 else None, out[1].data_ptr(), None, None,
           None, None, B, T0, T1, NH, 64, None)
    x = torch.cat([bufs[0][:, :T0], bufs[1]], 1).float()
    q, k, v = (t.transpose(1, 2).contiguous() for t in x.unbind(2))
    want = (torch.softmax(q @ k.transpose(2, 3).contiguous() / 8, -1) @ v).transpose(1, 2).reshape(B, T0 + T1, C)
    got = torch.cat([out[0][:, :T0], out[1]], 1).float()
    assert torch.isfinite(got).all()
    assert float((got - want).norm() / want.norm()) <= (1e-2 if spread == 1.0 else 3e-2)
    if spread == 1.0:
        assert float((got - want).abs().max()) <= 2 * 2.0 ** -9 * 25 + 2.0 ** -7 * float(v.abs().max())


def _attention(bufs, T0, T1, NH):
    B, C = bufs[1].shape[0], NH * 64
    out = [torch.zeros((B, t, C), device="cuda", dtype=torch.bfloat16) for t in (max(T0, 1), T1)]
    L.call("sd3_flash_attention_bf16", bufs[0].data_ptr() if T0 else None, bufs[1].data_ptr(), out[0].data_ptr() if T0 else None, out[1].data_ptr(), None, None,
           None, None, B, T0, T1, NH, 64, None)
    torch.cuda.synchronize()
    return torch.cat([out[0][:, :T0], out[1]], 1)


# batches beyond what is resident at once in the kernel that splits the keys (three workgroups of 32 queries per compute unit)
@pytest.mark.parametrize("B,T0,T1,NH,kind", [(40, 0, 1, 24, "plain"), (24, 1, 31, 24, "plain"), (14, 33, 32, 24, "plain"), (10, 0, 97, 24, "plain"),
                                             (8, 5, 124, 24, "plain"), (4, 77, 256, 24, "plain"), (3, 33, 383, 24, "plain"), (4, 77, 256, 24, "growing"),
                                             (3, 33, 383, 24, "growing"), (10, 20, 100, 24, "low"), (4, 77, 256, 24, "low")])
def test_short_attention_bf16_of_a_batch_element_alone(B, T0, T1, NH, kind):
    """A batch element has the bits it has alone, where the other kernel takes it: one to fourteen key tiles, query blocks of one to four
    wavefronts. Keys that grow along the sequence (by 30) move the references of single blocks of queries, scores around -60 that of every run's
    first tile. The batch against fp32 softmax on the bf16 inputs as above (a rounded query moves the scores of these kinds by more)."""
    g = torch.Generator(device="cuda").manual_seed(B * 1000 + T1)
    bufs = [torch.randn((B, t, 3, NH, 64), device="cuda", generator=g) for t in (max(T0, 1), T1)]
    if kind == "growing":
        bufs[1][:, :, 1] *= torch.linspace(1.0, 30.0, T1, device="cuda").view(1, -1, 1, 1)
    if kind == "low":
        for t in bufs:
            t[:, :, 0, :, 0] = 16.0
            t[:, :, 1, :, 0] = -30.0
    bufs = [t.bfloat16() for t in bufs]
    got = _attention(bufs, T0, T1, NH)
    for e in {0, B // 2, B - 1}:
        assert torch.equal(_attention([t[e:e + 1].contiguous() for t in bufs], T0, T1, NH)[0], got[e]), e
    x = torch.cat([bufs[0][:, :T0], bufs[1]], 1).float()
    q, k, v = (t.transpose(1, 2).contiguous() for t in x.unbind(2))
    want = (torch.softmax(q @ k.transpose(2, 3).contiguous() / 8, -1) @ v).transpose(1, 2).reshape(B, T0 + T1, NH * 64)
    assert torch.isfinite(got).all()
    assert float((got.float() - want).norm() / want.norm()) <= (1e-2 if kind == "plain" else 3e-2)
