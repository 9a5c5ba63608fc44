"""fp32 attention of f16 pieces at the edges of its tiles and of its choices, at any scale and beyond the range of the pieces, against float64 arithmetic and the
fp32 instruction."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd import lib as L
from test_gpu_f32_kernels import test_attention_f32 as check_attention

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _pieces_afterwards():
    yield
    L.call("sd3_tune", b"attention_f32_no_pieces", 0)


def inputs(seed, B, NH, hs, Tq, Tk):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((B, t, NH * hs), device="cuda", generator=g) for t in (Tq, Tk, Tk)]


def exact(q, k, v, NH):
    B, Tq, C = q.shape
    h = [t.double().view(B, -1, NH, C // NH).transpose(1, 2).contiguous() for t in (q, k, v)]
    out = torch.softmax(h[0] @ h[1].transpose(2, 3).contiguous() / (C // NH) ** 0.5, -1) @ h[2]
    return out.transpose(1, 2).reshape(B, Tq, C)


def on_fp32_instruction(*args):
    L.call("sd3_tune", b"attention_f32_no_pieces", 1)
    out = M.mha(*args)
    L.call("sd3_tune", b"attention_f32_no_pieces", 0)
    return out


@pytest.mark.parametrize("B,NH,hs,Tq,Tk", [(1, 64, 64, 65, 1), (1, 64, 64, 127, 31), (1, 64, 64, 128, 32), (1, 32, 64, 129, 33), (2, 64, 64, 129, 63), (1, 22, 64, 257, 97),
                                           (5, 64, 64, 65, 64), (5, 64, 64, 100, 1), (5, 64, 64, 128, 65), (3, 64, 64, 257, 191), (1, 12, 64, 512, 97), (1, 64, 128, 65, 33), (2, 32, 128, 129, 65),
                                           (5, 64, 128, 100, 127)])
def test_edges(B, NH, hs, Tq, Tk):
    """One key tile (a run without keys) to six, whole and not, query blocks of 64 and 128, the runs side by side (up to 256 blocks of 128 queries) and one after the other."""
    check_attention(B, NH, hs, Tq, Tk)


@pytest.mark.parametrize("Tk", [1, 32, 33, 333])
def test_an_element_alone_and_in_a_batch(Tk):
    """Blocks of 64 queries, of 128 and runs one after the other have the same bits."""
    NH, args = 24, inputs(Tk, 5, 24, 64, 333, Tk)
    whole = M.mha(*args, NH)
    for n in (1, 2, 3):
        assert torch.equal(M.mha(*(t[:n].contiguous() for t in args), NH), whole[:n])


@pytest.mark.parametrize("hs,NH", [(64, 24), (128, 24)])
@pytest.mark.parametrize("q_exponent,k_exponent,v_exponent", [(0, 0, 0), (-40, 40, -60), (30, -30, 60), (3, 0, 0)])
def test_scales(hs, NH, q_exponent, k_exponent, v_exponent):
    """The error against float64 is no larger than the fp32 instruction's at any scale, a head of zero values and rows of either sign of scale included (1.25 times it: the errors of
    two sums of the same products may differ)."""
    q, k, v = inputs(hs, 1, NH, hs, 400, 333)
    q, k, v = q * 2.0 ** q_exponent, k * 2.0 ** k_exponent, v * 2.0 ** v_exponent
    v[:, :, :hs] = 0
    k[:, :, hs:2 * hs] = 0
    q[:, 5] *= 1e-6
    want = exact(q, k, v, NH)
    got, before = M.mha(q, k, v, NH), on_fp32_instruction(q, k, v, NH)
    assert (got[:, :, :hs] == 0).all()
    assert float((got.double() - want).norm()) <= 1.25 * float((before.double() - want).norm())


@pytest.mark.parametrize("B", [1, 4])
@pytest.mark.parametrize("hs", [64, 128])
def test_infinities_nans_and_values_beyond_the_pieces(hs, B):
    """What the pieces cannot hold gives what the fp32 instruction gives (to rounding), and changes nothing in other heads: infinities and NaNs in q, k and v, values that
    grow by 2^20 past the tiles that were looked at, a K and a V whose first tiles are zero."""
    NH = 24
    q, k, v = inputs(hs + 1, B, NH, hs, 300, 333)
    plain = M.mha(q, k, v, NH)
    at = lambda h: slice(h * hs, (h + 1) * hs)
    q[0, 7, 0] = float("inf")
    q[0, 9, hs] = float("nan")
    k[0, 100, 2 * hs] = float("inf")
    k[0, 40, 3 * hs + 1] = float("nan")
    v[0, 50, 4 * hs + 2] = float("-inf")
    v[0, 332, 5 * hs + 3] = float("nan")
    v[0, 200:, at(6)] *= 2.0 ** 20
    k[0, 290:, at(7)] *= 2.0 ** 10
    v[0, :280, at(8)] = 0
    k[0, :280, at(9)] = 0
    got, want = M.mha(q, k, v, NH), on_fp32_instruction(q, k, v, NH)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    for h in range(10):
        g, w = got[0, :, at(h)], want[0, :, at(h)]
        fine = torch.isfinite(w)
        # scores of up to 2^10 * 30 carry errors of 2^-24 of that, and an output as many; elsewhere rounding
        assert float((g - w)[fine].abs().max() / w[fine].abs().max()) <= (2e-2 if h == 7 else 1e-5) if fine.any() else True
    assert torch.equal(got[0, :, 10 * hs:], plain[0, :, 10 * hs:])
    assert torch.equal(got[1:], plain[1:])
