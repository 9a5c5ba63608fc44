"""fp32 attention of bf16 pieces at the edges of its tiles and of its choices, at any scale and beyond the range of the pieces, against float64 arithmetic and the
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


def by_pieces(*args):
    """What the kernel of pieces gives, and not the fp32 instruction in its place (whose last bits differ)."""
    out = M.mha(*args)
    assert not torch.equal(out, on_fp32_instruction(*args))
    return out


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


@pytest.mark.parametrize("B,NH,hs,Tq,Tk", [(1, 1536, 64, 65, 1), (1, 1536, 64, 127, 31), (1, 1536, 64, 128, 32), (1, 384, 64, 129, 33), (2, 384, 64, 129, 63), (1, 128, 64, 257, 97),
                                           (3, 192, 64, 128, 225), (1, 96, 64, 65, 481), (1, 48, 64, 129, 511), (1, 24, 64, 385, 512), (1, 19, 64, 800, 351), (1, 256, 64, 100, 161),
                                           (2, 96, 64, 65, 512), (2, 24, 64, 512, 513), (1, 24, 64, 1178, 253)])
def test_edges(B, NH, hs, Tq, Tk):
    """One key tile (a run without keys) to seventeen, whole and not, query blocks of 64 (up to 128 blocks of 128 queries in all) and 128, the runs side by side (up to 256) and one after
    the other. All have 96 blocks and 1536 blocks x tiles in an element, which is what sends them to this kernel."""
    check_attention(B, NH, hs, Tq, Tk)


@pytest.mark.parametrize("Tk", [481, 512, 544, 700])
def test_an_element_alone_and_in_a_batch(Tk):
    """Blocks of 64 queries, of 128 and runs one after the other have the same bits."""
    NH, args = 24, inputs(Tk, 5, 24, 64, 400, Tk)
    whole = by_pieces(*args, NH)
    for n in (1, 2, 3):  # 96, 192 and 288 blocks of 128 queries
        assert torch.equal(M.mha(*(t[:n].contiguous() for t in args), NH), whole[:n])


@pytest.mark.parametrize("hs,NH", [(64, 24)])
@pytest.mark.parametrize("q_exponent,k_exponent,v_exponent", [(0, 0, 0), (-40, 40, -60), (30, -30, 60), (3, 0, 0)])
def test_scales(hs, NH, q_exponent, k_exponent, v_exponent):
    """The error against float64 is no larger than the fp32 instruction's at any scale, a head of zero values and rows of either sign of scale included (1.25 times it: the errors of
    two sums of the same products may differ)."""
    q, k, v = inputs(hs, 1, NH, hs, 400, 500)
    q, k, v = q * 2.0 ** q_exponent, k * 2.0 ** k_exponent, v * 2.0 ** v_exponent
    v[:, :, :hs] = 0
    k[:, :, hs:2 * hs] = 0
    q[:, 5] *= 1e-6
    want = exact(q, k, v, NH)
    got, before = by_pieces(q, k, v, NH), on_fp32_instruction(q, k, v, NH)
    assert (got[:, :, :hs] == 0).all()
    assert float((got.double() - want).norm()) <= 1.25 * float((before.double() - want).norm())


@pytest.mark.parametrize("B", [1, 4])
@pytest.mark.parametrize("hs", [64])
def test_infinities_nans_and_values_beyond_the_pieces(hs, B):
    """What the pieces cannot hold gives what the fp32 instruction gives (to rounding), and changes nothing in other heads: infinities and NaNs in q, k and v, values of 2^112
    and more in v. Values that grow by 2^20 along the keys, and a K and a V whose first tiles are zero, are like any others."""
    NH = 24
    q, k, v = inputs(hs + 1, B, NH, hs, 400, 500)
    plain = by_pieces(q, k, v, NH)
    at = lambda h: slice(h * hs, (h + 1) * hs)
    q[0, 7, 0] = float("inf")
    q[0, 9, hs] = float("nan")
    k[0, 100, 2 * hs] = float("inf")
    k[0, 40, 3 * hs + 1] = float("nan")
    v[0, 50, 4 * hs + 2] = float("-inf")
    v[0, 332, 5 * hs + 3] = float("nan")
    v[0, 200:, at(6)] *= 2.0 ** 20
    k[0, 290:, at(7)] *= 2.0 ** 10
    v[0, 100, 10 * hs] = 2.0 ** 120
    v[0, :280, at(8)] = 0
    k[0, :280, at(9)] = 0
    got, want = M.mha(q, k, v, NH), on_fp32_instruction(q, k, v, NH)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    for h in range(11):
        g, w = got[0, :, at(h)], want[0, :, at(h)]
        fine = torch.isfinite(w)
        if h == 7:  # scores of up to 2^10 * 30, whose own rounding shows: no further from float64 than the fp32 instruction (1.25 as below)
            truth = exact(q[:1, :, at(7)], k[:1, :, at(7)], v[:1, :, at(7)], 1)[0]
            assert float((g.double() - truth).norm()) <= 1.25 * float((w.double() - truth).norm())
        elif fine.any():
            assert float((g - w)[fine].abs().max() / w[fine].abs().max()) <= 1e-5
    assert torch.equal(got[0, :, 11 * hs:], plain[0, :, 11 * hs:])
    assert torch.equal(got[1:], plain[1:])


def spread(kind, e, hs, NH, Tq=400, Tk=500):
    """q, k and v whose values differ by 2^e within a channel, a token or a head, so that results consist of the small ones, and the channels to look at."""
    q, k, v = inputs(hs + e, 1, NH, hs, Tq, Tk)
    heads = [t.view(1, -1, NH, hs) for t in (q, k, v)]
    qh, kh, vh = heads
    looked_at = torch.ones(hs, dtype=torch.bool, device="cuda")
    c = 5
    if kind in ("a token of V that no query looks at", "a token of K that no query looks at", "a key that takes nearly all and has no value"):
        # channel 0 of K moves a key's scores of all queries, by 8 to 9 * sqrt(1 / hs) of it
        qh[..., 0] = 8 + torch.rand((1, Tq, NH), device="cuda", generator=torch.Generator(device="cuda").manual_seed(e))
        kh[..., 0] = 0
    if kind == "a channel of V":
        vh[..., c] *= 2.0 ** e
        looked_at[c] = False
    elif kind == "a token of V that no query looks at":
        kh[:, 1, :, 0] = -400
        vh[:, 1] *= 2.0 ** e
    elif kind == "a token of K that no query looks at":
        kh[:, 1, :, 0] = -1000 - 2.0 ** e
    elif kind == "a channel of K that q leaves out":
        kh[..., c] *= 2.0 ** e
        qh[..., c] = 0
    elif kind == "a channel of q that K leaves out":
        qh[..., c] *= 2.0 ** e
        kh[..., c] = 0
    elif kind == "a channel in another unit":
        kh[..., c] *= 2.0 ** e
        qh[..., c] *= 2.0 ** -e
    else:
        kh[:, 0] = 0
        kh[:, 0, :, 0] = e * hs ** 0.5 / 8 / 1.4426950408889634
        vh[:, 0] = 0
    return q, k, v, looked_at.repeat(NH)


@pytest.mark.parametrize("hs,NH", [(64, 24)])
@pytest.mark.parametrize("e", [7, 12, 16, 20, 40, 60])
@pytest.mark.parametrize("kind", ["a channel of V", "a token of V that no query looks at", "a token of K that no query looks at", "a channel of K that q leaves out",
                                  "a channel of q that K leaves out", "a channel in another unit", "a key that takes nearly all and has no value"])
def test_small_values_beside_large_ones(kind, e, hs, NH):
    """Values far below the largest of their head, channel or token count in full: no more error than the fp32 instruction's (1.25 times it, as the errors of two sums of
    the same products may differ by chance)."""
    q, k, v, looked_at = spread(kind, e, hs, NH)
    want = exact(q, k, v, NH)[..., looked_at]
    err = [float((out[..., looked_at].double() - want).norm()) for out in (on_fp32_instruction(q, k, v, NH), by_pieces(q, k, v, NH))]
    print(f"fp32 instruction {err[0] / float(want.norm()):.2e}, pieces {err[1] / float(want.norm()):.2e}")
    assert err[1] <= 1.25 * err[0]


@pytest.mark.parametrize("hs,NH", [(64, 96)])
@pytest.mark.parametrize("B", [1, 2])
def test_one_key_gives_its_value(hs, NH, B):
    """The one weight is 1, so the result is the key's value to the last bit, from 2^-100 to 2^90 and 0 included."""
    q, k, v = inputs(hs + B, B, NH, hs, 2000, 1)
    v *= torch.exp2(torch.randint(-100, 91, v.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).float())
    v[..., 7] = 0
    assert torch.equal(M.mha(q, k, v, NH), v.expand(B, 2000, NH * hs))


@pytest.mark.parametrize("hs,NH", [(64, 24)])
@pytest.mark.parametrize("kind", ["normal", "equal weights", "positive values", "constant values", "few large scores"])
@pytest.mark.parametrize("Tq,Tk", [(8192, 32), (2816, 77), (1664, 154), (400, 1178), (400, 4250)])
def test_error_is_no_larger_than_the_fp32_instructions(Tq, Tk, kind, hs, NH):
    """Sums whose terms cancel, whose terms all have one sign (where rounding to one side would add up), constants, and few terms. 1.25 as above; 2^-24: results that
    one of the two happens to hold exactly."""
    q, k, v = inputs(hs + Tk, 1, NH, hs, Tq, Tk)
    q *= {"equal weights": 1e-3, "few large scores": 6.0}.get(kind, 1.0)
    v = {"positive values": v.abs(), "constant values": torch.full_like(v, 1 + 2.0 ** -12 + 2.0 ** -23)}.get(kind, v)
    want = exact(q, k, v, NH)
    err = [float((out.double() - want).norm() / want.norm()) for out in (on_fp32_instruction(q, k, v, NH), by_pieces(q, k, v, NH))]
    print(f"fp32 instruction {err[0]:.2e}, pieces {err[1]:.2e}")
    assert err[1] <= 1.25 * err[0] + 2.0 ** -24
