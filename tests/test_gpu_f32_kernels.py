"""The fp32 matrix kernels of the GEMM and attention operators at the edges of their tiles, against float64 arithmetic."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd import lib as L

pytestmark = pytest.mark.gpu
U = 2.0 ** -24  # unit roundoff of fp32


@pytest.fixture(autouse=True)
def _automatic_tile_afterwards():
    yield
    L.call("sd3_tune", b"gemm_f32_tile", -1)


@pytest.mark.parametrize("m,k,n", [(1, 4, 4), (33, 36, 68), (128, 32, 128), (129, 64, 132), (154, 1536, 1540), (257, 100, 64), (65, 2052, 36)])
def test_gemm_f32_every_tile_shape(m, k, n):
    """Rows, columns and depths on and beside the multiples of the tiles (32, 64, 128 and 32 k values). The bound is that of a sum of k
    products in any order, (k + 2) u (|x| |W| + |b|) element by element; the tile shapes agree bit for bit (same order of k)."""
    g = torch.Generator(device="cuda").manual_seed(m * 31 + k)
    x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, n), (n,)))
    want = x.double() @ W.double() + b.double()
    bound = (k + 2) * U * (x.double().abs() @ W.double().abs() + b.double().abs())
    first = None
    for tile in (-1, 0, 1, 2, 3, 4):
        L.call("sd3_tune", b"gemm_f32_tile", tile)
        y = M.linear(x, W, b)
        assert ((y.double() - want).abs() <= bound).all(), tile
        first = y if first is None else first
        assert torch.equal(y, first), tile


def test_gemm_f32_column_window_and_unaligned_rows():
    """Columns n0.. of a wider weight (whole 16-byte chunks), and strides that are not made of such chunks (the element-wise kernel)."""
    g = torch.Generator(device="cuda").manual_seed(5)
    for m, k, nmax, n0, n in ((40, 96, 200, 100, 68), (40, 95, 201, 3, 77)):
        x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, nmax), (nmax,)))
        y = M.partial_linear(x, W, b, n0, n)
        xd, Wd, bd = x.double(), W[:, n0:n0 + n].double(), b[n0:n0 + n].double()
        assert ((y.double() - (xd @ Wd + bd)).abs() <= (k + 2) * U * (xd.abs() @ Wd.abs() + bd.abs())).all()


@pytest.mark.parametrize("B,NH,hs,Tq,Tk", [(1, 1, 64, 1, 1), (2, 3, 64, 15, 17), (1, 2, 64, 33, 65), (1, 24, 64, 300, 129), (1, 2, 128, 17, 16),
                                           (2, 1, 128, 100, 1000), (1, 12, 128, 530, 47), (1, 2, 40, 20, 30)])
def test_attention_f32(B, NH, hs, Tq, Tk):
    """One query, one key, partly empty tiles, wavefronts without keys, both shapes of either head size and a head size of the general
    kernel. Bound: a score carries (hs + 3) u sum|q k| / sqrt(hs), a weighted mean of values twice the largest score error (to first order)
    plus the rounding of sums over Tk keys, the exponential's included."""
    g = torch.Generator(device="cuda").manual_seed(Tq * 7 + Tk)
    q, k, v = (torch.randn((B, t, NH * hs), device="cuda", generator=g) for t in (Tq, Tk, Tk))
    out = M.mha(q, k, v, NH)
    heads = [t.double().view(B, -1, NH, hs).transpose(1, 2).contiguous() for t in (q, k, v)]
    kt = heads[1].transpose(2, 3).contiguous()
    want = torch.softmax(heads[0] @ kt / hs ** 0.5, -1) @ heads[2]
    score_err = (hs + 3) * U * float((heads[0].abs() @ kt.abs()).max()) / hs ** 0.5
    bound = (2 * score_err + (Tk + 8) * U) * float(v.abs().max())
    assert float((out.double() - want.transpose(1, 2).reshape(B, Tq, -1)).abs().max()) <= bound
