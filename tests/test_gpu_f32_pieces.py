"""fp32 products of f16 pieces at the edges of their tiles, beyond the range of the pieces and in blocks, against float64 arithmetic and the fp32 instruction."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd import lib as L
from sd3_c_amd.params import block_param_shapes

pytestmark = pytest.mark.gpu
U = 2.0 ** -24  # unit roundoff of fp32


@pytest.fixture(autouse=True)
def _automatic_choice_afterwards():
    yield
    L.call("sd3_tune", b"gemm_f32_tile", -1)
    L.call("sd3_tune", b"gemm_f32_no_pieces", 0)


@pytest.mark.parametrize("m,k,n", [(1, 512, 4), (31, 256, 36), (33, 384, 68), (65, 768, 64), (129, 512, 132), (257, 640, 260), (300, 1536, 1540)])
def test_every_tile_shape(m, k, n):
    """Rows and columns on and beside the multiples of the tiles (32 to 256), depths from the smallest on. Bound: a product of pieces lacks less than 3 u of itself
    (u of either value, u for l*l), and of its additions three per 32 values round: less than a sum of k products in any order, (k + 2) u (|x| |W| + |b|). The
    shapes agree bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(m * 31 + k)
    x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, n), (n,)))
    want = x.double() @ W.double() + b.double()
    bound = (k + 2) * U * (x.double().abs() @ W.double().abs() + b.double().abs())
    first = None
    for shape in (-1, 0, 1, 2, 3, 4, 5):
        L.call("sd3_tune", b"gemm_f32_tile", shape)
        y = M.linear(x, W, b)
        assert ((y.double() - want).abs() <= bound).all(), shape
        first = y if first is None else first
        assert torch.equal(y, first), shape


@pytest.mark.parametrize("scale_x,scale_w", [(1e-18, 1e-12), (1e15, 1e18), (1e-30, 1e28)])
def test_small_and_large_values(scale_x, scale_w):
    """Powers of two bring the values into the range of the pieces: the error is that of the tile kernel at any scale (twice it, as two sums of one product may differ)."""
    g = torch.Generator(device="cuda").manual_seed(7)
    x, W, b = scale_x * torch.randn((200, 512), device="cuda", generator=g), scale_w * torch.randn((512, 192), device="cuda", generator=g), torch.zeros(192, device="cuda")
    want = x.double() @ W.double()
    err = []
    for choice in (1, 0):
        L.call("sd3_tune", b"gemm_f32_no_pieces", choice)
        err.append(float((M.linear(x, W, b).double() - want).norm() / want.norm()))
    assert err[1] <= 2 * err[0]


@pytest.mark.parametrize("shape", [0, 1, 2, 3, 4, 5])
def test_infinities_nans_and_values_beyond_bf16(shape):
    """What has no pieces (infinities, NaNs, values much larger than the first of their row, in x and in W) gives what the fp32 instruction gives, and changes nothing else."""
    g = torch.Generator(device="cuda").manual_seed(shape)
    m, k, n = 150, 512, 140
    x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, n), (n,)))
    L.call("sd3_tune", b"gemm_f32_tile", shape)
    plain = M.linear(x, W, b)
    x[3, 5], x[40, 17], x[77, 200] = float("inf"), float("-inf"), float("nan")
    x[90, 9] = 3.4e38
    W[11, 33], W[100, 139] = float("inf"), float("nan")
    W[9, 7] = 1.0
    got = M.linear(x, W, b)
    L.call("sd3_tune", b"gemm_f32_no_pieces", 1)
    want = M.linear(x, W, b)
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
    rows = torch.ones(m, dtype=torch.bool)
    rows[[3, 40, 77, 90]] = False
    cols = torch.ones(n, dtype=torch.bool)
    cols[[33, 139]] = False
    cols[7] = False
    assert torch.equal(got[rows][:, cols], plain[rows][:, cols])
    assert float(((got[90] - want[90])[finite[90]]).abs().max()) <= (k + 2) * U * 3.4e38 * 4


@pytest.mark.parametrize("shape", [0, 1, 2, 3, 4, 5])
def test_rows_and_columns_of_any_scale(shape):
    """Rows of x and columns of W from 2^-40 to 2^40, a row whose first 64 and one whose first 200 values are zero, one of zeros, one that grows by 2^20 and a column that does (formed anew
    by the fp32 instruction), one that starts 2^9 above the rest and one that grows by 2^10. Bound as above: relative to |x| |W| of the element itself."""
    g = torch.Generator(device="cuda").manual_seed(shape + 50)
    m, k, n = 150, 512, 140
    x, W, b = torch.randn((m, k), device="cuda", generator=g), torch.randn((k, n), device="cuda", generator=g), torch.zeros(n, device="cuda")
    x *= torch.ldexp(torch.ones(m), torch.randint(-40, 41, (m,), generator=torch.Generator().manual_seed(1))).cuda()[:, None]
    W *= torch.ldexp(torch.ones(n), torch.randint(-40, 41, (n,), generator=torch.Generator().manual_seed(2))).cuda()
    x[3, :64], x[4, :200], x[5] = 0, 0, 0
    x[9, 64:] *= 2.0 ** 20
    x[70, :64] *= 2.0 ** 9
    x[71, 64:] *= 2.0 ** 10
    W[100:, 17] *= 2.0 ** 20
    W[:64, 130] = 0
    L.call("sd3_tune", b"gemm_f32_tile", shape)
    y = M.linear(x, W, b)
    bound = (k + 2) * U * (x.double().abs() @ W.double().abs())
    assert ((y.double() - x.double() @ W.double()).abs() <= bound).all()


@pytest.mark.parametrize("Tc,Tx,dual", [(77, 1000, True), (5, 2049, False)])
def test_blocks_in_batches(Tc, Tx, dual):
    """Blocks whose layers all go by pieces: an element alone has the bits that it has in a batch, every shape has them too,
    and the fp32 instruction's results are as far away as two sums of 512 to 2048 products in other orders (1e-6) in six layers behind one another."""
    C, NH = 512, 8
    g = torch.Generator(device="cuda").manual_seed(Tx)
    P = {k: 0.05 * torch.randn(s, device="cuda", generator=g) for k, s in block_param_shapes(C, 4, dual, True, False, 64).items()}
    y, c, x = (torch.randn(s, device="cuda", generator=g) for s in ((2, C), (2, Tc, C), (2, Tx, C)))

    def run(n, at=0):
        out = M.Dit_block(y[at:at + n].contiguous(), c[at:at + n].clone(), x[at:at + n].clone(), P, n, Tc, Tx, C, NH, 4, dual, True, False)
        torch.cuda.synchronize()
        return out

    both = run(2)
    for e in (0, 1):
        for a, b in zip(run(1, e), both):
            assert torch.equal(a[0], b[e])
    for shape in (0, 2, 4, 5):
        L.call("sd3_tune", b"gemm_f32_tile", shape)
        forced = run(1)
        again = run(2)
        for a, b in zip(forced, again):
            assert torch.equal(a[0], b[0])
    L.call("sd3_tune", b"gemm_f32_no_pieces", 1)
    for a, b in zip(run(2), both):
        assert not torch.equal(a, b) and float((a - b).norm()) <= 1e-5 * float(a.norm())
