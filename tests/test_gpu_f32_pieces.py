"""fp32 products of bf16 pieces at the edges of their tiles, beyond the range of the pieces and in blocks, against float64 arithmetic and the fp32 instruction."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd import lib as L
from sd3_c_amd.params import block_param_shapes
from test_gpu_f32_kernels import test_gemm_f32_every_tile_shape as check_tile_kernel

pytestmark = pytest.mark.gpu
U = 2.0 ** -24  # unit roundoff of fp32


@pytest.fixture(autouse=True)
def _automatic_choice_afterwards():
    yield
    L.call("sd3_tune", b"gemm_f32_tile", -1)
    L.call("sd3_tune", b"gemm_f32_no_pieces", 0)


@pytest.mark.parametrize("m,k,n", [(1, 512, 4), (31, 640, 36), (33, 1152, 68), (65, 768, 64), (129, 512, 132), (257, 640, 260), (300, 1536, 1540)])
def test_every_tile_shape(m, k, n):
    """Rows and columns on and beside the multiples of the tiles (32 to 256), depths from the smallest on. Bound: a product of pieces lacks at most
    u of itself (m*l, l*m: 2^-25 each), and the additions of 32 products and of their sum to the sum of those before round less often than a sum of k products in any
    order does, (k + 2) u (|x| |W| + |b|). The shapes agree bit for bit."""
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


@pytest.mark.parametrize("scale_x,scale_w", [(1e-18, 1e-12), (1e15, 1e18), (1e-30, 1e28), (1e-36, 1e34), (1e-41, 1e37), (1e37, 1e-41), (1e-20, 1e-20)])
def test_small_and_large_values(scale_x, scale_w):
    """The error is that of the tile kernel at any scale, values below 2^-110 (whose pieces would be below the bf16 range) and subnormal ones, sums of 2^96 and more (formed anew) and
    subnormal results included (twice it, as two sums of one product may differ)."""
    g = torch.Generator(device="cuda").manual_seed(7)
    x, W, b = scale_x * torch.randn((200, 512), device="cuda", generator=g), scale_w * torch.randn((512, 192), device="cuda", generator=g), torch.zeros(192, device="cuda")
    want = x.double() @ W.double()
    err = []
    for choice in (1, 0):
        L.call("sd3_tune", b"gemm_f32_no_pieces", choice)
        err.append(float((M.linear(x, W, b).double() - want).norm() / want.norm()))
    assert err[1] <= 2 * err[0]


@pytest.mark.parametrize("shape", [0, 1, 2, 3, 4, 5])
def test_infinities_nans_and_values_beyond_the_pieces(shape):
    """What has no pieces (infinities, NaNs, values of 2^112 and more, in x and in W) gives what the fp32 instruction gives, and changes nothing else."""
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
    """Rows of x and columns of W from 2^-40 to 2^40, a row whose first 64 and one whose first 200 values are zero, one of zeros, one that grows by 2^20 and a column that does,
    one that starts 2^9 above the rest and one that grows by 2^10. Bound as above: relative to |x| |W| of the element itself."""
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


def spread(kind, e, m, k, n):
    """Operands whose values differ by powers of two of up to e within a row of x, a column of W or both, so that a result can consist of the small ones."""
    g = torch.Generator(device="cuda").manual_seed(k + e)
    x, W = torch.randn((m, k), device="cuda", generator=g), torch.randn((k, n), device="cuda", generator=g)
    channel = 0 if kind.endswith("first") else k // 2 + 3
    if kind.startswith("a large channel of x that W leaves out"):
        x[:, channel] *= 2.0 ** e
        W[channel] = 0
    elif kind.startswith("a large channel of W that x leaves out"):
        W[channel] *= 2.0 ** e
        x[:, channel] = 0
    elif kind.startswith("a channel in another unit"):
        x[:, channel] *= 2.0 ** e
        W[channel] *= 2.0 ** -e
    else:  # every channel in a unit of its own
        d = torch.exp2((torch.rand(k, device="cuda", generator=g) * 2 - 1) * e).clamp_(2.0 ** -60, 2.0 ** 60)
        x *= d
        W /= d[:, None]
    return x, W


@pytest.mark.parametrize("e", [-40, 7, 12, 16, 20, 27, 60])
@pytest.mark.parametrize("kind", ["a large channel of x that W leaves out, the first", "a large channel of x that W leaves out", "a large channel of W that x leaves out, the first",
                                  "a large channel of W that x leaves out", "a channel in another unit, the first", "a channel in another unit", "every channel in a unit of its own"])
@pytest.mark.parametrize("k", [512, 1536])
def test_channels_of_any_magnitude(kind, e, k):
    """Values far below the largest of their row or column count in full: element by element the bound of a sum of k products (as above), and in all no more error than
    the fp32 instruction's (1.25 times it, as the errors of two sums of the same products may differ by chance)."""
    x, W = spread(kind, e, 150, k, 140)
    b = torch.zeros(140, device="cuda")
    want, bound = x.double() @ W.double(), (k + 2) * U * (x.double().abs() @ W.double().abs())
    err = []
    for choice in (1, 0):
        L.call("sd3_tune", b"gemm_f32_no_pieces", choice)
        diff = (M.linear(x, W, b).double() - want).abs()
        err.append(float(diff.norm()))
    assert (diff <= bound).all()
    assert err[1] <= 1.25 * err[0]


@pytest.mark.parametrize("shape", [-1, 0, 1, 2, 3, 4, 5])
def test_single_products(shape):
    """Rows of x with one value that is not zero: every result is one product, which lacks at most 2^-24 of itself for the products of pieces that are not formed and is added
    to what is small beside it within a unit in the last place (2 u) whichever way that rounds: 3 u and 2^-8 of it for the sums of the smaller ones. Powers of two of
    2^-60 to 2^60, and values of 1 + 2^-11 and 1 + 2^-12 + 2^-23, whose low bits all count."""
    m, k, n = 512, 512, 140
    g = torch.Generator(device="cuda").manual_seed(shape + 3)
    value = torch.randn(m, device="cuda", generator=g) * torch.exp2(torch.randint(-60, 61, (m,), device="cuda", generator=g).float())
    value[:3] = 1 + 2.0 ** -11
    value[3:6] = 1 + 2.0 ** -12 + 2.0 ** -23
    W = torch.randn((k, n), device="cuda", generator=g) * torch.exp2(torch.randint(-20, 21, (k, 1), device="cuda", generator=g).float())
    W[:, :3] = 1 + 2.0 ** -11
    W[:, 3:6] = 1 + 2.0 ** -12 + 2.0 ** -23
    x = torch.zeros((m, k), device="cuda")
    x[torch.arange(m), torch.randperm(k, generator=torch.Generator().manual_seed(1)).cuda()] = value
    L.call("sd3_tune", b"gemm_f32_tile", shape)
    want = x.double() @ W.double()
    assert ((M.linear(x, W, torch.zeros(n, device="cuda")).double() - want).abs() <= 3.02 * U * want.abs()).all()


@pytest.mark.parametrize("x_of,w_of", [("normal", "normal"), ("positive", "positive"), ("1 + 2^-11", "1 + 2^-11"), ("positive", "1 + 2^-12 + 2^-23"), ("gelu", "normal"), ("one in 16", "normal")])
@pytest.mark.parametrize("k", [512, 1536, 6144])
def test_error_is_no_larger_than_the_fp32_instructions(x_of, w_of, k):
    """Sums whose terms cancel, whose terms all have one sign (where rounding to one side would add up), constants, and few terms. 1.25: two sums of the same
    products may differ by chance; u: results that one of the two happens to hold exactly."""
    g = torch.Generator(device="cuda").manual_seed(k)

    def make(kind, *shape):
        t = torch.randn(shape, device="cuda", generator=g)
        return {"normal": t, "positive": t.abs(), "1 + 2^-11": torch.full_like(t, 1 + 2.0 ** -11), "1 + 2^-12 + 2^-23": torch.full_like(t, 1 + 2.0 ** -12 + 2.0 ** -23),
                "gelu": torch.nn.functional.gelu(t, approximate="tanh"), "one in 16": t * (torch.rand(shape, device="cuda", generator=g) < 1 / 16)}[kind]

    x, W, b = make(x_of, 300, k), make(w_of, k, 260), torch.zeros(260, device="cuda")
    want = x.double() @ W.double()
    err = []
    for choice in (1, 0):
        L.call("sd3_tune", b"gemm_f32_no_pieces", choice)
        err.append(float((M.linear(x, W, b).double() - want).norm() / want.norm()))
    print(f"fp32 instruction {err[0]:.2e}, pieces {err[1]:.2e}")
    assert err[1] <= 1.25 * err[0] + U


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


@pytest.mark.parametrize("shape", [-1, 0, 1, 2, 3, 4, 5])
@pytest.mark.parametrize("k", [512, 640])
def test_column_windows_and_outputs_at_any_float(k, shape):
    """Columns n0.. of a wider weight have the bits of that part of the weight by itself, outputs may begin at any float and nothing beside them is written, also in rows and
    columns that are formed anew (values of 2^113 and more, an infinity). Bound as above."""
    m, nmax, n0, n = 70, 240, 100, 132
    g = torch.Generator(device="cuda").manual_seed(k)
    x, W, b = (torch.randn(s, device="cuda", generator=g) for s in ((m, k), (k, nmax), (nmax,)))
    x[33] *= 2.0 ** 113
    W[7, n0 + 66] = float("inf")
    L.call("sd3_tune", b"gemm_f32_tile", shape)
    part, bias = W[:, n0:n0 + n].contiguous(), b[n0:n0 + n].contiguous()
    want = M.linear(x, part, bias)
    assert torch.equal(M.partial_linear(x, W, b, n0, n), want)
    fine = torch.arange(n, device="cuda") != 66
    exact = x.double() @ part[:, fine].double() + bias[fine].double()
    assert ((want[:, fine].double() - exact).abs() <= (k + 2) * U * (x.double().abs() @ part[:, fine].double().abs() + bias[fine].double().abs())).all()
    assert torch.isinf(want[:, 66]).all()
    for off in (1, 2, 3):
        buf = torch.full((m * n + 8,), 7.0, device="cuda")
        L.call("sd3_linear", x.data_ptr(), part.data_ptr(), bias.data_ptr(), buf.data_ptr() + 4 * off, m, k, n, None)
        torch.cuda.synchronize()
        assert torch.equal(buf[off:off + m * n].view(m, n), want) and bool((buf[:off] == 7).all()) and bool((buf[off + m * n:] == 7).all()), off


@pytest.mark.parametrize("m,k,n", [(154, 1536, 1540), (154, 1568, 1540), (257, 480, 64)])
def test_deep_products_of_the_tile_kernel(m, k, n):
    """The fp32 instruction at depths of many whole K tiles: asked for, and where they are not whole groups of four."""
    L.call("sd3_tune", b"gemm_f32_no_pieces", 1)
    check_tile_kernel(m, k, n)
