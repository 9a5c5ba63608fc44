"""Operand rows of more than 2^22 values, whose offsets inside a tile do not fit 32 bits for every tile shape: bf16 and fp8 products, exact on small integers."""
import pytest
import torch

from gpu_util import M  # noqa: F401  (loads the package)
from sd3_c_amd import lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1 << 22, (1 << 22) + 128])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_products_of_long_rows(kind, k):
    """On both sides of the limit. Values of -1, 0 and 1 (nine in ten of them 0): every partial sum is an integer below 2^24, so the result is exact."""
    m, n = 3, 68
    g = torch.Generator(device="cuda").manual_seed(k)

    def digits(rows):
        return torch.randint(-10, 11, (rows, k), device="cuda", generator=g, dtype=torch.int8).div(10, rounding_mode="trunc")

    a, w = digits(m), digits(n)
    want = torch.stack([(w.short() * a[i].short()).sum(1, dtype=torch.int64) for i in range(m)]).float()
    bias = torch.zeros(n, device="cuda")
    out = torch.full((m, n), 7.0, device="cuda")
    if kind == "bf16":
        A, W = a.bfloat16(), w.bfloat16()
        probs = (L.GemmBf16Problem * 1)(L.GemmBf16Problem(A.data_ptr(), W.data_ptr(), bias.data_ptr(), out.data_ptr(), m, n, k, None, 0, None, None, 1, None, None))
        for tile in (0, 64064, 256):
            L.call("sd3_gemm_bf16_force_tile", tile)
            out.fill_(7.0)
            L.call("sd3_gemm_bf16_grouped", probs, 1, 0, 1, None)
            L.call("sd3_gemm_bf16_force_tile", 0)
            assert torch.equal(out, want), tile
    else:
        one = {-1: 0xB8, 0: 0, 1: 0x38}  # e4m3
        A, W = (((t == 1) * one[1] + (t == -1) * one[-1]).to(torch.uint8) for t in (a, w))
        ones = torch.ones(n, device="cuda")
        L.call("sd3_gemm_fp8", A.data_ptr(), ones.data_ptr(), W.data_ptr(), ones.data_ptr(), bias.data_ptr(), out.data_ptr(), m, n, k, 0, 1, None)
        assert torch.equal(out, want)


@pytest.mark.parametrize("beyond", [0, 64])
@pytest.mark.parametrize("tile", [64064, 128, 128064, 64128, 256, 128256, 256128, 192256])
def test_bf16_tiles_at_the_reach_of_their_offsets(tile, beyond):
    """The deepest rows that a tile addresses by 32-bit offsets, and one K tile more. The last rows of both operands are reached; each has a one in front
    and its number at its end, so that a row taken for another shows: exact."""
    m, n = (tile, tile) if tile < 1000 else divmod(tile, 1000)
    k = ((1 << 32) - 128) // (max(m, n) - 1) // 128 * 64 + beyond
    A, W = (torch.zeros((rows, k), device="cuda", dtype=torch.bfloat16) for rows in (m, n))
    for t in (A, W):
        t[:, -1] = torch.arange(1, t.shape[0] + 1, device="cuda")
        t[:, 0] = 1.0
    want = A[:, -1:].float() * W[:, -1].float() + 1.0
    bias, out = torch.zeros(n, device="cuda"), torch.full((m, n), 7.0, device="cuda")
    probs = (L.GemmBf16Problem * 1)(L.GemmBf16Problem(A.data_ptr(), W.data_ptr(), bias.data_ptr(), out.data_ptr(), m, n, k, None, 0, None, None, 1, None, None))
    for forced in (0, tile):
        L.call("sd3_gemm_bf16_force_tile", forced)
        out.fill_(7.0)
        L.call("sd3_gemm_bf16_grouped", probs, 1, 0, 1, None)
        L.call("sd3_gemm_bf16_force_tile", 0)
        assert torch.equal(out, want), forced


@pytest.mark.parametrize("rows,beyond", [(128, 0), (128, 128), (1024, 0)])
def test_fp8_tiles_at_the_reach_of_their_offsets(rows, beyond):
    """The same with fp8 operands (numbers of 1 to 16): the deepest rows that 128x128 tiles address, one K tile more, and enough rows for 256x256 tiles."""
    m, n = rows, 256 if rows > 128 else 128
    k = ((1 << 32) - 128) // ((255 if rows > 128 else 127) * 128) * 128 + beyond
    A, W = (torch.zeros((r, k), device="cuda", dtype=torch.uint8) for r in (m, n))
    for t in (A, W):
        t[:, -1] = (torch.arange(t.shape[0], device="cuda") % 16 + 1).float().to(torch.float8_e4m3fn).view(torch.uint8)
        t[:, 0] = 0x38
    want = torch.outer(*((torch.arange(t, device="cuda") % 16 + 1).float() for t in (m, n))) + 1.0
    ones, bias, out = torch.ones(max(m, n), device="cuda"), torch.zeros(n, device="cuda"), torch.full((m, n), 7.0, device="cuda")
    for tile in (0, 256, 128):
        L.call("sd3_gemm_bf16_force_tile", tile)
        out.fill_(7.0)
        L.call("sd3_gemm_fp8", A.data_ptr(), ones.data_ptr(), W.data_ptr(), ones.data_ptr(), bias.data_ptr(), out.data_ptr(), m, n, k, 0, 1, None)
        L.call("sd3_gemm_bf16_force_tile", 0)
        assert torch.equal(out, want), tile
