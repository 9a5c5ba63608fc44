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
