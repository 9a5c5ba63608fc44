"""Every tile shape of the bf16 GEMM at the edges of its tiles and of its ring of K tiles."""
import pytest
import torch

from gpu_util import M  # noqa: F401  (loads the package)
from sd3_c_amd import lib as L

pytestmark = pytest.mark.gpu
SHAPES = (64064, 128064, 64128, 128, 256128, 128256, 192256, 256, 0)


def _grouped(problems, epi, f32):
    arr = (L.GemmBf16Problem * len(problems))(*problems)
    L.call("sd3_gemm_bf16_grouped", arr, len(problems), epi, f32, None)


# K tiles of 64: fewer than the ring's stages, as many, one more, odd and even counts beyond (q|k|v, epilogue 5, has three times a multiple of 64 columns)
SIZES = [(1, 64, 64), (63, 192, 128), (65, 576, 192), (127, 320, 320), (129, 192, 384), (257, 384, 448), (300, 1536, 1536)]


@pytest.mark.parametrize("m,n,k,epi,f32", [s + e for e in ((0, 1), (1, 0), (3, 1), (4, 1), (5, 0)) for s in SIZES if e[0] != 5 or s[1] % 192 == 0])
def test_bf16_tile_shapes(m, n, k, epi, f32):
    """Two problems per launch (the second with 40 rows), forced to every shape: equal bits, and for the plain bias the float64 product
    within (k + 1) u (|A| |W| + |b|), u the roundoff of fp32 (the operands are exact bf16 values)."""
    g = torch.Generator(device="cuda").manual_seed(m * 7 + k)
    rows = (m, 40)
    A = [torch.randn((r, k), device="cuda", generator=g).bfloat16() for r in rows]
    W = [(0.1 * torch.randn((n, k), device="cuda", generator=g)).bfloat16() for _ in rows]
    bias, gate, rms = (torch.randn(s, device="cuda", generator=g) for s in ((n,), (max(rows), n), (64,)))  # (a gate row for every row of either problem)
    resid = [torch.randn((r, n), device="cuda", generator=g) for r in rows]
    per = max(1, m // 3)
    first = None
    try:
        for tile in SHAPES:
            L.call("sd3_gemm_bf16_force_tile", tile)
            out = [torch.zeros((r, n), device="cuda", dtype=torch.float32 if f32 else torch.bfloat16) for r in rows]
            _grouped([L.GemmBf16Problem(A[i].data_ptr(), W[i].data_ptr(), bias.data_ptr(), out[i].data_ptr(), r, n, k, gate.data_ptr(), n, resid[i].data_ptr(),
                                        resid[0].data_ptr(), min(per, 40), rms.data_ptr(), rms.data_ptr()) for i, r in enumerate(rows)], epi, f32)
            if epi == 0:
                for i in range(2):
                    a, w = A[i].double(), W[i].double().t().contiguous()
                    bound = (k + 1) * 2.0 ** -24 * (a.abs() @ w.abs() + bias.double().abs())
                    assert ((out[i].double() - (a @ w + bias.double())).abs() <= bound).all(), tile
            first = out if first is None else first
            assert all(torch.equal(x, y) for x, y in zip(out, first)), tile
    finally:
        L.call("sd3_gemm_bf16_force_tile", 0)


# columns: fewer than four, one, two and three beyond a group of four; `off`: elements between a 16-byte boundary and the output (and residual)
@pytest.mark.parametrize("m,n,k,off", [(1, 1, 64, 0), (65, 66, 128, 0), (130, 131, 320, 1), (200, 257, 192, 3), (64, 128, 64, 1), (257, 192, 128, 2)])
@pytest.mark.parametrize("epi,f32", [(0, 1), (0, 0), (1, 0), (2, 1), (3, 1), (4, 1), (4, 0)])
def test_bf16_rows_that_are_not_whole_groups_of_four(m, n, k, off, epi, f32):
    """Rows of any length at any element: equal bits on every tile shape, nothing written beside the output, and for the plain bias the
    float64 product within (k + 1) u (|A| |W| + |b|) (bf16 outputs: rounded once more, 2^-8 of the value)."""
    g = torch.Generator(device="cuda").manual_seed(m * 11 + n)
    A = torch.randn((m, k), device="cuda", generator=g).bfloat16()
    W = (0.1 * torch.randn((n, k), device="cuda", generator=g)).bfloat16()
    per = max(1, m // 3)
    batches = (m + per - 1) // per
    bias, gate, table = (torch.randn(s, device="cuda", generator=g) for s in ((n,), (batches, n), (per, n)))
    resid = torch.randn(m * n + 8, device="cuda", generator=g)
    dt = torch.float32 if f32 else torch.bfloat16
    first = None
    try:
        for tile in SHAPES:
            L.call("sd3_gemm_bf16_force_tile", tile)
            out = torch.full((m * n + 16,), 7.0, device="cuda", dtype=dt)
            _grouped([L.GemmBf16Problem(A.data_ptr(), W.data_ptr(), bias.data_ptr(), out.data_ptr() + off * out.element_size(), m, n, k, gate.data_ptr(), n,
                                        resid.data_ptr() + 4 * off, table.data_ptr(), per, None, None)], epi, f32)
            torch.cuda.synchronize()
            assert bool((out[:off] == 7).all()) and bool((out[off + m * n:] == 7).all()), tile
            if epi == 0:
                a, w = A.double(), W.double().t().contiguous()
                want = a @ w + bias.double()
                bound = (k + 1) * 2.0 ** -24 * (a.abs() @ w.abs() + bias.double().abs()) + (0 if f32 else 2.0 ** -8) * want.abs()
                assert ((out[off:off + m * n].view(m, n).double() - want).abs() <= bound).all(), tile
            first = out if first is None else first
            assert torch.equal(out, first), tile
    finally:
        L.call("sd3_gemm_bf16_force_tile", 0)
