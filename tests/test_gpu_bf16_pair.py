"""The two out-projections of a block with dual attention: one launch on the small tiles, one after the other on the others."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd import lib as L
from sd3_c_amd.params import block_param_shapes

pytestmark = pytest.mark.gpu


# rows below, at and past the edges of the tiles; K tiles of 64: 1 (fewer than the ring's stages), 5, 6 and 8
@pytest.mark.parametrize("B,Tc,Tx,C", [(1, 1, 1, 64), (1, 3, 63, 320), (2, 0, 65, 384), (3, 40, 129, 384), (1, 77, 257, 512)])
@pytest.mark.parametrize("discard", [False, True])
def test_block_does_not_depend_on_the_tile_of_its_projections(B, Tc, Tx, C, discard):
    """Equal bits for every forced tile (256 takes two launches) and for the chosen one, in place, twice in a row."""
    g = torch.Generator(device="cuda").manual_seed(B * 100 + Tx)
    P = {k: 0.1 * torch.randn(s, device="cuda", generator=g) for k, s in block_param_shapes(C, 2, True, True, discard, 64).items()}
    y, c, x = (torch.randn(s, device="cuda", generator=g) for s in ((B, C), (B, Tc, C), (B, Tx, C)))
    first = None
    try:
        for tile in (256, 64064, 128064, 64128, 128, 256128, 128256, 192256, 0, 0):
            L.call("sd3_gemm_bf16_force_tile", tile)
            got = M.Dit_block(y, c.clone(), x.clone(), P, B, Tc, Tx, C, C // 64, 2, True, True, discard, precision="bf16")
            torch.cuda.synchronize()
            assert torch.isfinite(got[1]).all()
            first = got if first is None else first
            assert torch.equal(got[0], first[0]) and torch.equal(got[1], first[1]), tile
    finally:
        L.call("sd3_gemm_bf16_force_tile", 0)


@pytest.mark.parametrize("B,Tc,Tx,C", [(1, 3, 63, 320), (2, 0, 65, 384), (1, 77, 257, 512)])
@pytest.mark.parametrize("discard", [False, True])
def test_block_without_qk_norm_on_every_tile(B, Tc, Tx, C, discard):
    """The same without the qk-norm, which 256x192 tiles (192) cannot fuse: every tile that a caller can force takes the whole block."""
    g = torch.Generator(device="cuda").manual_seed(B * 100 + Tx + 1)
    P = {k: 0.1 * torch.randn(s, device="cuda", generator=g) for k, s in block_param_shapes(C, 2, True, False, discard, 64).items()}
    y, c, x = (torch.randn(s, device="cuda", generator=g) for s in ((B, C), (B, Tc, C), (B, Tx, C)))
    first = None
    try:
        for tile in (256, 192, 64064, 128064, 64128, 128, 256128, 128256, 192256, 0):
            L.call("sd3_gemm_bf16_force_tile", tile)
            got = M.Dit_block(y, c.clone(), x.clone(), P, B, Tc, Tx, C, C // 64, 2, True, False, discard, precision="bf16")
            torch.cuda.synchronize()
            first = got if first is None else first
            assert torch.equal(got[0], first[0]) and torch.equal(got[1], first[1]), tile
    finally:
        L.call("sd3_gemm_bf16_force_tile", 0)


@pytest.mark.parametrize("B,Tc,Tx,C", [(1, 3, 63, 320), (2, 5, 129, 128)])
def test_streams_that_are_not_16_byte_aligned(B, Tc, Tx, C):
    """Streams that begin one float after a 16-byte boundary: outputs and residuals go element by element, on every tile with equal bits, and
    differ from the aligned ones by no more than bf16 rounding (their LayerNorm sums in another order)."""
    g = torch.Generator(device="cuda").manual_seed(Tx)
    P = {k: 0.1 * torch.randn(s, device="cuda", generator=g) for k, s in block_param_shapes(C, 2, True, True, False, 64).items()}
    y, c, x = (torch.randn(s, device="cuda", generator=g) for s in ((B, C), (B, Tc, C), (B, Tx, C)))

    def at(t, off):
        buf = torch.empty(t.numel() + 4, device="cuda")
        return buf[off:off + t.numel()].view(t.shape).copy_(t)

    def block(off):
        got = M.Dit_block(y, at(c, off), at(x, off), P, B, Tc, Tx, C, C // 64, 2, True, True, False, precision="bf16")
        torch.cuda.synchronize()
        return got

    aligned, first = block(0), None
    try:
        for tile in (256, 64064, 128064, 64128, 128, 256128, 128256, 192256, 0):
            L.call("sd3_gemm_bf16_force_tile", tile)
            got = block(1)
            first = got if first is None else first
            assert torch.equal(got[0], first[0]) and torch.equal(got[1], first[1]), tile
    finally:
        L.call("sd3_gemm_bf16_force_tile", 0)
    for a, b in zip(first, aligned):
        assert float((a - b).norm()) <= 2.0 ** -8 * float(b.norm())
