"""The bf16 copies of a block's weights are kept as K tiles (K/64, N, 64): blocks whose layers have one, a few and odd numbers of such tiles and
numbers of columns on both sides of the tiles' edges, against the fp32 path, which reads the bound weights in place."""
import pytest
import torch

from gpu_util import M
from sd3_c_amd.params import block_param_shapes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Tc,Tx,C,E", [(1, 3, 5, 64, 1), (2, 9, 70, 192, 3), (1, 40, 130, 320, 2), (1, 77, 257, 448, 4)])
def test_bf16_block_with_any_number_of_weight_tiles(B, Tc, Tx, C, E):
    """The update of the residual streams alone (not the residual beside it): eight roundings of operands to bf16 lie in a row, 2^-8 each at most, which
    as independent errors is sqrt(8) 2^-8 = 1.1e-2, here doubled; a weight tile or column out of place would be of order 1."""
    g = torch.Generator(device="cuda").manual_seed(C + E)
    P = {k: 0.1 * torch.randn(s, device="cuda", generator=g) for k, s in block_param_shapes(C, E, True, True, False, 64).items()}
    y, c, x = (torch.randn(s, device="cuda", generator=g) for s in ((B, C), (B, Tc, C), (B, Tx, C)))
    new = {p: M.Dit_block(y, c.clone(), x.clone(), P, B, Tc, Tx, C, C // 64, E, True, True, False, precision=p) for p in ("fp32", "bf16")}
    for a, b, old in zip(new["bf16"], new["fp32"], (c, x)):
        assert float((b - old).norm()) > 0.1 * float(old.norm())  # (the update is not lost in the residual)
        assert float((a - b).norm()) <= 2e-2 * float((b - old).norm())
