"""Gated bf16 layers whose wavefronts have rows of one, two and more batch elements, in the ring kernel's tiles and in the persistent kernel's: a batch element
against itself alone, the same bits."""
import numpy as np
import pytest

from gpu_util import M, dev, dev_params, host
from sd3_c_amd import lib as L
from sd3_c_amd.params import block_param_shapes, synthetic_params_numpy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [0, 64064, 64128, 128064, 128, 128256, 256128, 192, 192256, 256])
@pytest.mark.parametrize("Tc,Tx", [(3, 7), (15, 33), (64, 65), (77, 200), (130, 256)])
def test_gates_of_rows_of_several_batch_elements(tile, Tc, Tx):
    """Wavefronts have 16, 32, 64 or 128 consecutive rows: up to 18 elements of 7 rows, boundaries inside of them and between them; whole tiles of 256 rows (the persistent kernel's
    form without conditions) and the last ones of a matrix. (Tiles of 256x192 have no norms in their epilogue, and 48 columns a wavefront.)"""
    B, C, NH, qk = 5, 256, 4, tile != 192
    rng = np.random.Generator(np.random.Philox(Tx))
    P = dev_params(synthetic_params_numpy(block_param_shapes(C, 4, True, qk, False, C // NH), 5, 0.05, 0.05))
    y, c, x = (rng.standard_normal(s, dtype=np.float32) for s in ((B, C), (B, Tc, C), (B, Tx, C)))

    def run(b0, b1):
        cg, xg = M.Dit_block(dev(y[b0:b1]), dev(c[b0:b1].copy()), dev(x[b0:b1].copy()), P, b1 - b0, Tc, Tx, C, NH, 4, True, qk, False, precision="bf16")
        return host(cg), host(xg)

    L.check(L.load().sd3_tune(b"gemm_bf16_tile", tile))
    try:
        cg, xg = run(0, B)
    finally:
        L.check(L.load().sd3_tune(b"gemm_bf16_tile", 0))
    for b in range(B):
        c1, x1 = run(b, b + 1)
        assert np.array_equal(cg[b:b + 1], c1) and np.array_equal(xg[b:b + 1], x1)
