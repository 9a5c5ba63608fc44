"""The fp32 GEMMs' epilogues: gates of rows that belong to one, two and more batch elements within a wavefront's rows, and the tanh-GELU's error."""
import math

import numpy as np
import pytest
import torch

from gpu_util import F32_TOL, M, dev, dev_params, host, max_abs
import oracle_lib as ol
from sd3_c_amd.params import block_param_shapes, synthetic_params_numpy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,NH", [(128, 2), (512, 8)])  # the fp32 instruction's kernel, the pieces kernel
@pytest.mark.parametrize("Tc,Tx", [(3, 7), (15, 17), (31, 33), (64, 65)])
def test_gates_of_rows_of_several_batch_elements(C, NH, Tc, Tx):
    """Wavefronts have 16 to 64 consecutive rows: several elements of 3 and 7 rows, two of 33 or 65. Each element against itself alone, the same bits;
    the first against the oracle."""
    B = 5
    rng = np.random.Generator(np.random.Philox(Tc))
    P = synthetic_params_numpy(block_param_shapes(C, 2, False, True, False, C // NH), 3, 0.05, 0.05)
    y, c, x = (rng.standard_normal(s, dtype=np.float32) for s in ((B, C), (B, Tc, C), (B, Tx, C)))
    dP = dev_params(P)

    def run(b0, b1):
        cg, xg = M.Dit_block(dev(y[b0:b1]), dev(c[b0:b1].copy()), dev(x[b0:b1].copy()), dP, b1 - b0, Tc, Tx, C, NH, 2, False, True, False, precision="fp32")
        return host(cg), host(xg)

    cg, xg = run(0, B)
    for b in range(B):
        c1, x1 = run(b, b + 1)
        assert np.array_equal(cg[b:b + 1], c1) and np.array_equal(xg[b:b + 1], x1)
    if C == 128:
        co, xo = ol.orc_dit_block(y[:1], c[:1], x[:1], P, NH, 2, False, True, False)
        assert max_abs(cg[:1], co) <= F32_TOL and max_abs(xg[:1], xo) <= F32_TOL


@pytest.mark.parametrize("scale", [0.01, 0.3, 1.0, 3.0, 6.0])
def test_gelu_tanh_error_against_64_bits(scale):
    """Relative 2-norm of the error: at most 2^-24 (a result rounded once has 2^-24/sqrt(3) on average, and the polynomial and the exponential add about as much where the
    gate is neither 0 nor 1); the formula with fp32's tanh has 2.8e-8 to 4.1e-8 at these scales."""
    x = scale * torch.randn(1 << 20, device="cuda:0", generator=torch.Generator(device="cuda:0").manual_seed(1))
    v = x.double()
    want = 0.5 * v * (1 + torch.tanh(math.sqrt(2 / math.pi) * (v + 0.044715 * v ** 3)))
    err = M.gelu_tanh(x).double() - want
    assert err.norm() <= 2.0 ** -24 * want.norm()


def test_gelu_tanh_of_what_is_not_ordinary():
    x = torch.tensor([0.0, -0.0, 3e38, -3e38, 2e19, -2e19, math.inf, -13.0, 1e-40, -1e-40], device="cuda:0")
    got = M.gelu_tanh(x).tolist()
    assert got[:8] == [0.0, 0.0, x[2].item(), 0.0, x[4].item(), 0.0, math.inf, 0.0]
    assert all(abs(g - w / 2) <= 2.0 ** -149 for g, w in zip(got[8:], x[8:].tolist()))
    assert all(math.isnan(g) for g in M.gelu_tanh(torch.tensor([-math.inf, math.nan], device="cuda:0")).tolist())
