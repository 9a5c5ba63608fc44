"""The modulation projections of one block (few-row linear layers) at widths around their column groups and slices of K."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import BF16_REL_L2, F32_TOL, M, dev, dev_params, host, max_abs, rel_l2
from sd3_c_amd.params import block_param_shapes, synthetic_params_numpy

pytestmark = pytest.mark.gpu


# fp32: 32 columns and 32 slices of K per workgroup. Widths below one slice's row, not a multiple of four (no wide loads), one chunk short
# of and just past a column group, several; one, five and nine rows (nine run as two groups)
@pytest.mark.parametrize("C,NH", [(6, 2), (24, 2), (30, 2), (36, 3), (100, 4), (132, 2)])
@pytest.mark.parametrize("B", [1, 5, 9])
def test_modulation_fp32_vs_oracle(B, C, NH):
    rng = np.random.Generator(np.random.Philox(C * 10 + B))
    P = synthetic_params_numpy(block_param_shapes(C, 2, True, True, False, C // NH), C + B, 0.1, 0.1)
    y, c, x = (rng.standard_normal(s, dtype=np.float32) for s in ((B, C), (B, 3, C), (B, 5, C)))
    co, xo = ol.orc_dit_block(y, c, x, P, NH, 2, True, True, False)
    cg, xg = M.Dit_block(dev(y), dev(c), dev(x), dev_params(P), B, 3, 5, C, NH, 2, True, True, False)
    assert max_abs(host(cg), co) <= F32_TOL and max_abs(host(xg), xo) <= F32_TOL


# bf16: 64 columns and 16 slices; a row's modulation (and so its block) is what it is alone
@pytest.mark.parametrize("C,NH", [(64, 1), (320, 5)])
def test_modulation_bf16(C, NH):
    B = 5
    rng = np.random.Generator(np.random.Philox(C))
    P = synthetic_params_numpy(block_param_shapes(C, 4, True, True, False, 64), C, 0.05, 0.05)
    dP = dev_params(P)
    y, c, x = (rng.standard_normal(s, dtype=np.float32) for s in ((B, C), (B, 3, C), (B, 70, C)))

    def run(prec, sel):
        cg, xg = M.Dit_block(dev(y[sel]), dev(c[sel]), dev(x[sel]), dP, len(y[sel]), 3, 70, C, NH, 4, True, True, False, precision=prec)
        return host(cg), host(xg)

    c16, x16 = run("bf16", slice(0, B))
    co, xo = ol.orc_dit_block(y, c, x, P, NH, 4, True, True, False)
    assert rel_l2(c16, co) <= BF16_REL_L2 and rel_l2(x16, xo) <= BF16_REL_L2
    c1, x1 = run("bf16", slice(3, 4))
    assert np.array_equal(c1[0], c16[3]) and np.array_equal(x1[0], x16[3])
