"""The FP32 local search's product with its operand formed on the way (k_gemm_local in csrc/t2x_gemm.hip)
at the edges of its tiles: rows that end inside the first 64 and the second 64 of a tile or span particles
of one tile, 1, 37 and 149 translations (one column, one and two column tiles). diff2 against the FP64
oracle within the bound of the local-search parity tests.
"""
import numpy as np
import pytest

import estep_harness as H
from test_gpu_local import LOCAL360_BARS, localise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offsets", [0.5, 3.3, 6.8])
@pytest.mark.parametrize("n,sigma", [(1, 3.0), (3, 5.0), (7, 14.0)])
def test_rows(gpu_device, n, sigma, offsets):
    wl = localise(H.Workload("refine64", n=n, seed_offset=57, K=2,
                             overrides=dict(offset_range_px=offsets, offset_step_px=1.0)), sigma)
    o = wl.run_oracle(n_debug=n, fine_cap=1024)["dbg"]["coarse_diff2"]
    g = wl.run_gpu(dev=gpu_device, n_debug=n, fine_cap=1024)["dbg"]["coarse_diff2"]
    valid = o > -998
    assert valid.any() and np.array_equal(valid, g > -998)
    e = H.rel(g[valid], o[valid])
    print(f"{valid.sum()} samples, coarse diff2 max rel {e:.3e}")
    assert e < LOCAL360_BARS[0][0]
