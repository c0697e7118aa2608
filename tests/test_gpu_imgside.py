"""The image-side rows of the coarse GEMM (k_coarse_imgside) at the edges of their split: rows shorter
than a wave's pixels, of one and of two staged chunks (over 2048 pixels), and 1, 9, 37 translations (below,
above and far above a group of eight rows), few particles (one translation a workgroup) and enough for
full groups, in each precision. diff2 against the FP64 oracle within each precision's bound of the
local-search parity tests.
"""
import numpy as np
import pytest

import estep_harness as H
import t2x_py as T
from test_gpu_local import LOCAL360_BARS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box,size,n,offsets", [(64, 10, 2, 0.5), (64, 30, 700, 1.5), (64, 44, 1900, 3.3),
                                                (96, 90, 2, 1.5), (96, 90, 1, 3.3)], ids=str)
def test_image_rows(gpu_device, box, size, n, offsets):
    for prec in (T.T2X_PREC_FP32, T.T2X_PREC_FP16X3, T.T2X_PREC_BF16X3):
        wl = H.Workload("refine64", n=n, seed_offset=83, current_size=size, coarse_size=size, precision=prec,
                        overrides=dict(ori_size=box, offset_range_px=offsets, offset_step_px=1.0, healpix_order=0))
        o = wl.run_oracle(n_debug=n, fine_cap=1024)["dbg"]["coarse_diff2"]
        g = wl.run_gpu(dev=gpu_device, n_debug=n, fine_cap=1024)["dbg"]["coarse_diff2"]
        valid = o > -998
        assert valid.any() and np.array_equal(valid, g > -998)
        e = H.rel(g[valid], o[valid])
        print(f"precision {prec}: coarse diff2 max rel {e:.3e}")
        assert e < LOCAL360_BARS[prec][0]
