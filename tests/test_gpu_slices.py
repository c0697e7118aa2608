"""Reference slices of the coarse pass (slice_chunk in csrc/t2x_estep.hip) against the FP64 oracle, at
the edges of the pixel chunks and of the volume's cells: from 9 pixels to two chunks (just under, just
over and well over 1024 pixels), so that waves end inside a quad and chunks inside a wave, with volume
widths of every remainder modulo the cell's three, global and local searches, 3D and 2D references.
diff2 within each precision's bound of the local-search parity tests (BF16x3, of 16 mantissa bits, 1e-4;
the others 1e-5).
"""
import numpy as np
import pytest

import estep_harness as H
import t2x_py as T
from test_gpu_local import LOCAL360_BARS, localise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("local", [False, True])
@pytest.mark.parametrize("name,size", [("refine64", 6), ("refine64", 20), ("refine64", 50), ("refine64", 52),
                                       ("refine64", 64), ("class2d64", 6), ("class2d64", 52)])
def test_slices(gpu_device, name, size, local):
    for prec in (T.T2X_PREC_FP32, T.T2X_PREC_FP16X3, T.T2X_PREC_BF16X3):
        wl = H.Workload(name, n=3, seed_offset=73, current_size=size, coarse_size=size, precision=prec,
                        K=2, overrides=dict(offset_range_px=1.0))
        if local:
            wl = localise(wl, 12.0 if name == "refine64" else 0.0, 15.0)
        o = wl.run_oracle(n_debug=3, fine_cap=4096)["dbg"]["coarse_diff2"]
        g = wl.run_gpu(dev=gpu_device, n_debug=3, fine_cap=4096)["dbg"]["coarse_diff2"]
        valid = o > -998
        assert valid.any() and np.array_equal(valid, g > -998)
        e = H.rel(g[valid], o[valid])
        print(f"precision {prec}: coarse diff2 max rel {e:.3e}")
        assert e < LOCAL360_BARS[prec][0]
