"""The INT8 bounds GEMM of the pruned coarse pass (csrc/t2x_prune.hip) at its edges: every forced batch
must give what the exhaustive pass gives (T2X_PRUNE_FORCE takes the bounds also where they would not
pay, so that wrong bounds would drop tiles that matter).

Edges: numbers of translations from 1 to 441 (the 8- and 24-particle base stages, the unstaged form,
particles that end inside 16-row blocks, span row tiles, or fill one row each), ragged particle and
orientation counts, low sets of 64 pixels up to every pixel, references of very different power,
classes and directions that are not scored, one pass at the current size, 2D references, optics and
image groups, each precision. Poses, dLL, significance and fine-sample counts are identical, weighted
sums and backprojections within the order of the store's atomic sums (1e-9, 1e-6).
"""
import ctypes as C

import numpy as np
import pytest

import estep_harness as H
import t2x_py as T
from test_gpu_coarse_prune import run, same

pytestmark = pytest.mark.gpu

FP32, BF16X3, FP16X3, FP16X2 = T.T2X_PREC_FP32, T.T2X_PREC_BF16X3, T.T2X_PREC_FP16X3, T.T2X_PREC_FP16X2


def check(wl, dev, monkeypatch):
    monkeypatch.setenv("T2X_PRUNE_FORCE", "1")
    ex, none = run(wl, dev, True)
    pr, cnt = run(wl, dev, False)
    print(f"\n[bounds] {cnt[0]:.0f} of {cnt[1]:.0f} tiles pruned")
    assert none == (0, 0) and cnt[1] > 0
    same(pr, ex)
    return cnt


def three_poses(truth):
    """Particles in three poses in turn: a tile of many particles is needed for three blocks at most, and
    bounds that go to a neighbour drop it."""
    n = len(truth["rot"])
    for k in ("rot", "tilt", "psi"):
        truth[k][:] = truth[k][np.arange(n) % 3].copy()
    truth["x"][:] = 0
    truth["y"][:] = 0


@pytest.mark.parametrize("offsets,n", [((0.5, 1.0), 300), ((1.0, 1.0), 61), ((2.0, 1.0), 40), ((2.5, 1.0), 33),
                                       ((3.3, 1.0), 27), ((4.0, 1.0), 9), ((11.5, 1.0), 3)],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("prec", [FP32, FP16X2])
def test_translations(gpu_device, monkeypatch, offsets, n, prec):
    wl = H.Workload("refine64", n=n, seed_offset=91, precision=prec, snr=3.0, truth_hook=three_poses,
                    overrides=dict(offset_range_px=offsets[0], offset_step_px=offsets[1]))
    cnt = check(wl, gpu_device, monkeypatch)
    assert cnt[0] > 0.7 * cnt[1]


@pytest.mark.parametrize("prec", [FP32, BF16X3, FP16X3, FP16X2])
@pytest.mark.parametrize("radius", ["0.35", "0.82", "1.5"])
def test_prefixes(gpu_device, monkeypatch, prec, radius):
    monkeypatch.setenv("T2X_PRUNE_RADIUS", radius)
    monkeypatch.setenv("T2X_BATCH", "7")
    wl = H.Workload("refine64", n=17, K=3, seed_offset=92, precision=prec, snr=1.0, overrides=dict(resolution=9.0))
    wl.ref_re[1] *= np.float32(1e-3)      # a class of hardly any power, and one with far too much
    wl.ref_im[1] *= np.float32(1e-3)
    wl.ref_re[2] *= np.float32(30)
    wl.ref_im[2] *= np.float32(30)
    cnt = check(wl, gpu_device, monkeypatch)
    assert cnt[0] > 0.5 * cnt[1]   # two of the classes without any doubt


@pytest.mark.parametrize("prec", [FP32, FP16X3])
def test_unscored_and_groups(gpu_device, monkeypatch, prec):
    wl = H.Workload("refine64", n=12, K=2, seed_offset=93, precision=prec, snr=0.5, old_offsets=True)
    nd = wl.info.nr_dir
    wl.pdf_dir[::3] = 0.0
    wl.pdf_dir[nd:nd + 40] = 0.0
    wl.pdf_dir /= wl.pdf_dir.sum()
    s2 = wl.sigma2
    wl.set_groups([s2, 1.7 * s2], group_of=np.arange(12) % 3, optics_of=np.arange(12) % 2, scale=[0.8, 1.0, 1.3],
                  dvp=np.full((2, wl.N // 2 + 1), 10.0))
    assert check(wl, gpu_device, monkeypatch)[0] > 0
    wl.pdf_class[:] = [0.0, 1.0]
    assert check(wl, gpu_device, monkeypatch)[0] > 0


@pytest.mark.parametrize("prec", [FP32, BF16X3])
def test_2d_and_one_pass(gpu_device, monkeypatch, prec):
    wl = H.Workload("class2d64", n=37, K=5, seed_offset=94, precision=prec, snr=0.5)
    assert check(wl, gpu_device, monkeypatch)[0] > 0
    wl = H.Workload("refine64", n=5, seed_offset=95, precision=prec, snr=0.5)
    wl.cfg.adaptive_oversampling = 0
    assert check(wl, gpu_device, monkeypatch)[0] > 0


@pytest.mark.parametrize("prec", [FP32, FP16X3])
def test_largest_low_set(gpu_device, monkeypatch, prec):
    """One pass at current size 190: 14,000 pixels, of which the low set takes the most that its LDS row
    holds (8,192), at 0.80 of the radius (9,000 pixels) as with every pixel asked for."""
    wl = H.Workload("class2d64", n=6, K=3, seed_offset=98, precision=prec, snr=1.0, current_size=190,
                    overrides=dict(ori_size=200, particle_diameter=300.0, blob_radius=60.0))
    wl.cfg.adaptive_oversampling = 0
    for radius in ("0.8", "1.5"):
        monkeypatch.setenv("T2X_PRUNE_RADIUS", radius)
        assert check(wl, gpu_device, monkeypatch)[0] > 0


def test_zero_references(gpu_device, monkeypatch):
    """References of zeros: every bound is its particle's constant, nothing is dropped. (The weighted sums
    run over every sample of the search in FP32 in no fixed order: two exhaustive runs differ by up to
    1.5e-9, so the poses and counts alone are compared.)"""
    monkeypatch.setenv("T2X_PRUNE_FORCE", "1")
    wl = H.Workload("refine64", n=4, seed_offset=96, precision=FP32)
    wl.ref_re[0][:] = 0
    wl.ref_im[0][:] = 0
    ex, _ = run(wl, gpu_device, True)
    pr, cnt = run(wl, gpu_device, False)
    assert cnt[0] == 0 < cnt[1]
    for k in ("best_hidden", "dLL", "nr_significant_coarse", "nr_fine_samples"):
        assert np.array_equal(pr["out"][k], ex["out"][k]), k


def test_fp32_class256(gpu_device, monkeypatch):
    """The benchmark workload's shapes in plain FP32: most tiles are pruned, unforced."""
    monkeypatch.setenv("T2X_BATCH", "6")
    wl = H.Workload("class256", n=8, seed_offset=97, precision=FP32)
    ex, _ = run(wl, gpu_device, True)
    pr, cnt = run(wl, gpu_device, False)
    assert cnt[0] > 0.5 * cnt[1]
    same(pr, ex)
