"""The pruned coarse pass (t2x_estep_config.coarse_exhaustive 0) against the exhaustive one.

The coarse diff2 of a sample is a sum of non-negative pixel terms (1/2 minv |ctf F - X_t|^2, plus a
constant). An INT8 GEMM over a low set of the |frequency|-ordered coarse pixels, with its quantisation
errors and the rest of the pixels bounded by Cauchy-Schwarz, gives each 64-column block's lower bound; per
particle the full diff2 of one row of its most promising block gives an upper bound of its minimum (the
seed); the full GEMM then computes the tiles with a block not more than the negligible-weight cut (60,
plus one for rounding) above the seed. Every skipped block is one the selection already treats as
negligible, so poses, dLL, the significant sets, the weighted sums and the backprojections are those of
the exhaustive pass: identical, up to the run-to-run order of the store's atomic sums (weighted sums 1e-9,
backprojections 1e-6).

A call's first batch decides by a sample of its particles whether the pass is taken, and with which low
set; a batch whose list is too long (35% of the tiles; 60% in FP32) runs all its tiles and turns the pass
off for the rest of the call.

Covered: the three split precisions at class256 shapes (where most tiles are pruned; FP32 in
test_gpu_prune_bounds.py), a call that prunes nothing, a first low set that is too small, ragged batches,
batches that stop pruning, graph replays, operands of 4 GiB and more.
"""
import ctypes as C

import numpy as np
import pytest

import estep_harness as H
import t2x_py as T

pytestmark = pytest.mark.gpu


def run(wl, dev, exhaustive):
    lib = T.load()
    wl.cfg.coarse_exhaustive = 1 if exhaustive else 0
    T.check(lib.t2x_stats_reset(dev))
    r = wl.run_gpu(dev=dev)
    st = T.Stats()
    T.check(lib.t2x_stats_get(dev, C.byref(st)))
    wl.cfg.coarse_exhaustive = 0
    return r, (st.coarse_tiles_pruned, st.coarse_tiles_checked)


def same(g, ref):
    assert np.array_equal(g["out"]["best_hidden"], ref["out"]["best_hidden"])
    assert np.array_equal(g["out"]["dLL"], ref["out"]["dLL"])
    assert np.array_equal(g["out"]["nr_significant_coarse"], ref["out"]["nr_significant_coarse"])
    assert np.array_equal(g["out"]["nr_fine_samples"], ref["out"]["nr_fine_samples"])
    for k, v in ref["wsum"].items():
        if np.abs(v).sum() > 0:
            assert H.rel_norm(g["wsum"][k], v) < 1e-9, k
    for c in range(len(ref["bp"])):
        for q in (0, 1):
            if np.abs(ref["bp"][c][q]).sum() > 0:
                assert H.rel_norm(g["bp"][c][q], ref["bp"][c][q]) < 1e-6, (c, q)


@pytest.mark.parametrize("prec", [T.T2X_PREC_FP16X2, T.T2X_PREC_FP16X3, T.T2X_PREC_BF16X3])
def test_pruned_equals_exhaustive_class256(gpu_device, monkeypatch, prec):
    monkeypatch.setenv("T2X_BATCH", "6")   # 14 particles: batches of 6, 6 and 2
    wl = H.Workload("class256", n=14, seed_offset=81, precision=prec)
    ex, cnt_e = run(wl, gpu_device, True)
    pr, cnt_p = run(wl, gpu_device, False)
    print(f"\n[prune] class256 precision {prec}: {cnt_p[0]:.0f} of {cnt_p[1]:.0f} tiles pruned")
    assert cnt_e == (0, 0)
    assert cnt_p[1] > 0 and cnt_p[0] > 0.5 * cnt_p[1]
    same(pr, ex)


def test_call_that_does_not_prune_pays_for_a_sample(gpu_device):
    """Thirty times the noise: nothing prunes, and the bounds are those of a sample of the batch alone."""
    lib = T.load()
    wl = H.Workload("refine64", n=160, seed_offset=82, precision=T.T2X_PREC_FP16X2,
                    maximum_significants=200, overrides=dict(healpix_order=3))
    wl.sigma2 *= 30.0   # (the model points at it)
    pr, cnt = run(wl, gpu_device, False)
    st = T.Stats()
    T.check(lib.t2x_stats_get(gpu_device, C.byref(st)))
    ex, _ = run(wl, gpu_device, True)
    print(f"\n[prune] refine64: {cnt[0]:.0f} of {cnt[1]:.0f} tiles pruned, {st.coarse_bound_flop:.3g} bound flops")
    assert cnt[0] == 0 and 0 < cnt[1] <= 102 * 288 / 4   # a batch: 12,960 rows, 36,864 orientations
    assert 0 < st.coarse_bound_flop <= st.coarse_diff2_flop / 4
    same(pr, ex)


def test_pruned_small_prefix(gpu_device, monkeypatch):
    """A first low set of a quarter of the pixels keeps too many tiles: the call takes every pixel."""
    monkeypatch.setenv("T2X_BATCH", "6")
    monkeypatch.setenv("T2X_PRUNE_RADIUS", "0.5")
    wl = H.Workload("class256", n=12, seed_offset=83, precision=T.T2X_PREC_FP16X2)
    ex, _ = run(wl, gpu_device, True)
    pr, cnt = run(wl, gpu_device, False)
    print(f"\n[prune] class256, prefix radius 0.5: {cnt[0]:.0f} of {cnt[1]:.0f} tiles pruned")
    assert cnt[0] > 0.9 * cnt[1] > 0
    same(pr, ex)


def test_pruned_graph_replays_count_tiles(gpu_device, monkeypatch):
    """Batches replayed from a graph prune as the eager ones, and the tile counters see them."""
    lib = T.load()
    monkeypatch.setenv("T2X_BATCH", "4")   # 16 particles: a captured batch and two replays
    wl = H.Workload("class256", n=16, seed_offset=85, precision=T.T2X_PREC_FP16X2)
    eager, cnt_e = run(wl, gpu_device, False)
    wl.cfg.launch_graph = 1
    graph, cnt_g = run(wl, gpu_device, False)
    wl.cfg.launch_graph = 0
    st = T.Stats()
    T.check(lib.t2x_stats_get(gpu_device, C.byref(st)))
    print(f"\n[prune] graph: {st.n_graph_launches} graph launches, {cnt_g[0]:.0f} of {cnt_g[1]:.0f} tiles "
          f"pruned (eager {cnt_e[0]:.0f} of {cnt_e[1]:.0f})")
    assert st.n_graph_launches >= 2
    assert cnt_g == cnt_e
    same(graph, eager)


@pytest.mark.parametrize("prec", [T.T2X_PREC_FP32, T.T2X_PREC_FP16X2, T.T2X_PREC_BF16X3])
def test_later_batches_that_do_not_prune(gpu_device, monkeypatch, prec):
    """Five batches, of which the first two prune and the particles of the others (an optics group of
    thirty times the noise) do not: the pass is turned off after the third, and the exhaustive GEMM of
    the last two, whose shape has not been tuned in the process, runs eagerly before it is captured."""
    lib = T.load()
    monkeypatch.setenv("T2X_BATCH", "24")
    wl = H.Workload("refine64", n=120, seed_offset=87, precision=prec, snr=1.0,
                    maximum_significants=200, overrides=dict(healpix_order=3))
    later = (np.arange(120) >= 48).astype(int)
    wl.set_groups([wl.sigma2, 30.0 * wl.sigma2], group_of=np.zeros(120, int), optics_of=later)
    tiles = 16 * 288   # of a batch: 24 x 81 rows and 36,864 orientations, 128 x 128
    wl.cfg.launch_graph = 1
    graph, cnt_g = run(wl, gpu_device, False)   # first, so that no exhaustive launch has been tuned
    wl.cfg.launch_graph = 0
    st = T.Stats()
    T.check(lib.t2x_stats_get(gpu_device, C.byref(st)))
    eager, cnt_e = run(wl, gpu_device, False)
    ex, _ = run(wl, gpu_device, True)
    print(f"\n[prune] precision {prec}: {st.n_graph_launches} graph launches, {cnt_g[0]:.0f} of {cnt_g[1]:.0f} tiles "
          f"pruned (eager {cnt_e[0]:.0f} of {cnt_e[1]:.0f})")
    assert st.n_graph_launches == 3   # batches 2 (captured), 3 (replayed) and 5 (captured)
    assert cnt_g[1] == cnt_e[1] == 3 * tiles
    assert 1.7 * tiles < cnt_g[0] < 2.1 * tiles and cnt_g[0] == cnt_e[0]
    same(graph, ex)
    same(eager, ex)


@pytest.mark.parametrize("prec", [T.T2X_PREC_FP16X2, T.T2X_PREC_FP16X3, T.T2X_PREC_BF16X3])
def test_long_list_runs_all_tiles(gpu_device, monkeypatch, prec):
    """A batch behind one that pruned, with a list too long for the listed GEMM: all tiles, by the
    256 x 256 kernel (258), with the exhaustive pass's results."""
    lib = T.load()
    monkeypatch.setenv("T2X_BATCH", "64")
    wl = H.Workload("refine64", n=128, seed_offset=88, precision=prec, snr=1.0,
                    maximum_significants=200, overrides=dict(healpix_order=3))
    later = (np.arange(128) >= 64).astype(int)
    wl.set_groups([wl.sigma2, 30.0 * wl.sigma2], group_of=np.zeros(128, int), optics_of=later)
    pr, cnt = run(wl, gpu_device, False)
    st = T.Stats()
    T.check(lib.t2x_stats_get(gpu_device, C.byref(st)))
    ex, _ = run(wl, gpu_device, True)
    tiles = 41 * 288   # of a batch: 64 x 81 rows
    assert cnt[1] == 2 * tiles and 0.65 * tiles < cnt[0] < tiles
    assert st.gemm_tile_used == 258
    same(pr, ex)


@pytest.mark.parametrize("prec", [T.T2X_PREC_FP16X3, T.T2X_PREC_BF16X3, T.T2X_PREC_FP16X2])
def test_operands_beyond_4_gib(gpu_device, prec):
    """320 particles, 421 translations and 10,000 pixels: 5.4 GB of rows in each half. The three-product
    precisions prune as they run exhaustively; FP16X2 refuses them either way."""
    lib = T.load()
    wl = H.Workload("class2d64", n=320, seed_offset=89, precision=prec, snr=1.0, current_size=160,
                    overrides=dict(ori_size=160, particle_diameter=250.0, blob_radius=50.0, offset_range_px=11.5))
    wl.cfg.adaptive_oversampling = 0
    if prec == T.T2X_PREC_FP16X2:
        for exhaustive in (True, False):
            with pytest.raises(RuntimeError, match="4 GiB"):
                run(wl, gpu_device, exhaustive)
        return
    pr, cnt = run(wl, gpu_device, False)
    st = T.Stats()
    T.check(lib.t2x_stats_get(gpu_device, C.byref(st)))
    print(f"\n[prune] {st.P_coarse} pixels: {cnt[0]:.0f} of {cnt[1]:.0f} tiles pruned")
    assert 320 * wl.info.nr_trans * 2 * st.P_coarse * 2 > 1 << 32 and cnt[0] > 0
    ex, _ = run(wl, gpu_device, True)
    same(pr, ex)
