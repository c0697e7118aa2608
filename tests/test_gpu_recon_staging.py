"""Reconstruction inputs and maps through the page-locked slots (totals of 16 MiB and more, pieces of
4 MiB with remainders) against the plain copies of page-locked arrays, and the buffers and plans kept
between calls of changing sizes: each size again after another one, and the FSC between them.

The values are the same doubles on both ways; the weight floor's sums may differ in their last bits
between runs: 1e-12 relative (FP64 epsilon times the few thousand terms of a block's shell).
"""
import time

import numpy as np
import pytest
import torch

import estep_harness as H
import t2x_py as T
from test_gpu_recon import rand_volumes

pytestmark = pytest.mark.gpu


def run(dev, p, arrays, pinned):
    if pinned:
        arrays = [torch.empty(a.shape, dtype=torch.float64, pin_memory=True).copy_(torch.from_numpy(a)).numpy() for a in arrays]
        out = torch.zeros((p.ori_size,) * 3, dtype=torch.float64, pin_memory=True).numpy()
    else:
        out = np.zeros((p.ori_size,) * 3)
    T.check(T.load().t2x_reconstruct(dev, p, *[T.dptr(a) for a in arrays], None, T.dptr(out)), "reconstruct")
    return out


def test_staged_equals_plain(gpu_device):
    maps = {}
    for ori, r_max in [(32, 8), (130, 40), (128, 33), (32, 8), (130, 40), (140, 45)]:
        p = T.recon_params(ori, r_max)
        arrays = [np.ascontiguousarray(a) for a in rand_volumes(p, np.random.default_rng(ori + r_max))]
        a, b = run(gpu_device, p, arrays, False), run(gpu_device, p, arrays, True)
        print(f"box {ori}, r_max {r_max}: {sum(x.nbytes for x in arrays) / 2**20:.1f} MiB in", flush=True)
        assert np.isfinite(a).all() and np.abs(a).max() > 0
        assert H.rel_norm(a, b) < 1e-12
        if (ori, r_max) in maps:
            assert H.rel_norm(a, maps[ori, r_max]) < 1e-12
        maps[ori, r_max] = a
        fsc = np.zeros(ori // 2 + 1)
        T.check(T.load().t2x_fsc(gpu_device, ori, T.dptr(a), T.dptr(a), T.dptr(fsc)), "fsc")
        assert np.abs(fsc - 1).max() < 1e-9   # of a map with itself


def test_refused_call_leaves_no_copies(gpu_device):
    """r_max beyond the tau2 spectrum with page-locked arrays: nothing is on its way when the call returns
    (1.4 GB, 24 ms of the link at 57 GB/s, had been queued)."""
    p = T.recon_params(64, 120, do_map=True)
    n = p.pad_size * p.pad_size * (p.pad_size // 2 + 1)
    arrays = [torch.zeros(n, dtype=torch.float64, pin_memory=True).numpy() for _ in range(3)]
    out, tau2 = np.zeros((64,) * 3), np.ones(33)
    waits = []
    for _ in range(3):
        torch.cuda.synchronize()
        st = T.load().t2x_reconstruct(gpu_device, p, *[T.dptr(a) for a in arrays], T.dptr(tau2), T.dptr(out))
        t = time.perf_counter()
        torch.cuda.synchronize()   # the whole device
        waits.append(time.perf_counter() - t)
        assert st == T.T2X_EINVAL
    assert min(waits) < 0.005
