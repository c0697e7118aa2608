"""The work a user of t2x has it do, as measurable cases through the public C ABI (include/t2x.h).

Three kinds of case:

  estep   one expectation step of an iteration over a set of particles: the references set, the
          backprojectors zeroed, t2x_estep, the backprojected volumes of every class read back.
          Global 3D searches, 2D classification and local searches, in every cross-term precision.
  mstep   the reconstruction side of an iteration: two half-maps reconstructed and their FSC.
  train   one forward and backward pass of the pose-proposal network.

All particles are synthetic: Gaussian-blob molecules, projected, CTF-modulated and noised with the
signal-to-noise ratios, offsets and samplings of t2x_py/workloads.py, made on the GPU from the seed
alone. `exact` restates each kind in 64-bit torch from the formulas, without the library.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "t2-relion_amd", "python"))
import t2x_py as T  # noqa: E402

PRECISIONS = {"fp32": T.T2X_PREC_FP32, "bf16x3": T.T2X_PREC_BF16X3, "fp16x3": T.T2X_PREC_FP16X3,
              "fp16x2": T.T2X_PREC_FP16X2}
GPU = "cuda"
N_BINS = 768             # proposal network: 4 classes x 192 directions
MASK_EDGE = 5            # px
SIGMA2_OFFSET = 100.0    # A^2 (relion_refine --offset 10)
ADAPTIVE_FRACTION = 0.999

# What an E-step case says beyond this is said in the case.
ESTEP = dict(kind="estep", ref_dim=3, K=1, order=0, psi=0.0, sigma_ang=0.0, oversampling=1, precision="fp32",
             later=False, noise_background=False, host_images=False, zipf=0.0, snr_low=0.03, snr_high=0.03)


# ---------------------------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------------------------

def listed():
    """Each is a workload of this repository (t2x_py/workloads.py) or a state of one in a later iteration."""
    refine64 = dict(ESTEP, box=64, pixel=2.0, order=2, range_px=5.0, step_px=1.0, diameter=120.0, resolution=30.0,
                    blobs=200, snr_low=0.05, snr_high=0.05)
    class256 = dict(ESTEP, box=256, pixel=1.1, K=4, order=3, range_px=6.0, step_px=1.5, diameter=240.0,
                    resolution=10.0, blobs=800)
    class2d128 = dict(ESTEP, ref_dim=2, box=128, pixel=2.0, K=100, psi=6.0, range_px=5.0, step_px=1.0, diameter=200.0,
                      resolution=12.0, blobs=300, zipf=1.2, snr_low=0.01, snr_high=0.1)
    class2d64 = dict(ESTEP, ref_dim=2, box=64, pixel=2.0, K=4, psi=6.0, range_px=5.0, step_px=1.0, diameter=110.0,
                     resolution=20.0, blobs=150, snr_low=0.05, snr_high=0.05)
    local360 = dict(ESTEP, box=360, pixel=0.9, order=5, sigma_ang=3.0, range_px=3.0, step_px=0.5, diameter=300.0,
                    blobs=1500, snr_low=0.02, snr_high=0.02, later=True)
    return [
        # one particle a call, as a per-particle driver makes it: latency, launches, host tables
        dict(refine64, name="refine64_single", n=1),
        # the whole small 3D refinement, in plain FP32
        dict(refine64, name="refine64_fp32", n=1000),
        # 3D classification: the plain FP32 path, then the fastest path over several batches
        dict(class256, name="class256_fp32", n=800),
        dict(class256, name="class256_fp16x2", n=4000, precision="fp16x2"),
        # the same in a later iteration from host memory: norm and scale corrections, two optics groups, four
        # image groups, known offsets, relion_refine's default noise-filled mask background
        dict(class256, name="class256_later_fp16x3", n=1000, precision="fp16x3", later=True, noise_background=True,
             host_images=True),
        # 2D classification with uneven classes, and its small form in FP32
        dict(class2d128, name="class2d128_fp16x2", n=8192, precision="fp16x2"),
        dict(class2d64, name="class2d64_fp32", n=2000),
        # local refinement late in a run (current size 206), and at its start with fewer particles in FP32
        dict(local360, name="local360_bf16x3", n=3000, resolution=3.5, precision="bf16x3"),
        dict(local360, name="local360_fp32", n=500, resolution=7.0),
        # M-step of a 3D class: two half-maps of a 256 box at 4.7 A and their FSC; the same of a small box
        dict(kind="mstep", name="mstep256", box=256, r_max=60, do_map=True, blobs=800),
        dict(kind="mstep", name="mstep64", box=64, r_max=20, do_map=False, blobs=200),
        # one optimiser step's pass of the pose-proposal network, at its training batch
        dict(kind="train", name="proposal_step256", batch=256, bf16=True),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _even(x):
    return 2 * max(1, int(round(x / 2)))


def draw(rng):
    """One more case: the same kinds, precisions and options over the sizes in between, odd ones among them."""
    kind = rng.choices(["global", "2d", "local", "mstep", "train"], [8, 5, 4, 2, 1])[0]
    if kind == "mstep":
        box = _even(_log_uniform(rng, 48, 288))
        return dict(kind="mstep", box=box, r_max=rng.randint(box // 8, box // 3), do_map=rng.random() < 0.5,
                    blobs=rng.randint(100, 600))
    if kind == "train":
        return dict(kind="train", batch=rng.randint(1, 384), bf16=rng.random() < 0.8)
    precision = rng.choice(list(PRECISIONS))
    later = rng.random() < 0.5
    box = _even(_log_uniform(rng, 48, 200 if kind == "2d" else 300))
    pixel = round(rng.uniform(0.8, 2.5), 2)
    diameter = round(box * pixel * rng.uniform(0.6, 0.84), 1)
    # signal-to-noise ratio: the signal energy over the noise of a Fourier component as in the listed workloads
    # (100 at refine64, 1,000 at class256)
    snr = 2 * _log_uniform(rng, 100, 1000) / box ** 2
    # the resolution reached so far: a Fourier shell between a tenth and a third of the box
    resolution = round(box * pixel / rng.uniform(box / 10.0, box / 3.0), 2)
    # a molecule whose blobs (about 170 voxels each) fill between a thirtieth and half of its ball
    ball = 4 / 3 * math.pi * (0.8 * diameter / (2 * pixel)) ** 3
    blobs = int(min(600, max(40, ball * _log_uniform(rng, 0.03, 0.5) / 170)))
    case = dict(ESTEP, box=box, pixel=pixel, diameter=diameter, resolution=resolution, blobs=blobs,
                snr_low=snr, snr_high=snr, precision=precision, later=later, noise_background=rng.random() < 0.25,
                host_images=rng.random() < 0.25, range_px=round(rng.uniform(2.0, 6.0), 1))
    case["step_px"] = round(case["range_px"] / rng.uniform(2.0, 6.0), 2)
    if kind == "2d":
        case.update(ref_dim=2, K=int(round(_log_uniform(rng, 2, 100))), psi=rng.choice([5.0, 6.0, 8.0, 10.0, 12.0]),
                    zipf=rng.choice([0.0, 1.2]), snr_low=snr / 2, snr_high=2 * snr)
    elif kind == "global":
        case.update(K=rng.randint(1, 5), order=rng.choice([1, 2, 2, 3]))
        if box < 100 and rng.random() < 0.2:
            case.update(oversampling=rng.choice([0, 2]), order=1)
    else:
        case.update(order=rng.choice([3, 4, 5]), sigma_ang=round(rng.uniform(2.0, 5.0), 1), K=rng.randint(1, 2),
                    later=True)
    case["n"] = 1
    most = 1.2e13 if precision == "fp32" else 3e13   # below the listed cases of the same path
    if kind == "local":
        most = 4e11
    cap = min(6000, int(most / work(case)["flops"]), int(1.2e9 / box ** 2 / 4))
    case["n"] = max(1, int(_log_uniform(rng, max(1, cap / 60), max(2, cap))))
    return case


# ---------------------------------------------------------------------------------------------
# Sizes and grids (HealpixSampling and MlOptimiser::updateImageSizeAndResolutionPointers)
# ---------------------------------------------------------------------------------------------

class Sizes:
    """Image sizes of an E-step case's two passes and its sampling counts."""

    def __init__(self, c):
        N, pix = c["box"], c["pixel"]
        self.N = N
        self.ang = 360.0 / (6 * 2 ** c["order"]) if c["ref_dim"] == 3 else c["psi"]
        self.current = min(2 * (int(N * pix / c["resolution"] + 0.5) + 10), N)
        coarse_res = self.ang / 360.0 * math.pi * c["diameter"] / (1.2 if c["ref_dim"] == 3 else 1.5)
        self.coarse = min(2 * math.ceil(pix * N / coarse_res), self.current)
        self.first = self.current if c["oversampling"] == 0 else self.coarse   # image size of the first pass
        self.r_max = self.current // 2
        self.pad = 2 * (2 * self.r_max + 1) + 1
        self.xdim = self.pad // 2 + 1
        self.n_voxels = (self.pad if c["ref_dim"] == 3 else 1) * self.pad * self.xdim
        self.n_dir = 12 * 4 ** c["order"] if c["ref_dim"] == 3 else 1
        self.n_psi = math.ceil(360.0 / self.ang)
        step, reach = c["step_px"] * pix, c["range_px"] * pix
        m = math.ceil(reach / step)
        self.trans = [(x * step, y * step) for x in range(-m, m + 1) for y in range(-m, m + 1)
                      if (x * step) ** 2 + (y * step) ** 2 < reach * reach + 0.001]
        self.step = step


def _pixels(size, origin):
    """(x, y, shell, projected) of the pixels of a pass: FFTW half layout, the Friedel half of x = 0 left out;
    `origin`: whether the zero frequency is one of them (the weighted sums), or not (diff2)."""
    xs = size // 2 + 1
    y = np.arange(size)
    y = np.where(y < xs, y, y - size)[:, None] + np.zeros((1, xs), int)
    x = np.arange(xs)[None, :] + np.zeros((size, 1), int)
    shell = np.floor(np.sqrt(x * x + y * y) + 0.5).astype(int)
    keep = (shell < xs) & ~((x == 0) & (y < 0))
    if not origin:
        keep &= shell > 0
    return x[keep], y[keep], shell[keep], (x * x + y * y <= (xs - 1) ** 2)[keep]


def _local_rows(c, s):
    """Expected orientations in range of one particle of a local search."""
    cap = (1 - math.cos(math.radians(min(180.0, 3 * c["sigma_ang"])))) / 2
    return max(1.0, s.n_dir * cap) * min(s.n_psi, max(1.0, s.n_psi * 6 * c["sigma_ang"] / 360))


def work(case):
    """E-step: every sample of the first pass scored once (4 flops per pixel of the complex cross term, the
    definition of the search); the images, references and priors read, the volumes and metadata written once."""
    if case["kind"] == "train":
        B = case["batch"]
        per = 2 * (32 * 32 * 9 * 32 + 16 * 16 * 288 * 64 + 8 * 8 * 576 * 128 + 4 * 4 * 1152 * 128 + 2048 * (N_BINS + 2))
        n_par = 32 * 10 + 64 * 289 + 128 * 577 + 128 * 1153 + 2049 * (N_BINS + 2)
        return {"bytes": 4.0 * (B * (4096 + N_BINS + 5) + 2 * n_par), "flops": 3.0 * B * per}
    if case["kind"] == "mstep":
        pad, ori = 4 * case["r_max"] + 3, case["box"]
        big, fft = (2 * ori) ** 3, 2.5 * math.log2(max(2, ori)) * 3
        return {"bytes": 2.0 * (24 * pad * pad * (pad // 2 + 1) + 8 * ori ** 3) + 16.0 * ori ** 3,
                "flops": 2 * fft * big + 2 * fft * ori ** 3}
    s = Sizes(case)
    rows = case["K"] * (_local_rows(case, s) if case["sigma_ang"] else s.n_dir * s.n_psi)
    P = len(_pixels(s.first, False)[0])
    return {"bytes": case["n"] * (4.0 * s.N ** 2 + 400) + case["K"] * s.n_voxels * (8.0 + 24.0),
            "flops": 4.0 * case["n"] * rows * len(s.trans) * P}


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------

def _euler(rot, tilt, psi):
    """Euler_angles2matrix as nine arrays (degrees)."""
    a, b, g = (np.radians(v) for v in (rot, tilt, psi))
    ca, sa, cb, sb, cg, sg = np.cos(a), np.sin(a), np.cos(b), np.sin(b), np.cos(g), np.sin(g)
    return np.stack([cg * cb * ca - sg * sa, cg * cb * sa + sg * ca, -cg * sb,
                     -sg * cb * ca - cg * sa, -sg * cb * sa + cg * ca, sg * sb, sb * ca, sb * sa, cb], -1)


def _blobs(r, n, radius):
    """Centres in a ball, widths and amplitudes of one molecule: [n][5]."""
    d = r.normal(size=(n, 3))
    d *= (radius * r.uniform(0, 1, (n, 1)) ** (1 / 3)) / np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([d, r.uniform(1.5, 3.0, (n, 1)), r.uniform(0.5, 1.0, (n, 1))], 1)


def _reference(blobs, N, pad, r_max, cutoff, flat):
    """Fourier transform / N^2 of a molecule on the projector grid (padding 2), low-passed at shell `cutoff`;
    `flat`: the central plane alone (a 2D class average). float32 (re, im) on the GPU."""
    b = torch.tensor(blobs, device=GPU)
    h, xdim = pad // 2, pad // 2 + 1
    k = torch.arange(-h, h + 1, device=GPU, dtype=torch.float64)

    def axis(f, i):   # [len(f)][blobs]: the separable factor of axis i
        f = f[:, None] / (2 * N)
        return torch.polar(torch.exp(-2 * math.pi ** 2 * b[None, :, 3] ** 2 * f * f), -2 * math.pi * f * b[None, :, i])

    gx, gy, gz = (axis(f, i).to(torch.complex64) for i, f in enumerate((k[h:], k, k[h:h + 1] if flat else k)))
    amp = (b[:, 4] * (2 * math.pi * b[:, 3] ** 2) ** 1.5 / N ** 2).to(torch.complex64)
    gx = (gx * amp).T.contiguous()
    F = torch.stack([(gy * z) @ gx for z in gz])
    kz = k[h:h + 1] if flat else k
    r2 = kz[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, h:] ** 2
    shell = torch.sqrt(r2) / 2
    low = (0.5 + 0.5 * torch.cos(math.pi * ((shell - cutoff + 1) / 2).clamp(0, 1))) * (r2 <= (2 * r_max) ** 2)
    F = (F * low.to(torch.float32)).reshape(-1)
    return F.real.contiguous(), F.imag.contiguous()


def _ctf(p, N, pix, x, y):
    """CTF of every particle (p: defocus u, v, angle; 300 kV, 2.7 mm, 0.1) at the frequencies (x, y): [n][P]."""
    kv = 300e3
    lam = 12.2643247 / math.sqrt(kv * (1.0 + kv * 0.978466e-6))
    k1, k2 = math.pi * lam, math.pi / 2 * 2.7e7 * lam ** 3
    k3 = math.atan(0.1 / math.sqrt(1 - 0.01))
    u, v, a = (torch.tensor(p[key], device=GPU)[:, None] for key in ("defocus_u", "defocus_v", "defocus_angle"))
    s, co = torch.sin(a * math.pi / 180), torch.cos(a * math.pi / 180)
    X, Y = x[None] / (N * pix), y[None] / (N * pix)
    u2 = X * X + Y * Y
    phase = (co * co * -u + s * s * -v) * X * X + 2 * co * s * (v - u) * X * Y + (s * s * -u + co * co * -v) * Y * Y
    r = -torch.sin(k1 * phase + k2 * u2 * u2 - k3)
    return torch.where(r.abs() < 1e-8, torch.where(r >= 0, 1e-8, -1e-8).to(r.dtype), r)


def _particles(c, s, r):
    """True poses, offsets, CTFs and the metadata of n particles."""
    n, K, flat = c["n"], c["K"], c["ref_dim"] == 2
    freq = 1.0 / np.arange(1, K + 1) ** c["zipf"]
    p = dict(cls=r.choice(K, n, p=freq / freq.sum()), rot=r.uniform(-180, 180, n),
             tilt=np.degrees(np.arccos(r.uniform(-1, 1, n))), psi=r.uniform(-180, 180, n),
             x=r.uniform(-0.8, 0.8, n) * c["range_px"], y=r.uniform(-0.8, 0.8, n) * c["range_px"],
             defocus_u=r.uniform(10000, 30000, n), defocus_v=r.uniform(10000, 30000, n),
             defocus_angle=r.uniform(0, 180, n), snr=np.exp(r.uniform(np.log(c["snr_low"]), np.log(c["snr_high"]), n)),
             old_x=np.zeros(n), old_y=np.zeros(n), norm=np.ones(n), group=np.zeros(n, int), optics=np.zeros(n, int))
    if flat:
        p["rot"], p["tilt"] = np.zeros(n), np.zeros(n)
    if c["later"]:   # offsets found before, norms, image and optics groups
        p["old_x"], p["old_y"] = (r.integers(-2, 3, n).astype(float) for _ in range(2))
        p["norm"] = r.uniform(0.9, 1.1, n)
        p["group"], p["optics"] = r.integers(0, 4, n), r.integers(0, 2, n)
    e = r.normal(0, 1, (3, n)) / 3 * c["sigma_ang"] if c["sigma_ang"] else np.zeros((3, n))
    p["prior_rot"], p["prior_psi"] = p["rot"] + e[0], (p["psi"] + e[2] + 180) % 360 - 180
    p["prior_tilt"] = np.clip(p["tilt"] + e[1], 0, 180)
    if c["sigma_ang"]:   # a local search's driver takes particles in order of their prior orientation
        cell = np.stack([p["prior_psi"], (p["prior_rot"] % 360) // 10,
                         np.clip((np.cos(np.radians(p["prior_tilt"])) + 1) * 18, 0, 35) // 1])
        order = np.lexsort(cell)
        p = {k: v[order] for k, v in p.items()}
    return p


def _images(c, s, p, blobs, gen):
    """Noisy CTF-modulated projections (float32, on the GPU) and the mean noise variance."""
    N, pix, n = s.N, c["pixel"], c["n"]
    A = torch.tensor(_euler(p["rot"], p["tilt"], p["psi"]).reshape(n, 3, 3), device=GPU)
    mol = torch.tensor(np.stack(blobs), device=GPU)
    g = torch.arange(N, device=GPU, dtype=torch.float32) - N // 2
    fx = torch.arange(N // 2 + 1, device=GPU, dtype=torch.float64)
    fy = torch.fft.fftfreq(N, 1.0 / N, device=GPU, dtype=torch.float64)
    gx, gy = (v.reshape(-1) for v in torch.meshgrid(fy, fx, indexing="ij")[::-1])
    out, var_sum = torch.empty(n, N, N, device=GPU), 0.0
    step = max(1, int(2e8 / (N * c["blobs"])))
    for b0 in range(0, n, step):
        i = slice(b0, min(n, b0 + step))
        m = mol[torch.tensor(p["cls"][i], device=GPU)]
        xy = torch.einsum("bij,bkj->bik", A[i, :2], m[..., :3])
        cx = xy[:, 0] + torch.tensor(p["x"][i], device=GPU)[:, None]
        cy = xy[:, 1] + torch.tensor(p["y"][i], device=GPU)[:, None]
        w = (-0.5 / m[..., 3] ** 2).float()[:, None]
        ex = torch.exp((g[None, :, None] - cx[:, None].float()) ** 2 * w)
        ey = torch.exp((g[None, :, None] - cy[:, None].float()) ** 2 * w)
        ey *= (m[..., 4] * math.sqrt(2 * math.pi) * m[..., 3]).float()[:, None]
        img = torch.bmm(ey, ex.transpose(1, 2).contiguous())
        q = {k: p[k][i] for k in ("defocus_u", "defocus_v", "defocus_angle")}
        ctf = _ctf(q, N, pix, gx, gy).reshape(-1, N, N // 2 + 1).float()
        img = torch.fft.irfft2(torch.fft.rfft2(img) * ctf, s=(N, N))
        sd = torch.sqrt(img.var(dim=(1, 2)) / torch.tensor(p["snr"][i], device=GPU)).float()
        var_sum += float((sd ** 2).sum())
        img += torch.randn(img.shape, device=GPU, generator=gen) * sd[:, None, None]
        out[i] = img * torch.tensor(p["norm"][i], device=GPU).float()[:, None, None]
    for b in range(n if c["later"] else 0):   # the offsets of the images before they were found
        if p["old_x"][b] or p["old_y"][b]:
            out[b] = torch.roll(out[b], (-int(p["old_y"][b]), -int(p["old_x"][b])), (0, 1))
    return out, var_sum / n


def _estep_inputs(c, seed):
    """Everything an E-step is given, from the seed alone: torch and numpy only."""
    s = Sizes(c)
    r = np.random.default_rng([seed, 1])
    gen = torch.Generator(device=GPU)
    gen.manual_seed(seed)
    blobs = [_blobs(r, c["blobs"], 0.8 * c["diameter"] / (2 * c["pixel"])) for _ in range(c["K"])]
    p = _particles(c, s, r)
    images, var = _images(c, s, p, blobs, gen)
    cutoff = s.N * c["pixel"] / c["resolution"]
    refs = [_reference(b, s.N, s.pad, s.r_max, cutoff, c["ref_dim"] == 2) for b in blobs]
    # noise spectra: the images' white noise through the soft mask
    g = np.arange(s.N) - s.N // 2
    rad = c["diameter"] / (2 * c["pixel"])
    d = np.sqrt(g[:, None] ** 2 + g[None] ** 2)
    mask = 0.5 + 0.5 * np.cos(np.pi * np.clip((d - rad) / MASK_EDGE, 0, 1))
    n_og, xs = 2 if c["later"] else 1, s.N // 2 + 1
    level = var * float((mask ** 2).mean()) / (2 * s.N ** 2)
    sigma2 = level * (1 + 0.2 * np.arange(n_og)[:, None]) * (1 + 0.1 * np.cos(np.arange(xs) / 7.0))[None]
    pdf_class = r.uniform(0.5, 1.5, c["K"])
    pdf_dir = r.uniform(0.5, 1.5, (c["K"], s.n_dir))
    dvp = 30 * np.exp(-np.arange(xs) / (0.2 * xs))[None] + np.zeros((c["K"], 1))
    return dict(sizes=s, p=p, images=images, refs=refs, sigma2=np.ascontiguousarray(sigma2),
                pdf_class=pdf_class / pdf_class.sum(), pdf_dir=np.ascontiguousarray(pdf_dir / pdf_dir.sum()),
                scale=np.array([0.9, 1.0, 1.05, 1.1]) if c["later"] else np.ones(1), dvp=np.ascontiguousarray(dvp),
                n_og=n_og)


def _mstep_inputs(c, seed):
    """Backprojected sums of two half-sets: a molecule's transform times a weight that falls with the frequency
    (planes through the origin) with the noise of finite data, and its tau2 spectrum. Host doubles, as
    BackProjector holds them."""
    r_max, N = c["r_max"], c["box"]
    pad = 4 * r_max + 3
    r = np.random.default_rng([seed, 2])
    gen = torch.Generator(device=GPU)
    gen.manual_seed(seed)
    re, im = _reference(_blobs(r, c["blobs"], 0.3 * N), N, pad, r_max, 0.8 * r_max, False)
    h = pad // 2
    k = torch.arange(-h, h + 1, device=GPU, dtype=torch.float64)
    rad = torch.sqrt(k[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, h:] ** 2).reshape(-1)
    inside = rad <= 2 * r_max
    V = torch.complex(re.double(), im.double())
    noise = 0.02 * float(V.abs()[inside].square().mean().sqrt())
    halves = []
    for _ in range(2):
        def normal():
            return torch.randn(V.shape, device=GPU, generator=gen, dtype=torch.float64)
        w = 2000.0 / (1 + rad) * torch.exp(0.3 * normal()) * inside
        d = (V + noise * torch.complex(normal(), normal())) * w
        halves.append(tuple(t.contiguous().cpu().numpy() for t in (d.real, d.imag, w)))
    shells = np.arange(N // 2 + 1)
    tau2 = noise ** 2 * (1 + 50 * np.exp(-shells / (0.3 * r_max)))
    return halves, np.ascontiguousarray(tau2)


def _train_inputs(c, seed):
    """Weights (He-uniform), noisy crops, labels and shift targets of one training batch."""
    r = np.random.default_rng([seed, 3])
    par = []
    for cin, cout in ((1, 32), (32, 64), (64, 128), (128, 128)):
        par += [r.uniform(-1, 1, cout * 9 * cin) * math.sqrt(6 / (9 * cin)), 0.05 * r.normal(size=cout)]
    par += [r.uniform(-1, 1, 2048 * (N_BINS + 2)) * math.sqrt(6 / 2048), 0.05 * r.normal(size=N_BINS + 2)]
    B = c["batch"]
    y, x = np.mgrid[0:64, 0:64]
    cen = r.uniform(20, 44, (B, 2, 1, 1))
    img = 2 * np.exp(-((y - cen[:, 0]) ** 2 + (x - cen[:, 1]) ** 2) / 60) + r.normal(size=(B, 64, 64))
    return dict(params=np.concatenate(par).astype(np.float32), x=img.astype(np.float32),
                label=r.integers(0, N_BINS, B).astype(np.int32),
                shift=np.ascontiguousarray(r.uniform(-1, 1, (B, 2)).astype(np.float32)))


# ---------------------------------------------------------------------------------------------
# Running
# ---------------------------------------------------------------------------------------------

_HANDLE = []


def _device():
    """The device handle, opened once and kept, as a program does."""
    if not _HANDLE:
        h = C.c_void_p()
        T.check(T.load().t2x_device_open(0, C.byref(h)), "t2x_device_open")
        _HANDLE.append(h)
    return _HANDLE[0]


def _prepare_estep(c, seed):
    inp = _estep_inputs(c, seed)
    s, p, n, K, flat = inp["sizes"], inp["p"], c["n"], c["K"], c["ref_dim"] == 2
    later = c["later"]
    cfg = T.EstepConfig(ori_size=s.N, pixel_size=c["pixel"], current_size=s.current, coarse_size=s.coarse, nr_classes=K,
                        ref_dim=c["ref_dim"], healpix_order=c["order"], psi_step=s.ang,
                        offset_range=c["range_px"] * c["pixel"], offset_step=c["step_px"] * c["pixel"],
                        adaptive_oversampling=c["oversampling"], adaptive_fraction=ADAPTIVE_FRACTION,
                        particle_diameter=c["diameter"], width_mask_edge=MASK_EDGE,
                        do_zero_mask=0 if c["noise_background"] else 1, random_seed=seed, sigma2_fudge=1.0,
                        do_norm_correction=1 if later else 0, avg_norm_correction=1.0,
                        do_scale_correction=1 if later else 0, nr_groups=len(inp["scale"]),
                        nr_optics_groups=inp["n_og"], do_ctf_correction=1, sigma2_offset=SIGMA2_OFFSET,
                        orientational_prior_mode=1 if c["sigma_ang"] else 0, sigma_rot=c["sigma_ang"],
                        sigma_tilt=c["sigma_ang"], sigma_psi=c["sigma_ang"], precision=PRECISIONS[c["precision"]])
    pin = (T.ParticleIn * n)()
    for i in range(n):
        q = pin[i]
        q.ctf = T.CtfParams(300.0, 2.7, 0.1, p["defocus_u"][i], p["defocus_v"][i], p["defocus_angle"][i], 0.0, 0.0, 1.0)
        q.old_offset_x, q.old_offset_y = p["old_x"][i], p["old_y"][i]
        q.prior_offset_x, q.prior_offset_y = (p["old_x"][i], p["old_y"][i]) if later else (999.0, 999.0)
        q.norm_correction = p["norm"][i]
        q.prior_rot, q.prior_tilt, q.prior_psi = ((p["prior_rot"][i], p["prior_tilt"][i], p["prior_psi"][i])
                                                  if c["sigma_ang"] else (999.0, 999.0, 999.0))
        q.group_id, q.optics_group, q.part_id = int(p["group"][i]), int(p["optics"][i]), i
    images = inp["images"].cpu().numpy() if c["host_images"] else inp["images"]
    out = (T.ParticleOut * n)()
    fields = np.frombuffer(out, dtype=np.dtype(
        [(f, {C.c_double: "f8", C.c_long: "i8", C.c_int: "i4"}[t]) for f, t in T.ParticleOut._fields_]))
    wsum, sums = T.make_wsum(K, s.n_dir, s.N, inp["n_og"], len(inp["scale"]))
    bp = [np.zeros((K, s.n_voxels)) for _ in range(3)]
    model = T.Model(T.dptr(inp["sigma2"]), T.dptr(inp["pdf_class"]), T.dptr(inp["pdf_dir"]), None,
                    T.dptr(inp["scale"]), T.dptr(inp["dvp"]))
    torch.cuda.synchronize()   # the library has its own stream
    return dict(kind="estep", dev=_device(), sizes=s, flat=flat, cfg=cfg, pin=pin, images=images, out=out,
                particles={f: fields[f] for f in fields.dtype.names if f != "pad0"}, wsum=wsum, sums=sums, bp=bp,
                model=model, n=n, K=K, on_device=0 if c["host_images"] else 1, refs=inp["refs"], keep=inp)


def prepare(case, seed):
    if case["kind"] == "estep":
        return _prepare_estep(case, seed)
    if case["kind"] == "mstep":
        halves, tau2 = _mstep_inputs(case, seed)
        N = case["box"]
        return dict(kind="mstep", dev=_device(), halves=halves, tau2=tau2, n=N,
                    params=T.recon_params(N, case["r_max"], do_map=case["do_map"]),
                    maps=[np.zeros((N, N, N)) for _ in range(2)], fsc=np.zeros(N // 2 + 1))
    st = _train_inputs(case, seed)
    T.check(T.load().t2x_proposal_init(_device(), N_BINS, 1), "t2x_proposal_init")
    return dict(st, kind="train", dev=_device(), batch=case["batch"], bf16=1 if case["bf16"] else 0,
                loss=C.c_double(), grad=np.zeros_like(st["params"]),
                outputs=np.zeros((case["batch"], N_BINS + 2), np.float32))


def _ptr(t):
    return C.cast(C.c_void_p(t.data_ptr()), C.POINTER(C.c_float))


def _run_estep(st):
    lib, dev, s, dim = T.load(), st["dev"], st["sizes"], 2 if st["flat"] else 3
    for k, (re, im) in enumerate(st["refs"]):
        T.check(lib.t2x_projector_set(dev, k, dim, s.pad, s.r_max, 2.0, _ptr(re), _ptr(im)), "t2x_projector_set")
        T.check(lib.t2x_backprojector_init(dev, k, dim, s.pad, s.r_max, 2.0), "t2x_backprojector_init")
    for a in st["sums"].values():
        a[:] = 0
    images = st["images"].data_ptr() if st["on_device"] else st["images"].ctypes.data
    T.check(lib.t2x_estep(dev, C.byref(st["cfg"]), C.byref(st["model"]), st["n"], images, st["on_device"], st["pin"],
                          st["out"], C.byref(st["wsum"]), None), "t2x_estep")
    re, im, w = st["bp"]
    for k in range(st["K"]):
        T.check(lib.t2x_backprojector_get(dev, k, T.dptr(re[k]), T.dptr(im[k]), T.dptr(w[k])), "t2x_backprojector_get")
    return dict(particles=st["particles"], sums=st["sums"], bp_re=re, bp_im=im, bp_weight=w)


def run(state):
    lib, dev = T.load(), state["dev"]
    if state["kind"] == "estep":
        return _run_estep(state)
    if state["kind"] == "mstep":
        tau2 = T.dptr(state["tau2"])
        for (re, im, w), vol in zip(state["halves"], state["maps"]):
            T.check(lib.t2x_reconstruct(dev, C.byref(state["params"]), T.dptr(re), T.dptr(im), T.dptr(w), tau2,
                                        T.dptr(vol)), "t2x_reconstruct")
        T.check(lib.t2x_fsc(dev, state["n"], T.dptr(state["maps"][0]), T.dptr(state["maps"][1]), T.dptr(state["fsc"])),
                "t2x_fsc")
        return dict(maps=state["maps"], fsc=state["fsc"])
    par = state["params"]
    T.check(lib.t2x_proposal_set_params(dev, T.fptr(par), par.size), "t2x_proposal_set_params")
    T.check(lib.t2x_proposal_loss_grad(dev, state["batch"], T.fptr(state["x"]),
                                       state["label"].ctypes.data_as(C.POINTER(C.c_int)), T.fptr(state["shift"]), 1.0,
                                       state["bf16"], C.byref(state["loss"]), T.fptr(state["grad"]),
                                       T.fptr(state["outputs"])), "t2x_proposal_loss_grad")
    return dict(loss=state["loss"].value, grad=state["grad"], outputs=state["outputs"])


# ---------------------------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------------------------

def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    if case["kind"] == "mstep":
        halves, tau2 = _mstep_inputs(case, seed)
        maps = [_exact_reconstruct(case, *h, tau2) for h in halves]
        return dict(maps=[m.cpu().numpy() for m in maps], fsc=_exact_fsc(*maps))
    if case["noise_background"]:
        return None   # the background is drawn inside the library
    if case["sigma_ang"]:   # samples of the search that torch would take longer than 20 s over
        s = Sizes(case)
        if case["n"] * case["K"] * _local_rows(case, s) * len(_pixels(s.first, False)[0]) > 8e9:
            return None
    return ExactEstep(case, _estep_inputs(case, seed)).result()


def _exact_train(c, seed):
    q = _train_inputs(c, seed)
    flat = torch.tensor(q["params"], device=GPU, dtype=torch.float64, requires_grad=True)
    at = [0]

    def take(*shape):
        at[0] += math.prod(shape)
        return flat[at[0] - math.prod(shape):at[0]].reshape(shape)

    B = c["batch"]
    a = torch.tensor(q["x"], device=GPU, dtype=torch.float64)[:, None]
    for cin, cout in ((1, 32), (32, 64), (64, 128), (128, 128)):
        w, b = take(cout, 3, 3, cin), take(cout)
        cols = torch.nn.functional.unfold(a, 3, padding=1, stride=2)            # [B][cin * 9][pixels]
        z = w.permute(0, 3, 1, 2).reshape(cout, -1) @ cols.permute(1, 0, 2).reshape(cin * 9, -1) + b[:, None]
        side = a.shape[2] // 2
        a = torch.relu(z).reshape(cout, B, side, side).permute(1, 0, 2, 3)
    feat = a.permute(0, 2, 3, 1).reshape(B, -1)
    w, b = take(N_BINS + 2, 2048), take(N_BINS + 2)
    y = feat @ w.T + b
    label = torch.tensor(q["label"], device=GPU, dtype=torch.int64)
    shift = torch.tensor(q["shift"], device=GPU, dtype=torch.float64)
    loss = torch.nn.functional.cross_entropy(y[:, :-2], label) + ((y[:, -2:] - shift) ** 2).sum(1).mean()
    loss.backward()
    return dict(loss=float(loss.detach()), grad=flat.grad.cpu().numpy(), outputs=y.detach().cpu().numpy())


def _exact_reconstruct(c, re, im, w, tau2):
    N, r_max = c["box"], c["r_max"]
    pad = 4 * r_max + 3
    h, xh, dims = pad // 2, pad // 2 + 1, (pad, pad, pad // 2 + 1)
    D = torch.complex(*(torch.tensor(v, device=GPU).reshape(dims) for v in (re, im)))
    W = torch.tensor(w, device=GPU).reshape(dims).clone()
    k = torch.arange(-h, h + 1, device=GPU)
    r2 = k[:, None, None] ** 2 + k[None, :, None] ** 2 + k[None, None, h:] ** 2
    big = (2 * r_max) ** 2
    W *= r2 <= big
    D = D * (r2 <= big)
    rad = torch.sqrt(r2.double())
    if c["do_map"]:
        t = torch.tensor(tau2, device=GPU)[torch.floor(rad / 2 + 0.5).long().clamp(max=N // 2)]
        W = torch.where(r2 < big, W + 1 / (8 * t), W)
    shell = torch.floor(rad / 2).long()
    avg = torch.zeros(r_max, device=GPU, dtype=torch.float64)
    cnt = torch.zeros_like(avg)
    m = r2 < big
    avg.index_add_(0, shell[m], W[m])
    cnt.index_add_(0, shell[m], torch.ones_like(W[m]))
    W = torch.maximum(W, (avg / (1000 * cnt))[shell.clamp(max=r_max - 1)])
    D = torch.where(W != 0, D / W, D)
    P = 2 * N
    Ph = P // 2 + 1
    G = torch.zeros(P, P, Ph, device=GPU, dtype=torch.complex128)
    if Ph > xh:
        D = D * (r2 <= (xh - 1) ** 2)
        row = k % P
        G[row[:, None], row[None, :], :xh] = D
    else:
        q = torch.arange(P, device=GPU)
        row = torch.where(q < Ph, q, q - P) + h
        G = D[row[:, None], row[None, :], :Ph].clone()
    q = torch.arange(P, device=GPU)
    G *= 1 - 2 * ((q[:, None, None] + q[None, :, None] + q[None, None, :Ph]) & 1).double()
    for j in (0, P // 2):   # the half-complex transform's self-conjugate planes
        pl = G[:, :, j]
        G[:, :, j] = 0.5 * (pl + torch.conj(torch.roll(torch.flip(pl, (0, 1)), (1, 1), (0, 1))))
    vol = torch.fft.irfftn(G, s=(P, P, P), norm="forward")
    a = P // 2 - N // 2
    vol = vol[a:a + N, a:a + N, a:a + N].clone() / (8 * N)
    g = torch.arange(N, device=GPU, dtype=torch.float64) - N // 2
    r = torch.sqrt(g[:, None, None] ** 2 + g[None, :, None] ** 2 + g[None, None] ** 2)
    rc = 0.5 + 0.5 * torch.cos(math.pi * ((N / 2 + 3 - r) / 3).clamp(0, 1))
    rc = torch.where(r < N / 2, torch.zeros_like(rc), rc)
    bg = (rc * vol).sum() / rc.sum()
    vol = (1 - rc) * vol + rc * bg
    return vol / torch.sinc(r / (2 * N)) ** 2


def _exact_fsc(m1, m2):
    N = m1.shape[0]
    a, b = torch.fft.rfftn(m1), torch.fft.rfftn(m2)
    k = torch.arange(N, device=GPU)
    k = torch.where(k < N // 2 + 1, k, k - N).double()
    x = torch.arange(N // 2 + 1, device=GPU).double()
    shell = torch.floor(torch.sqrt(k[:, None, None] ** 2 + k[None, :, None] ** 2 + x[None, None] ** 2) + 0.5).long()
    m = shell <= N // 2
    num, d1, d2 = (torch.zeros(N // 2 + 1, device=GPU, dtype=torch.float64).index_add_(0, shell[m], v[m])
                   for v in ((a.conj() * b).real, a.abs() ** 2, b.abs() ** 2))
    return (num / torch.sqrt(d1 * d2)).cpu().numpy()


def _healpix_angles(order, x, y, face):
    """(rot, tilt) in degrees of the NEST pixel (x, y) of a base face (Gorski et al. 2005)."""
    nside = 1 << order
    jr = ((2, 2, 2, 2, 3, 3, 3, 3, 4, 4, 4, 4)[face] << order) - x - y - 1
    fact2 = 4.0 / (12 * nside * nside)
    shift = 0
    if jr < nside:
        nr, z = jr, 1.0 - jr * jr * fact2
    elif jr > 3 * nside:
        nr = 4 * nside - jr
        z = nr * nr * fact2 - 1.0
    else:
        nr, shift = nside, (jr - nside) & 1
        z = (2 * nside - jr) * (2 * nside * fact2)
    jp = ((1, 3, 5, 7, 0, 2, 4, 6, 1, 3, 5, 7)[face] * nr + x - y + 1 + shift) // 2
    jp = jp - 4 * nside if jp > 4 * nside else jp + 4 * nside if jp < 1 else jp
    phi = (jp - (shift + 1) * 0.5) * ((math.pi / 2.0) / nr)
    rot, tilt = phi * 180.0 / math.pi, math.acos(z) * 180.0 / math.pi
    return (rot - 360.0 if rot > 180.0 else rot), tilt


class ExactEstep:
    """The E-step in 64-bit torch: getFourierTransformsAndCtfs, both passes of getAllSquaredDifferences and
    convertAllSquaredDifferencesToWeights, storeWeightedSums and the backprojection."""

    def __init__(self, c, inp):
        self.c, self.inp, self.s = c, inp, inp["sizes"]
        s = self.s
        self.flat, self.K, self.n, self.over = c["ref_dim"] == 2, c["K"], c["n"], c["oversampling"]
        self.grids()
        dims = (s.pad, s.xdim) if self.flat else (s.pad, s.pad, s.xdim)
        self.vols = [torch.complex(re.double(), im.double()).reshape(dims) for re, im in inp["refs"]]
        self.og = torch.tensor(inp["p"]["optics"], device=GPU)
        self.sigma2 = torch.tensor(inp["sigma2"], device=GPU)
        self.scale = torch.tensor(inp["scale"], device=GPU)[torch.tensor(inp["p"]["group"], device=GPU)]
        self.old = torch.tensor(np.stack([inp["p"]["old_x"], inp["p"]["old_y"]], 1), device=GPU)
        # the offset prior's centre: 2D references have their classes', here 0; 3D the particle's
        self.prior_off = self.old.clone() if c["later"] and not self.flat else torch.zeros_like(self.old)
        self.first = self.table(s.first, False)
        self.second = self.table(s.current, False)
        self.store = self.table(s.current, True)
        self.preprocess()

    def grids(self):
        s, f = self.s, 1 << self.over
        sc = lambda d: (math.sin(d * math.pi / 180), math.cos(d * math.pi / 180))  # noqa: E731
        coarse, fine = [], []
        for pix in range(s.n_dir if not self.flat else 0):
            order = self.c["order"]
            face, q = pix >> (2 * order), pix & ((1 << (2 * order)) - 1)
            x = sum(((q >> (2 * b)) & 1) << b for b in range(order))
            y = sum(((q >> (2 * b + 1)) & 1) << b for b in range(order))
            coarse.append(_healpix_angles(order, x, y, face))
            fine.append([_healpix_angles(order + self.over, f * x + i, f * y + j, face)
                         for j in range(f) for i in range(f)])
        if self.flat:
            coarse, fine = [(0.0, 0.0)], [[(0.0, 0.0)]]
        step = 360.0 / s.n_psi
        psi = [i * step for i in range(s.n_psi)]
        sub = [[q - 0.5 * step + (0.5 + k) * step / f for k in range(f)] if f > 1 else [q] for q in psi]
        if self.flat and f > 1:
            sub = [[v - 360.0 if v > 180.0 else v for v in q] for q in sub]
        self.dir_deg, self.psi_deg = coarse, psi
        self.fine_deg, self.sub_psi = np.array(fine), np.array(sub)
        t = lambda v: torch.tensor(v, device=GPU, dtype=torch.float64)  # noqa: E731
        self.dir_sc, self.psi_sc = t([sc(a) + sc(b) for a, b in coarse]), t([sc(q) for q in psi])
        self.fine_sc = t([[sc(a) + sc(b) for a, b in d] for d in fine])
        self.sub_sc = t([[sc(q) for q in v] for v in sub])
        pix = self.c["pixel"]
        self.tx = t([x for x, _ in s.trans])
        self.ty = t([y for _, y in s.trans])
        off = [-0.5 * s.step + (0.5 + k) * s.step / f for k in range(f)] if f > 1 else [0.0]
        self.ftx = t([[(x + a) / pix for a in off for _ in off] for x, _ in s.trans])
        self.fty = t([[(y + b) / pix for _ in off for b in off] for _, y in s.trans])
        self.n_rot, self.n_tr = self.fine_sc.shape[1] * self.sub_sc.shape[1], len(off) ** 2

    def frames(self, d, q):
        """Projection frames of directions d and in-plane angles q (rows of sines and cosines): Euler matrix,
        its adjugate over the determinant, times the padding factor 2. Columns 0 and 1, as six arrays."""
        sa, ca, sb, cb = d.unbind(-1)
        sg, cg = q.unbind(-1)
        cc, cs, sc, ss = cb * ca, cb * sa, sb * ca, sb * sa
        A = [cg * cc - sg * sa, cg * cs + sg * ca, -cg * sb, -sg * cc - cg * sa, -sg * cs + cg * ca, sg * sb, sc, ss, cb]
        R = [A[8] * A[4] - A[7] * A[5], -(A[8] * A[1] - A[7] * A[2]), -(A[8] * A[3] - A[6] * A[5]),
             A[8] * A[0] - A[6] * A[2], A[7] * A[3] - A[6] * A[4], -(A[7] * A[0] - A[6] * A[1])]
        det = A[0] * R[0] + A[3] * R[1] + A[6] * (A[5] * A[1] - A[4] * A[2])
        # row-major inverse: (0,0), (0,1), (1,0), (1,1), (2,0), (2,1)
        return [(R[i] / det * 2.0)[..., None] for i in (0, 1, 2, 3, 4, 5)]

    def corners(self, f, x, y):
        """Corner indices, weights and the Friedel flip of the positions of pixels (x, y) in frames f."""
        s, h = self.s, self.s.pad // 2
        p = [f[0] * x + f[1] * y, f[2] * x + f[3] * y] + ([] if self.flat else [f[4] * x + f[5] * y])
        neg = p[0] < 0
        p = [torch.where(neg, -v, v) for v in p]
        lo = [torch.floor(v) for v in p]
        fr = [v - q for v, q in zip(p, lo)]
        i = [lo[0].long()] + [q.long() + h for q in lo[1:]]
        ok = (i[0] + 1 < s.xdim)
        for q in i[1:]:
            ok = ok & (q >= 0) & (q + 1 < s.pad)
        i = [q.clamp(0, m - 2) for q, m in zip(i, (s.xdim, s.pad, s.pad))]
        out = []
        for c in range(4 if self.flat else 8):
            b = [(c >> k) & 1 for k in range(3)]
            idx, w = i[1] + b[1], torch.ones_like(fr[0])
            if not self.flat:
                idx = (i[2] + b[2]) * s.pad + idx
            idx = idx * s.xdim + i[0] + b[0]
            for k, v in enumerate(fr):
                w = w * (v if b[k] else 1 - v)
            out.append((idx, w * ok))
        return out, neg

    def table(self, size, origin):
        x, y, shell, inside = _pixels(size, origin)
        if size < 2:
            raise ValueError("image size")
        t = dict(x=torch.tensor(x, device=GPU, dtype=torch.float64), y=torch.tensor(y, device=GPU, dtype=torch.float64),
                 shell=torch.tensor(shell, device=GPU), inside=torch.tensor(inside, device=GPU))
        t["minv"] = 1.0 / self.sigma2[:, t["shell"]]
        N = self.s.N
        t["ctf"] = _ctf(self.inp["p"], N, self.c["pixel"], t["x"], t["y"]) * self.scale[:, None]
        tx, ty = (self.tx / self.c["pixel"])[:, None], (self.ty / self.c["pixel"])[:, None]
        if size == self.s.first and not origin:
            a = -2 * math.pi / N * (tx[..., None] * t["x"] + ty[..., None] * t["y"])
            t["phase"] = torch.polar(torch.ones_like(a), a)[:, 0]
        return t

    def preprocess(self):
        c, s, p = self.c, self.s, self.inp["p"]
        N, xs = s.N, s.N // 2 + 1
        g = torch.arange(N, device=GPU)
        r = torch.sqrt(((g[:, None] - N // 2) ** 2 + (g[None] - N // 2) ** 2).double())
        rad = c["diameter"] / (2 * c["pixel"])
        rc = 0.5 + 0.5 * torch.cos(math.pi * ((rad + MASK_EDGE - r) / MASK_EDGE).clamp(0, 1))
        rc = torch.where(r < rad, torch.zeros_like(rc), rc)
        q = torch.arange(N, device=GPU)
        q = torch.where(q < xs, q, q - N)
        x = torch.arange(xs, device=GPU)
        shell = torch.floor(torch.sqrt((q[:, None] ** 2 + x[None] ** 2).double()) + 0.5).long()
        own = (shell > 0) & (shell < xs) & ~((x[None] == 0) & (q[:, None] < 0))
        wins = {k: ((t["y"].long() % N) * xs + t["x"].long(), 1 - 2 * ((t["x"] + t["y"]).long() & 1).double())
                for k, t in (("first", self.first), ("second", self.second), ("store", self.store))}
        parts = {k: [] for k in ("first", "second", "store", "raw", "power")}
        step = max(1, int(4e8 / (8 * N * N)))
        for b0 in range(0, self.n, step):
            i = slice(b0, min(self.n, b0 + step))
            img = self.inp["images"][i].double()
            if c["later"]:
                img = img / torch.tensor(p["norm"][i], device=GPU)[:, None, None]
                old = self.old[i].long()
                sy, sx = g[None] - old[:, 1:], g[None] - old[:, :1]
                ok = ((sy >= 0) & (sy < N))[:, :, None] & ((sx >= 0) & (sx < N))[:, None, :]
                b = torch.arange(len(img), device=GPU)[:, None, None]
                img = img[b, sy.clamp(0, N - 1)[:, :, None], sx.clamp(0, N - 1)[:, None, :]] * ok
            raw = torch.fft.rfft2(img).reshape(len(img), -1) / N ** 2
            bg = (rc * img).sum((1, 2), keepdim=True) / rc.sum()
            F = torch.fft.rfft2((1 - rc) * img + rc * bg).reshape(len(img), -1) / N ** 2
            for k, (w, sign) in wins.items():
                parts[k].append(F[:, w] * sign)
            parts["raw"].append(raw[:, wins["store"][0]] * wins["store"][1])
            m = own.reshape(-1).nonzero()[:, 0]
            parts["power"].append(torch.zeros(len(img), xs, device=GPU, dtype=torch.float64).index_add_(
                1, shell.reshape(-1)[m], F[:, m].abs() ** 2))
        self.X = {k: torch.cat(v) for k, v in parts.items()}
        if s.current == N:
            self.X["power"].zero_()
        self.high = self.X["power"][:, s.current // 2 + 1:].sum(1)

    def sample(self, vol, f, t):
        """Slices of a reference in frames f at the pixels of table t: [m][P]."""
        v = torch.zeros(f[0].shape[:-1] + t["x"].shape, device=GPU, dtype=torch.complex128)
        at, neg = self.corners(f, t["x"], t["y"])
        flat = self.vols[vol].reshape(-1)
        for idx, w in at:
            v += flat[idx] * w
        return torch.where(neg, v.conj(), v) * t["inside"]

    def translation_prior(self):
        pix2 = self.c["pixel"] ** 2
        dx = self.old[:, :1] + self.tx - self.prior_off[:, :1]
        dy = self.old[:, 1:] + self.ty - self.prior_off[:, 1:]
        v = torch.exp((dx * dx + dy * dy) * pix2 / (-2 * SIGMA2_OFFSET)) / (2 * math.pi * SIGMA2_OFFSET)
        return v / v.mean(1, keepdim=True)

    def walk(self, w, total):
        """The significance walk over one particle's candidate weights: (threshold, count)."""
        v = torch.sort(w, descending=True).values
        over = torch.cumsum(v, 0) > ADAPTIVE_FRACTION * total
        k = int(over.nonzero()[0, 0]) if bool(over.any()) else len(v) - 1
        return v[k], k + 1

    def global_pairs(self):
        """First pass of a global search: significant (particle, orientation, translation), their priors."""
        s, t = self.s, self.first
        Norient = s.n_dir * s.n_psi
        O, nt, P = self.K * Norient, len(s.trans), len(t["x"])
        F = torch.empty(O, P, device=GPU, dtype=torch.complex128)
        d = torch.arange(Norient, device=GPU) // s.n_psi
        q = torch.arange(Norient, device=GPU) % s.n_psi
        step = max(1, int(2e7 / P))
        for k in range(self.K):
            for o0 in range(0, Norient, step):
                i = slice(o0, min(Norient, o0 + step))
                F[k * Norient + i.start:k * Norient + i.stop] = self.sample(
                    k, self.frames(self.dir_sc[d[i]], self.psi_sc[q[i]]), t)
        F2 = (F.abs() ** 2).T.contiguous()
        F = torch.view_as_real(F).reshape(O, 2 * P)
        pd = torch.tensor(self.inp["pdf_dir"], device=GPU)
        prior_o = (pd / pd.mean()).repeat_interleave(s.n_psi, 1).reshape(-1)
        prior_t = self.translation_prior()
        found, self.n_sig, self.first_pass = [], np.zeros(self.n, np.int64), []
        step = max(1, int(1.5e9 / (8 * O * nt)))
        for b0 in range(0, self.n, step):
            i = slice(b0, min(self.n, b0 + step))
            X, ctf, mv = self.X["first"][i], t["ctf"][i], t["minv"][self.og[i]]
            m = len(X)
            A = ((mv * ctf * X)[:, None] * t["phase"]).reshape(m * nt, P)
            d2 = (torch.view_as_real(A).reshape(m * nt, 2 * P) @ F.T).reshape(m, nt, O).neg_()
            d2 += ((0.5 * mv * ctf * ctf) @ F2)[:, None]
            C0 = self.high[i] / 2 + 0.5 * (mv * X.abs() ** 2).sum(1)
            d2 += C0[:, None, None]
            low = d2.amin((1, 2))
            d2 -= low[:, None, None]
            keep = d2 if self.over == 0 else None
            w = torch.where(d2 > 700, torch.zeros_like(d2), torch.exp(-d2))
            w *= prior_o
            w *= prior_t[i][:, :, None]
            total = w.sum((1, 2))
            for b in range(m):
                e = (w[b] > (1 - ADAPTIVE_FRACTION) * total[b] / (O * nt)).nonzero()
                v = w[b][e[:, 0], e[:, 1]]
                thr, k = self.walk(v, total[b])
                e = e[v >= thr]
                self.n_sig[b0 + b] = k
                pr = prior_o[e[:, 1]] * prior_t[b0 + b][e[:, 0]]
                dd = keep[b][e[:, 0], e[:, 1]] if keep is not None else torch.zeros_like(pr)
                found.append((torch.full_like(e[:, 0], b0 + b), e[:, 1], e[:, 0], pr, dd))
                self.first_pass.append((low[b], total[b], thr))
        return [torch.cat(v) for v in zip(*found)]

    def local_pairs(self):
        """First pass of a local search, particle by particle over its orientations in range."""
        s, t, c = self.s, self.first, self.c
        dirs = torch.stack([self.dir_sc[:, 2] * self.dir_sc[:, 1], self.dir_sc[:, 2] * self.dir_sc[:, 0],
                            self.dir_sc[:, 3]], 1)
        psi = torch.tensor(self.psi_deg, device=GPU)
        prior_t, p, sig = self.translation_prior(), self.inp["p"], c["sigma_ang"]
        nt, P, Norient = len(s.trans), len(t["x"]), s.n_dir * s.n_psi
        ph = torch.view_as_real(t["phase"]).reshape(nt, 2 * P).T.contiguous()

        def gauss(diff):
            w = torch.where(diff < 3 * sig, torch.exp(-0.5 * (diff / sig) ** 2), torch.zeros_like(diff))
            if not bool((w > 0).any()):
                w[diff.argmin()] = 1.0
            return w / w.sum()

        found, self.n_sig, self.first_pass = [], np.zeros(self.n, np.int64), []
        for b in range(self.n):
            a, e = math.radians(p["prior_rot"][b]), math.radians(p["prior_tilt"][b])
            v = torch.tensor([math.sin(e) * math.cos(a), math.sin(e) * math.sin(a), math.cos(e)], device=GPU,
                             dtype=torch.float64)
            wd = gauss(torch.rad2deg(torch.acos((dirs * v).sum(1).clamp(-1, 1))))
            dp = (psi - p["prior_psi"][b]).abs()
            wp = gauss(torch.where(dp > 180, (dp - 360).abs(), dp))
            d, q = (wd > 0).nonzero()[:, 0], (wp > 0).nonzero()[:, 0]
            po = (wd[d][:, None] * wp[q][None]).reshape(-1)
            po = po / po.mean()
            dd, qq = d.repeat_interleave(len(q)), q.repeat(len(d))
            f = self.frames(self.dir_sc[dd], self.psi_sc[qq])
            X, ctf, mv = self.X["first"][b], t["ctf"][b], t["minv"][self.og[b]]
            rows = []
            step = max(1, int(2e7 / P))
            C0 = self.high[b] / 2 + 0.5 * (mv * X.abs() ** 2).sum()
            for k in range(self.K):
                for o0 in range(0, len(dd), step):
                    F = self.sample(k, [u[o0:o0 + step] for u in f], t)
                    Z = F * (mv * ctf * X.conj())
                    rows.append(C0 + (0.5 * mv * ctf * ctf * F.abs() ** 2).sum(1)[:, None]
                                - torch.view_as_real(Z).reshape(len(Z), 2 * P) @ ph)
            d2 = torch.cat(rows)
            prior = po.repeat(self.K)[:, None] * prior_t[b]
            low = d2.min()
            w = torch.where(d2 - low > 700, torch.zeros_like(d2), prior * torch.exp(low - d2))
            thr, self.n_sig[b] = self.walk(w[w > 0], w.sum())
            e = (w >= thr).nonzero()
            o = (dd * s.n_psi + qq).repeat(self.K) + torch.arange(self.K, device=GPU).repeat_interleave(len(dd)) * Norient
            found.append((torch.full_like(e[:, 0], b), o[e[:, 0]], e[:, 1], prior[e[:, 0], e[:, 1]],
                          torch.zeros(len(e), device=GPU, dtype=torch.float64)))
            self.first_pass.append((low, w.sum(), thr))
        return [torch.cat(v) for v in zip(*found)]

    def fine_frames(self, o):
        """Frames of the oversampled rotations of orientations o: six [m][rot][1], and their classes."""
        s = self.s
        Norient = s.n_dir * s.n_psi
        d, q = (o % Norient) // s.n_psi, o % s.n_psi
        nd, nq = self.fine_sc.shape[1], self.sub_sc.shape[1]
        D = self.fine_sc[d][:, :, None].expand(-1, -1, nq, -1).reshape(len(o), nd * nq, 4)
        Q = self.sub_sc[q][:, None].expand(-1, nd, -1, -1).reshape(len(o), nd * nq, 2)
        return self.frames(D, Q), o // Norient

    def slices(self, o, t):
        f, cls = self.fine_frames(o)
        F = torch.empty(len(o), self.n_rot, len(t["x"]), device=GPU, dtype=torch.complex128)
        for k in torch.unique(cls).tolist():
            m = (cls == k).nonzero()[:, 0]
            F[m] = self.sample(k, [u[m] for u in f], t)
        return F

    def phases(self, tr, t):
        a = -2 * math.pi / self.s.N * (self.ftx[tr][..., None] * t["x"] + self.fty[tr][..., None] * t["y"])
        return torch.polar(torch.ones_like(a), a)

    def result(self):
        c, s, n = self.c, self.s, self.n
        b, o, tr, prior, d2c = self.local_pairs() if c["sigma_ang"] else self.global_pairs()
        R, Q = self.n_rot, self.n_tr
        m, t = len(b), self.second
        step = max(1, int(4e7 / (R * len(t["x"]))))
        if m * R * len(t["x"]) > 2e9:   # so many significant samples that torch would take longer than 20 s
            return None
        f64 = lambda *shape: torch.zeros(*shape, device=GPU, dtype=torch.float64)  # noqa: E731
        if self.over == 0:   # one pass: its own weights
            low, total, thr = (torch.stack(v) for v in zip(*self.first_pass))
            w = (prior * torch.exp(-d2c))[:, None, None]
        else:
            d2 = f64(m, R, Q)
            for e0 in range(0, m, step):
                i = slice(e0, min(m, e0 + step))
                X, ctf, mv = self.X["second"][b[i]], t["ctf"][b[i]], t["minv"][self.og[b[i]]]
                F = self.slices(o[i], t)
                Z = torch.view_as_real(F * (mv * ctf * X.conj())[:, None]).reshape(len(X), R, -1)
                ph = torch.view_as_real(self.phases(tr[i], t)).reshape(len(X), Q, -1).transpose(1, 2).contiguous()
                base = self.high[b[i]] / 2 + 0.5 * (mv * X.abs() ** 2).sum(1)
                n1 = torch.bmm(F.abs() ** 2, (0.5 * mv * ctf * ctf)[..., None])
                d2[i] = base[:, None, None] + n1 - torch.bmm(Z, ph)
            low = torch.full((n,), math.inf, device=GPU, dtype=torch.float64).scatter_reduce_(
                0, b, d2.amin((1, 2)), "amin")
            dd = d2 - low[b][:, None, None]
            w = torch.where(dd > 700, torch.zeros_like(dd), prior[:, None, None] * torch.exp(-dd))
            total = f64(n).index_add_(0, b, w.sum((1, 2)))
            thr = f64(n)
            start = torch.searchsorted(b, torch.arange(n + 1, device=GPU)).tolist()
            for k in range(n):
                v = w[start[k]:start[k + 1]].reshape(-1)
                thr[k] = self.walk(v[v > 0], total[k])[0]
        sig = w >= thr[b][:, None, None]
        wn = torch.where(sig, w / total[b][:, None, None], torch.zeros_like(w))
        out, best = self.poses(b, o, tr, wn)
        sums, norm, bp = self.sums(b, o, tr, wn)
        p = self.inp["p"]
        shells = self.store["shell"]
        ls = torch.log(2 * math.pi * self.sigma2[:, shells[shells > 0]]).sum(1)
        dLL = torch.log(total) - low - ls[self.og]
        nc = torch.tensor(p["norm"], device=GPU)
        if c["later"]:
            nc = nc * torch.sqrt(norm * 2)
            sums["avg_norm_correction"][0] = nc.sum()
        sums["LL"][0], sums["ave_Pmax"][0] = dLL.sum(), best.sum()
        count = lambda v: torch.zeros(n, device=GPU, dtype=torch.int64).index_add_(0, b, v)  # noqa: E731
        out.update(pmax=best, dLL=dLL, norm_correction=nc, sum_weight=total, min_diff2=low,
                   nr_significant_coarse=torch.tensor(self.n_sig),
                   nr_fine_samples=count(torch.full_like(b, R * Q)), nr_fine_significant=count(sig.sum((1, 2))))
        host = lambda d: {k: v.cpu().numpy() for k, v in d.items()}  # noqa: E731
        # the significant weight is the one sample's at which the walk stops: it jumps where another sample is it
        return dict(particles=dict(host(out), significant_weight=None), sums=host(sums), bp_re=bp[..., 0].cpu().numpy(), bp_im=bp[..., 1].cpu().numpy(),
                    bp_weight=bp[..., 2].cpu().numpy())

    def poses(self, b, o, tr, wn):
        """The most probable sample of each particle."""
        R, Q, n, s = self.n_rot, self.n_tr, self.n, self.s
        flat = wn.reshape(len(b), R * Q)
        v, k = flat.max(1)
        best = torch.zeros(n, device=GPU, dtype=torch.float64).scatter_reduce_(0, b, v, "amax")
        at = torch.full((n,), len(b), device=GPU).scatter_reduce_(
            0, b, torch.where(v == best[b], torch.arange(len(b), device=GPU), len(b)), "amin")
        o, tr, k = o[at], tr[at], k[at]
        Norient = s.n_dir * s.n_psi
        d, q = ((o % Norient) // s.n_psi).cpu().numpy(), (o % s.n_psi).cpu().numpy()
        ir, it = (k // Q).cpu().numpy(), k % Q
        nq = self.sub_sc.shape[1]
        rt = self.fine_deg.reshape(len(self.fine_deg), -1, 2)[d, ir // nq]
        out = dict(rot=torch.tensor(rt[:, 0]), tilt=torch.tensor(rt[:, 1]), psi=torch.tensor(self.sub_psi[q, ir % nq]),
                   xoff=self.old[:, 0] + self.ftx[tr, it], yoff=self.old[:, 1] + self.fty[tr, it],
                   iclass=o // Norient + 1, best_hidden=(o * len(s.trans) + tr) * R * Q + k)
        return out, best

    def sums(self, b, o, tr, wn):
        """storeWeightedSums and the backprojection of the samples with weights wn."""
        c, s, n, K, t = self.c, self.s, self.n, self.K, self.store
        R, Q, pix, xs = self.n_rot, self.n_tr, c["pixel"], s.N // 2 + 1
        Norient, n_og, n_grp = s.n_dir * s.n_psi, self.inp["n_og"], len(self.inp["scale"])
        f64 = lambda *shape: torch.zeros(*shape, device=GPU, dtype=torch.float64)  # noqa: E731
        sigma, norm, xa, aa = f64(n_og * xs), f64(n), f64(n_grp), f64(n_grp)
        bp = f64(K * s.n_voxels, 3)
        grp = torch.tensor(self.inp["p"]["group"], device=GPU)
        dvp = torch.tensor(self.inp["dvp"], device=GPU) > 3
        cls = o // Norient
        live = (wn.sum(2) > 0).nonzero()   # (pair, rotation) with a significant sample
        step = max(1, int(2e7 / len(t["x"])))
        lim = (2 * s.r_max) ** 2
        for e0 in range(0, len(live), step):
            i, r = live[e0:e0 + step].unbind(1)
            w, pb, oo = wn[i, r], b[i], o[i]
            X, raw, ctf, mv = self.X["store"][pb], self.X["raw"][pb], t["ctf"][pb], t["minv"][self.og[pb]]
            f, k = self.fine_frames(oo)
            f = [u[torch.arange(len(i), device=GPU), r] for u in f]
            F = torch.empty(len(i), len(t["x"]), device=GPU, dtype=torch.complex128)
            for q in torch.unique(k).tolist():
                g = (k == q).nonzero()[:, 0]
                F[g] = self.sample(q, [u[g] for u in f], t)
            F *= ctf
            ph = (self.phases(tr[i], t) * w[..., None]).sum(1)     # sum of w exp over the translations
            ws = w.sum(1)[:, None]
            cross = (F * (X * ph).conj()).real
            wd = ws * (F.abs() ** 2 + X.abs() ** 2) - 2 * cross
            sigma.index_add_(0, (self.og[pb][:, None] * xs + t["shell"]).reshape(-1), wd.reshape(-1))
            norm.index_add_(0, pb, wd.sum(1))
            if c["later"]:
                on = dvp[k][:, t["shell"]]
                sc = self.scale[pb]
                xa.index_add_(0, grp[pb], (cross * on).sum(1) / sc)
                aa.index_add_(0, grp[pb], (ws * F.abs() ** 2 * on).sum(1) / sc ** 2)
            # pixels inside the insertion radius, in the reference's order of operations
            xx, xy = f[0] * f[0] + f[2] * f[2], f[0] * f[1] + f[2] * f[3]
            yy = f[1] * f[1] + f[3] * f[3]
            if not self.flat:
                xx, xy, yy = xx + f[4] * f[4], xy + f[4] * f[5], yy + f[5] * f[5]
            y, x = t["y"], t["x"]
            disc = xy * xy * y * y - xx * (yy * y * y - lim)
            dd, qq = torch.sqrt(disc.clamp(min=0)) / xx, -xy * y / xx
            ok = (disc >= 0) & (x >= torch.ceil(qq - dd)) & (x <= torch.floor(qq + dd))
            if not self.flat:
                px, py, pz = f[0] * x + f[1] * y, f[2] * x + f[3] * y, f[4] * x + f[5] * y
                ok &= px * px + py * py + pz * pz <= lim
            at, neg = self.corners(f, x, y)
            val = raw * ph * (ctf * mv)
            val = torch.where(neg, val.conj(), val)
            v3 = torch.stack([val.real, val.imag, ws * ctf * ctf * mv], -1) * ok[..., None]
            for idx, cw in at:
                bp.index_add_(0, (k[:, None] * s.n_voxels + idx).reshape(-1), (v3 * cw[..., None]).reshape(-1, 3))
        hi = s.current // 2 + 1
        power = f64(n_og, xs).index_add_(0, self.og, self.X["power"])
        power[:, :hi] = 0
        norm += self.high
        per, pq = wn.sum((1, 2)), wn.sum(1)
        ox = self.old[b][:, :1] + self.ftx[tr]
        oy = self.old[b][:, 1:] + self.fty[tr]
        dx, dy = self.prior_off[b][:, :1] - ox, self.prior_off[b][:, 1:] - oy
        off = f64(2 * K)
        if self.flat:
            off.index_add_(0, 2 * cls, pix * (pq * ox).sum(1))
            off.index_add_(0, 2 * cls + 1, pix * (pq * oy).sum(1))
        sums = dict(sigma2_noise=sigma + power.reshape(-1), sumw_group=f64(n_og).index_add_(0, self.og[b], per),
                    pdf_class=f64(K).index_add_(0, cls, per),
                    pdf_direction=f64(K * s.n_dir).index_add_(0, cls * s.n_dir + (o % Norient) // s.n_psi, per),
                    prior_offset_class=off, sigma2_offset=(pix * pix * pq * (dx * dx + dy * dy)).sum()[None],
                    avg_norm_correction=f64(1), LL=f64(1), ave_Pmax=f64(1), wsum_signal_product=xa,
                    wsum_reference_power=aa)
        return sums, norm, bp.reshape(K, s.n_voxels, 3)
