// t2x_recon.hip — BackProjector::reconstruct (default skip_gridding branch) and getFSC on the
// GPU, all arithmetic in FP64 (backprojector.cpp:1344-1770, :2486-2600; fftw.cpp:481-523).
//
// Data flow for one class: the projector-layout data/weight volumes are uploaded once; one
// kernel per FFTW-layout voxel of the padded transform decentres, adds the MAP term and
// accumulates the per-shell weight sums (LDS partials per block, then the blocks summed in a
// fixed order; the partials' LDS atomics may reorder additions within a block, so the floor
// can differ in the last bits between runs); a second kernel writes the 2*ori-sized half-complex grid directly —
// division by max(weight, floor), Fourier window, CenterFFTbySign and Hermitian symmetrisation of
// the x = 0 / Nyquist planes fused per output voxel — followed by one hipFFT Z2D, a real-space
// window with the FFT normalisation, the soft spherical mask and the trilinear gridding
// correction. Volumes: 512^3 doubles for a 256 box (1 GiB each) fit easily in HBM.
#include "t2x_internal.h"

#include <hipfft/hipfft.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace t2x {

namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr int kShellBlocks = 256;   // partial-sum blocks of the shell reductions

__host__ __device__ inline long long fftw_logical(long long k, long long xsize, long long zdim)
{
    return k < xsize ? k : k - zdim;
}
__host__ __device__ inline long long wrapi(long long k, long long n) { return k < 0 ? k + n : k; }

struct ReconGeom {
    long long pad, xh, P, Ph, ori;
    double pf;
    long long max_r2, round_max_r2, win_r2;
    int r_max, do_map, minres_map;
    double tau2_fudge, normfft;
};

// decenter + MAP term: weights of the pad^3 FFTW-layout grid, and per-shell partial sums
// (shell = FLOOR(|k| / pf) over |k|^2 < round_max_r2) of the final weights.
__global__ void k_recon_weights(ReconGeom g, const double* __restrict__ w_in, const double* __restrict__ tau2,
                                double* __restrict__ Fw, double* __restrict__ part_sum, double* __restrict__ part_cnt,
                                int* err)
{
    extern __shared__ double sh[];
    double* ssum = sh;
    double* scnt = sh + g.r_max;
    for (int s = threadIdx.x; s < g.r_max; s += blockDim.x) { ssum[s] = 0.; scnt[s] = 0.; }
    __syncthreads();
    const long long nv = g.pad * g.pad * g.xh;
    const long long c0 = g.pad / 2;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < nv; e += (long long)gridDim.x * blockDim.x) {
        const long long j = e % g.xh, i = (e / g.xh) % g.pad, k = e / (g.xh * g.pad);
        const long long kp = fftw_logical(k, g.xh, g.pad), ip = fftw_logical(i, g.xh, g.pad), jp = j;
        const long long r2 = kp * kp + ip * ip + jp * jp;
        double w = 0.;
        if (r2 <= g.max_r2) w = w_in[((kp + c0) * g.pad + (ip + c0)) * g.xh + jp];
        if (g.do_map && r2 < g.max_r2) {
            const long long ires = llround(sqrt((double)r2) / g.pf);
            const double t = tau2[ires];
            double invtau2;
            if (t > 0.) invtau2 = 1. / (g.pf * g.pf * g.pf * g.tau2_fudge * t);
            else if (t < 1e-20) invtau2 = (w > 1e-20) ? 1. / (0.001 * w) : 0.;
            else { *err = 2; invtau2 = 0.; }
            if (ires >= g.minres_map) w = w + invtau2;
        }
        Fw[e] = w;
        if (r2 < g.round_max_r2) {
            const long long ires = (long long)floor(sqrt((double)r2) / g.pf);
            if (ires >= g.r_max) { *err = 3; continue; }
            atomicAdd(&ssum[ires], w);   // LDS partial: order within the block only
            atomicAdd(&scnt[ires], 1.);
        }
    }
    __syncthreads();
    for (int s = threadIdx.x; s < g.r_max; s += blockDim.x) {
        part_sum[(size_t)blockIdx.x * g.r_max + s] = ssum[s];
        part_cnt[(size_t)blockIdx.x * g.r_max + s] = scnt[s];
    }
}

// floor[s] = (sum over blocks in order) / (1000 * count)
__global__ void k_recon_floor(ReconGeom g, const double* part_sum, const double* part_cnt, int nblocks,
                              double* floorv, int* err)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.r_max) return;
    double a = 0., c = 0.;
    for (int b = 0; b < nblocks; b++) {
        a += part_sum[(size_t)b * g.r_max + s];
        c += part_cnt[(size_t)b * g.r_max + s];
    }
    if (c > 0. || a > 0.) floorv[s] = a / (1000. * c);
    else { floorv[s] = 0.; *err = 4; }
}

// data/weight at FFTW logical (kp, ip, jp) of the padded grid (0 outside it)
__device__ inline double2 recon_value(const ReconGeom& g, long long kp, long long ip, long long jp,
                                      const double* __restrict__ d_re, const double* __restrict__ d_im,
                                      const double* __restrict__ Fw, const double* __restrict__ floorv)
{
    const long long half = g.pad / 2;
    if (jp >= g.xh || kp > half || kp < -half || ip > half || ip < -half) return make_double2(0., 0.);
    const long long r2 = kp * kp + ip * ip + jp * jp;
    const long long e = (wrapi(kp, g.pad) * g.pad + wrapi(ip, g.pad)) * g.xh + jp;
    double re = 0., im = 0.;
    if (r2 <= g.max_r2) {
        const long long c0 = g.pad / 2;
        const long long src = ((kp + c0) * g.pad + (ip + c0)) * g.xh + jp;
        re = d_re[src];
        im = d_im[src];
    }
    const long long ires = (long long)floor(sqrt((double)r2) / g.pf);
    const double w = fmax(Fw[e], floorv[(ires < g.r_max) ? ires : (g.r_max - 1)]);
    if (w != 0.) { re /= w; im /= w; }
    return make_double2(re, im);
}

// 2*ori half-complex grid: window, CenterFFTbySign, Hermitian x = 0 / Nyquist planes
__global__ void k_recon_window(ReconGeom g, const double* __restrict__ d_re, const double* __restrict__ d_im,
                               const double* __restrict__ Fw, const double* __restrict__ floorv,
                               double2* __restrict__ W)
{
    const long long n = g.P * g.P * g.Ph;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x) {
        const long long j = e % g.Ph, i = (e / g.Ph) % g.P, k = e / (g.Ph * g.P);
        const long long kp = fftw_logical(k, g.Ph, g.P), ip = fftw_logical(i, g.Ph, g.P), jp = j;
        auto at = [&](long long a, long long b, long long c) -> double2 {
            if (g.Ph > g.xh) {   // zero-padding window: keep |k|^2 <= (XSIZE(in)-1)^2
                if (a * a + b * b + c * c > g.win_r2) return make_double2(0., 0.);
            }
            return recon_value(g, a, b, c, d_re, d_im, Fw, floorv);
        };
        double2 v = at(kp, ip, jp);
        if (jp == 0 || jp == g.P / 2) {
            // partner (-kp, -ip): logical index of the mirrored direct index (P-k)%P, (P-i)%P
            const long long k2 = (g.P - k) % g.P, i2 = (g.P - i) % g.P;
            const double2 u = at(fftw_logical(k2, g.Ph, g.P), fftw_logical(i2, g.Ph, g.P), jp);
            v = make_double2(0.5 * (v.x + u.x), 0.5 * (v.y - u.y));
        }
        if (((k ^ i ^ j) & 1) != 0) { v.x = -v.x; v.y = -v.y; }
        W[e] = v;
    }
}

// real-space window (Xmipp origins P/2 and ori/2) with the FFT normalisation, and the partial
// sums of the soft-mask background (r >= ori/2) per block
__global__ void k_recon_crop(ReconGeom g, const double* __restrict__ R, double* __restrict__ vol,
                             double* __restrict__ part_bg, double* __restrict__ part_w)
{
    const long long n = g.ori * g.ori * g.ori;
    const long long oP = g.P / 2, oO = g.ori / 2;
    const double radius = (double)g.ori / 2., radius_p = radius + 3.;
    double sbg = 0., sw = 0.;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x) {
        const long long x = e % g.ori, y = (e / g.ori) % g.ori, z = e / (g.ori * g.ori);
        const double v = R[((z - oO + oP) * g.P + (y - oO + oP)) * g.P + (x - oO + oP)] / g.normfft;
        vol[e] = v;
        const long long kk = z - oO, ii = y - oO, jj = x - oO;
        const double r = sqrt((double)(kk * kk + ii * ii + jj * jj));
        if (r < radius) continue;
        if (r > radius_p) { sw += 1.; sbg += v; }
        else {
            const double rc = 0.5 + 0.5 * cos(kPi * (radius_p - r) / 3.);
            sw += rc;
            sbg += rc * v;
        }
    }
    __shared__ double rb[1024], rw[1024];
    rb[threadIdx.x] = sbg;
    rw[threadIdx.x] = sw;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) { rb[threadIdx.x] += rb[threadIdx.x + s]; rw[threadIdx.x] += rw[threadIdx.x + s]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) { part_bg[blockIdx.x] = rb[0]; part_w[blockIdx.x] = rw[0]; }
}

// soft mask with the background average, then the trilinear gridding correction
__global__ void k_recon_finish(ReconGeom g, const double* part_bg, const double* part_w, int nblocks,
                               double* __restrict__ vol)
{
    __shared__ double bg;
    if (threadIdx.x == 0) {
        double a = 0., c = 0.;
        for (int b = 0; b < nblocks; b++) { a += part_bg[b]; c += part_w[b]; }
        bg = a / c;
    }
    __syncthreads();
    const long long n = g.ori * g.ori * g.ori;
    const long long oO = g.ori / 2;
    const double radius = (double)g.ori / 2., radius_p = radius + 3.;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x) {
        const long long x = e % g.ori, y = (e / g.ori) % g.ori, z = e / (g.ori * g.ori);
        const long long kk = z - oO, ii = y - oO, jj = x - oO;
        const double r = sqrt((double)(kk * kk + ii * ii + jj * jj));
        double v = vol[e];
        if (r >= radius) {
            if (r > radius_p) v = bg;
            else {
                const double rc = 0.5 + 0.5 * cos(kPi * (radius_p - r) / 3.);
                v = (1 - rc) * v + rc * bg;
            }
        }
        if (r > 0.) {
            const double rval = r / ((double)g.ori * g.pf);
            const double sinc = sin(kPi * rval) / (kPi * rval);
            v /= sinc * sinc;
        }
        vol[e] = v;
    }
}

// FSC partial sums per block and shell (shell = ROUND(|k|) < n/2+1), forward transforms / size
__global__ void k_fsc_partial(long long n, const double2* __restrict__ A, const double2* __restrict__ B,
                              double* __restrict__ part)   // [blocks][3][xh]
{
    extern __shared__ double sh[];
    const long long xh = n / 2 + 1;
    for (long long s = threadIdx.x; s < 3 * xh; s += blockDim.x) sh[s] = 0.;
    __syncthreads();
    const double scale = 1.0 / ((double)n * n * n);
    const long long tot = n * n * xh;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < tot; e += (long long)gridDim.x * blockDim.x) {
        const long long j = e % xh, i = (e / xh) % n, k = e / (xh * n);
        const long long kp = fftw_logical(k, xh, n), ip = fftw_logical(i, xh, n), jp = j;
        const long long idx = llround(sqrt((double)(kp * kp + ip * ip + jp * jp)));
        if (idx >= xh) continue;
        const double2 a = A[e], b = B[e];
        const double ar = a.x * scale, ai = a.y * scale, br = b.x * scale, bi = b.y * scale;
        atomicAdd(&sh[idx], ar * br + ai * bi);
        atomicAdd(&sh[xh + idx], ar * ar + ai * ai);
        atomicAdd(&sh[2 * xh + idx], br * br + bi * bi);
    }
    __syncthreads();
    for (long long s = threadIdx.x; s < 3 * xh; s += blockDim.x) part[(size_t)blockIdx.x * 3 * xh + s] = sh[s];
}

__global__ void k_fsc_final(long long n, const double* part, int nblocks, double* fsc)
{
    const long long xh = n / 2 + 1;
    const long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= xh) return;
    double num = 0., d1 = 0., d2 = 0.;
    for (int b = 0; b < nblocks; b++) {
        num += part[(size_t)b * 3 * xh + s];
        d1 += part[(size_t)b * 3 * xh + xh + s];
        d2 += part[(size_t)b * 3 * xh + 2 * xh + s];
    }
    fsc[s] = num / sqrt(d1 * d2);
}

// The device backprojector's FP32 complex data and weight (projector layout, as accumulated by the
// E-step) widened to the FP64 inputs of the reconstruction: the same values the host path reads
// back into BackProjector::data and ::weight.
__global__ void k_bp_widen(size_t n, const float2* __restrict__ d, const float* __restrict__ w,
                           double* __restrict__ re, double* __restrict__ im, double* __restrict__ wo)
{
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (size_t)gridDim.x * blockDim.x) {
        const float2 v = d[e];
        re[e] = v.x;
        im[e] = v.y;
        wo[e] = w[e];
    }
}

// The kept arena is given back after a call that needed more (a 256 box takes 4 GiB).
constexpr size_t kReconKeep = (size_t)8 << 30;

// Places of one call's buffers in the arena.
struct Arena {
    size_t bytes = 0;
    size_t take(size_t n) { const size_t o = bytes; bytes += (n + 255) / 256 * 256; return o; }
};

// The end of a call, on every way out: its copies are over (a caller's page-locked arrays are read and
// written by the device directly), and an arena that is too large to keep is given back.
struct ArenaRelease {
    ReconWork& w;
    hipStream_t st;
    ~ArenaRelease()
    {
        (void)hipStreamSynchronize(st);
        if (w.arena.bytes > kReconKeep) w.arena.release();
    }
};

// A piece of a transfer between the caller's pageable memory and the device.
struct Piece {
    char* dev;
    char* host;
    size_t bytes;
};

// Copies pieces of up to kPiece bytes between pageable host memory and the device, on the stream, through
// page-locked slots filled or emptied by several threads: a transfer from pageable memory passes the
// driver's staging buffer in one thread (25 GB/s of the link's 57). Small totals and memory the runtime
// knows (page-locked, device) go the plain way. To the device: the copies are queued on return, their
// slots reused in stream order; to the host: complete on return.
constexpr size_t kPiece = (size_t)4 << 20, kStagedMin = (size_t)16 << 20;
constexpr int kCopyThreads = 8;

int staged_copy(Device* d, const std::vector<Piece>& whole, bool to_device)
{
    hipStream_t st = d->stream;
    size_t total = 0;
    bool known = false;
    for (const Piece& w : whole) {
        total += w.bytes;
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, w.host) == hipSuccess) known |= at.type != hipMemoryTypeUnregistered;
        else (void)hipGetLastError();
    }
    if (total < kStagedMin || known || d->recon.host.ensure(kPiece * 2 * kCopyThreads) != T2X_OK) {
        for (const Piece& w : whole) {
            if (to_device) T2X_HIP(hipMemcpyAsync(w.dev, w.host, w.bytes, hipMemcpyHostToDevice, st));
            else T2X_HIP(hipMemcpyAsync(w.host, w.dev, w.bytes, hipMemcpyDeviceToHost, st));
        }
        if (!to_device) T2X_HIP(hipStreamSynchronize(st));
        return T2X_OK;
    }
    std::vector<Piece> pieces;
    for (const Piece& w : whole)
        for (size_t o = 0; o < w.bytes; o += kPiece) pieces.push_back({w.dev + o, w.host + o, std::min(kPiece, w.bytes - o)});
    T2X_HIP(hipStreamSynchronize(st));   // the slots' last use
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&](int t) {
        hipError_t e = hipSetDevice(d->id);
        hipEvent_t ev[2] = {nullptr, nullptr};
        for (hipEvent_t& x : ev)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&x, hipEventDisableTiming);
        char* slot[2] = {d->recon.host.as<char>() + (size_t)(2 * t) * kPiece,
                         d->recon.host.as<char>() + (size_t)(2 * t + 1) * kPiece};
        size_t held[2] = {pieces.size(), pieces.size()};   // to the host: the piece on its way to the slot
        int k = 0;
        auto empty = [&](int q) {   // the slot's copy is over; to the host: its piece into place
            if (held[q] == pieces.size()) return;
            if (e == hipSuccess) e = hipEventSynchronize(ev[q]);
            if (e == hipSuccess && !to_device) std::memcpy(pieces[held[q]].host, slot[q], pieces[held[q]].bytes);
            held[q] = pieces.size();
        };
        for (size_t i = (size_t)t; i < pieces.size() && e == hipSuccess; i += kCopyThreads, k ^= 1) {
            const Piece& p = pieces[i];
            empty(k);
            if (e != hipSuccess) break;
            if (to_device) std::memcpy(slot[k], p.host, p.bytes);
            e = to_device ? hipMemcpyAsync(p.dev, slot[k], p.bytes, hipMemcpyHostToDevice, st)
                          : hipMemcpyAsync(slot[k], p.dev, p.bytes, hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(ev[k], st);
            held[k] = i;
        }
        if (!to_device) {
            empty(k);
            empty(k ^ 1);
        }
        for (hipEvent_t x : ev)
            if (x) (void)hipEventDestroy(x);
        if (e != hipSuccess) err = (int)e;
    };
    std::vector<std::thread> th;
    try {
        for (int t = 1; t < kCopyThreads; t++) th.emplace_back(work, t);
    } catch (const std::system_error&) {   // no more threads: their share in this one
    }
    const int first = (int)th.size() + 1;
    work(0);
    for (int t = first; t < kCopyThreads; t++) work(t);
    for (std::thread& x : th) x.join();
    T2X_HIP((hipError_t)err.load());
    return T2X_OK;
}

// The n^3 double plan of a kind (0: Z2D, 1: D2Z), made when the size changes; its work area is placed by
// the caller (plan_work bytes, hipfftSetWorkArea).
int recon_plan(ReconWork& w, int kind, int n, hipStream_t st)
{
    if (w.plan_n[kind] == n) return T2X_OK;
    if (w.plan[kind]) (void)hipfftDestroy(w.plan[kind]);
    w.plan[kind] = 0;
    w.plan_n[kind] = 0;
    hipfftHandle h = 0;
    if (hipfftCreate(&h) != HIPFFT_SUCCESS) return T2X_EDEVICE;
    if (hipfftSetAutoAllocation(h, 0) != HIPFFT_SUCCESS ||
        hipfftMakePlan3d(h, n, n, n, kind == 0 ? HIPFFT_Z2D : HIPFFT_D2Z, &w.plan_work[kind]) != HIPFFT_SUCCESS ||
        hipfftSetStream(h, st) != HIPFFT_SUCCESS) {
        (void)hipfftDestroy(h);
        return T2X_EDEVICE;
    }
    w.plan[kind] = h;
    w.plan_n[kind] = n;
    return T2X_OK;
}

}  // namespace

}  // namespace t2x

using namespace t2x;

// Shared body of t2x_reconstruct (inputs from host arrays) and t2x_reconstruct_class (inputs from
// the device backprojector `bp`); the caller holds the device lock.
static int reconstruct_run(Device* d, const t2x_recon_params* p, const double* data_re, const double* data_im,
                           const double* weight, const ClassVolumes* bp, const double* tau2, double* vol_out)
{
    if (p->ref_dim != 3) { set_error("t2x_reconstruct: only 3D references are supported"); return T2X_EINVAL; }
    if (!p->skip_gridding) {
        set_error("t2x_reconstruct: the iterative gridding branch (--dont_skip_gridding) is not supported");
        return T2X_EINVAL;
    }
    if (p->ori_size < 2 || p->ori_size % 2 || p->r_max < 1 || p->padding_factor <= 0. ||
        p->pad_size != 2 * ((int)std::lround(p->padding_factor * p->r_max) + 1) + 1) {
        set_error("t2x_reconstruct: inconsistent sizes (pad_size must be 2*(ROUND(pf*r_max)+1)+1, even ori_size)");
        return T2X_EINVAL;
    }
    if (p->do_map && !tau2) { set_error("t2x_reconstruct: do_map needs tau2"); return T2X_EINVAL; }
    if (bp && (bp->b_ref_dim != p->ref_dim || bp->b_pad != p->pad_size || bp->b_rmax != p->r_max ||
               bp->b_pf != p->padding_factor)) {
        set_error("t2x_reconstruct_class: the backprojector's ref_dim/pad_size/r_max/padding_factor differ from the params");
        return T2X_EINVAL;
    }
    T2X_HIP(hipSetDevice(d->id));
    hipStream_t st = d->stream;

    ReconGeom g{};
    g.pad = p->pad_size;
    g.xh = g.pad / 2 + 1;
    g.pf = p->padding_factor;
    g.ori = p->ori_size;
    long long P = std::llround(g.pf * g.ori);
    P += P % 2;
    g.P = P;
    g.Ph = P / 2 + 1;
    const long long rr = std::llround(p->r_max * g.pf);
    g.max_r2 = rr * rr;
    g.round_max_r2 = std::llround(p->r_max * g.pf * p->r_max * g.pf);
    g.win_r2 = (g.xh - 1) * (g.xh - 1);
    g.r_max = p->r_max;
    g.do_map = p->do_map;
    g.minres_map = p->minres_map;
    g.tau2_fudge = p->tau2_fudge;
    g.normfft = (p->data_dim == 3) ? g.pf * g.pf * g.pf : g.pf * g.pf * g.pf * (double)g.ori;

    const size_t nv = (size_t)g.pad * g.pad * g.xh;
    const size_t nw = (size_t)P * P * g.Ph;
    const size_t nr = (size_t)P * P * P;
    const size_t no = (size_t)g.ori * g.ori * g.ori;
    const int nshell_tau = g.ori / 2 + 1;
    // the MAP shell index ROUND(|k|/pf) for |k|^2 < max_r2 stays below r_max + 1 <= ori/2 + 1
    if (p->do_map && (long long)p->r_max + 1 > nshell_tau) {
        set_error("t2x_reconstruct: r_max exceeds the tau2 spectrum (ori_size/2+1 shells)");
        return T2X_EINVAL;
    }
    ReconWork& rw = d->recon;
    if (recon_plan(rw, 0, (int)P, st) != T2X_OK) {
        set_error("t2x_reconstruct: hipFFT Z2D plan failed");
        return T2X_EDEVICE;
    }
    Arena ar;
    const size_t o_re = ar.take(nv * 8), o_im = ar.take(nv * 8), o_w = ar.take(nv * 8), o_Fw = ar.take(nv * 8),
                 o_tau = ar.take((size_t)nshell_tau * 8), o_ps = ar.take((size_t)kShellBlocks * g.r_max * 8),
                 o_pc = ar.take((size_t)kShellBlocks * g.r_max * 8), o_floor = ar.take((size_t)g.r_max * 8),
                 o_err = ar.take(sizeof(int)), o_W = ar.take(nw * 16), o_R = ar.take(nr * 8),
                 o_vol = ar.take(no * 8), o_bg = ar.take(kShellBlocks * 8), o_bw = ar.take(kShellBlocks * 8),
                 o_fft = ar.take(rw.plan_work[0]);
    ArenaRelease release{rw, st};
    T2X_TRY(rw.arena.ensure(ar.bytes));
    char* base = rw.arena.as<char>();
    auto at = [&](size_t o) { return reinterpret_cast<double*>(base + o); };
    double *b_re = at(o_re), *b_im = at(o_im), *b_w = at(o_w), *b_Fw = at(o_Fw), *b_tau = at(o_tau), *b_ps = at(o_ps),
           *b_pc = at(o_pc), *b_floor = at(o_floor), *b_R = at(o_R), *b_vol = at(o_vol), *b_bg = at(o_bg), *b_bw = at(o_bw);
    double2* b_W = reinterpret_cast<double2*>(base + o_W);
    int* b_err = reinterpret_cast<int*>(base + o_err);
    if (bp) {
        k_bp_widen<<<(unsigned)std::min<size_t>((nv + 255) / 256, 65536), 256, 0, st>>>(
            nv, bp->bp_data, bp->bp_weight, b_re, b_im, b_w);
        T2X_HIP(hipGetLastError());
    } else {
        T2X_TRY(staged_copy(d, {{(char*)b_re, (char*)data_re, nv * 8}, {(char*)b_im, (char*)data_im, nv * 8},
                                {(char*)b_w, (char*)weight, nv * 8}}, true));
    }
    if (p->do_map) T2X_HIP(hipMemcpyAsync(b_tau, tau2, (size_t)nshell_tau * 8, hipMemcpyHostToDevice, st));
    else T2X_HIP(hipMemsetAsync(b_tau, 0, (size_t)nshell_tau * 8, st));
    T2X_HIP(hipMemsetAsync(b_err, 0, sizeof(int), st));

    k_recon_weights<<<kShellBlocks, 256, 2 * sizeof(double) * g.r_max, st>>>(
        g, b_w, b_tau, b_Fw, b_ps, b_pc,
        b_err);
    T2X_HIP(hipGetLastError());
    k_recon_floor<<<(g.r_max + 255) / 256, 256, 0, st>>>(g, b_ps, b_pc, kShellBlocks,
                                                         b_floor, b_err);
    T2X_HIP(hipGetLastError());
    k_recon_window<<<(unsigned)std::min<size_t>((nw + 255) / 256, 65536), 256, 0, st>>>(
        g, b_re, b_im, b_Fw, b_floor, b_W);
    T2X_HIP(hipGetLastError());
    int herr = 0;
    T2X_HIP(hipMemcpyAsync(&herr, b_err, sizeof(int), hipMemcpyDeviceToHost, st));
    T2X_HIP(hipStreamSynchronize(st));
    if (herr == 2) { set_error("t2x_reconstruct: negative tau2 values"); return T2X_EINVAL; }
    if (herr == 3 || herr == 4) { set_error("t2x_reconstruct: empty or inconsistent weight shells"); return T2X_EINVAL; }

    if (hipfftSetWorkArea(rw.plan[0], base + o_fft) != HIPFFT_SUCCESS ||
        hipfftExecZ2D(rw.plan[0], reinterpret_cast<hipfftDoubleComplex*>(b_W), b_R) != HIPFFT_SUCCESS) {
        set_error("t2x_reconstruct: hipFFT Z2D failed");
        return T2X_EDEVICE;
    }
    k_recon_crop<<<kShellBlocks, 1024, 0, st>>>(g, b_R, b_vol, b_bg,
                                                b_bw);
    T2X_HIP(hipGetLastError());
    k_recon_finish<<<(unsigned)std::min<size_t>((no + 255) / 256, 65536), 256, 0, st>>>(
        g, b_bg, b_bw, kShellBlocks, b_vol);
    T2X_HIP(hipGetLastError());
    return staged_copy(d, {{(char*)b_vol, (char*)vol_out, no * 8}}, false);
}

extern "C" int t2x_reconstruct(t2x_device* hdev, const t2x_recon_params* p, const double* data_re,
                               const double* data_im, const double* weight, const double* tau2, double* vol_out)
{
    if (!hdev || !p || !data_re || !data_im || !weight || !vol_out) { set_error("null argument"); return T2X_EINVAL; }
    Device* d = reinterpret_cast<Device*>(hdev);
    std::lock_guard<std::mutex> lk(d->mtx);
    return reconstruct_run(d, p, data_re, data_im, weight, nullptr, tau2, vol_out);
}

extern "C" int t2x_reconstruct_class(t2x_device* hdev, int iclass, const t2x_recon_params* p, const double* tau2,
                                     double* vol_out)
{
    if (!hdev || !p || !vol_out) { set_error("null argument"); return T2X_EINVAL; }
    Device* d = reinterpret_cast<Device*>(hdev);
    std::lock_guard<std::mutex> lk(d->mtx);
    auto it = d->classes.find(iclass);
    if (it == d->classes.end() || !it->second.bp_data) {
        set_error("t2x_reconstruct_class: backprojector not initialised");
        return T2X_ESTATE;
    }
    return reconstruct_run(d, p, nullptr, nullptr, nullptr, &it->second, tau2, vol_out);
}

extern "C" int t2x_fsc(t2x_device* hdev, int n, const double* map1, const double* map2, double* fsc)
{
    if (!hdev || !map1 || !map2 || !fsc) { set_error("null argument"); return T2X_EINVAL; }
    if (n < 2) { set_error("t2x_fsc: n < 2"); return T2X_EINVAL; }
    Device* d = reinterpret_cast<Device*>(hdev);
    std::lock_guard<std::mutex> lk(d->mtx);
    T2X_HIP(hipSetDevice(d->id));
    hipStream_t st = d->stream;
    const long long N = n, xh = N / 2 + 1;
    const size_t nr = (size_t)N * N * N, nc = (size_t)N * N * xh;
    ReconWork& rw = d->recon;
    if (recon_plan(rw, 1, n, st) != T2X_OK) {
        set_error("t2x_fsc: hipFFT D2Z plan failed");
        return T2X_EDEVICE;
    }
    Arena ar;
    const size_t o_r1 = ar.take(nr * 8), o_r2 = ar.take(nr * 8), o_c1 = ar.take(nc * 16), o_c2 = ar.take(nc * 16),
                 o_part = ar.take((size_t)kShellBlocks * 3 * xh * 8), o_out = ar.take((size_t)xh * 8),
                 o_fft = ar.take(rw.plan_work[1]);
    ArenaRelease release{rw, st};
    T2X_TRY(rw.arena.ensure(ar.bytes));
    char* base = rw.arena.as<char>();
    double *r1 = reinterpret_cast<double*>(base + o_r1), *r2 = reinterpret_cast<double*>(base + o_r2),
           *part = reinterpret_cast<double*>(base + o_part), *out = reinterpret_cast<double*>(base + o_out);
    double2 *c1 = reinterpret_cast<double2*>(base + o_c1), *c2 = reinterpret_cast<double2*>(base + o_c2);
    T2X_TRY(staged_copy(d, {{(char*)r1, (char*)map1, nr * 8}, {(char*)r2, (char*)map2, nr * 8}}, true));
    if (hipfftSetWorkArea(rw.plan[1], base + o_fft) != HIPFFT_SUCCESS ||
        hipfftExecD2Z(rw.plan[1], r1, reinterpret_cast<hipfftDoubleComplex*>(c1)) != HIPFFT_SUCCESS ||
        hipfftExecD2Z(rw.plan[1], r2, reinterpret_cast<hipfftDoubleComplex*>(c2)) != HIPFFT_SUCCESS) {
        set_error("t2x_fsc: hipFFT D2Z failed");
        return T2X_EDEVICE;
    }
    k_fsc_partial<<<kShellBlocks, 256, 3 * sizeof(double) * xh, st>>>(N, c1, c2, part);
    T2X_HIP(hipGetLastError());
    k_fsc_final<<<(unsigned)((xh + 255) / 256), 256, 0, st>>>(N, part, kShellBlocks, out);
    T2X_HIP(hipGetLastError());
    T2X_HIP(hipMemcpyAsync(fsc, out, (size_t)xh * 8, hipMemcpyDeviceToHost, st));
    T2X_HIP(hipStreamSynchronize(st));
    return T2X_OK;
}
