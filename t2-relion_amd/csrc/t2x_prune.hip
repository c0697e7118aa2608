// t2x_prune.hip — exact lower bounds of the coarse diff2 from an INT8 GEMM (the pruned coarse pass).
//
// The coarse diff2 of (particle b, translation t, orientation n) is C_b + N1[b,n] - G with the
// cross term G = sum_k A[(b,t),k] B[n,k] over the coarse pixels (re/im interleaved), which are
// ordered by |frequency|. A prefix of n_low pixels (the low set) enters an INT8 GEMM, the rest
// (the high set) a Cauchy-Schwarz bound:
//   G = <A', B'>_low + G_high,  A'_k = w_k A_k,  B'_k = B_k / w_k,
//   <A', B'> = <Aq, Bq> + <dA, B'> + <Aq, dB>  <=  sA sB <qa, qb> + |dA| |B'| + |Aq| |dB|,
//   G_high <= 2 sqrt(N1h Ch)
// with Aq = sA qa, Bq = sB qb the quantised rows (qa, qb whole numbers of at most 127), dA = A' - Aq,
// dB = B' - Bq their exact errors (their norms are taken when the rows are quantised), N1h the N1
// term of the high set and Ch the image's energy there. So
//   lb = C_b + N1 - 2 sqrt(N1h Ch) - |dA| |B'| - |Aq| |dB| - margin - sA sB <qa, qb>
// is a lower bound of the diff2 the full GEMM computes: the margin 2 2^-9 sqrt(N1 Cl) (Cl the image's
// energy in the low set) covers the full pass's own rounding (FP16X2 drops the reference's low half:
// 2^-11 of sum |A||B| <= 2 sqrt(N1 Cl); the other precisions and the FP32 sums less). The bounds need
// no digit of the result, so they are taken at the matrix cores' INT8 rate whatever the precision of
// the pass, FP32 included: a tile whose bounds all lie beyond the negligible-weight cut above a
// computed value of its particle is not computed, the others are computed as the exhaustive pass does.
//
// The weights w_k (the fourth root of the references' mean power at pixel k) level the rows, so that a
// row's largest element is a few times its rms: the errors |dA| / |A'| and |dB| / |B'| are ~1%.
// sA is one scale per particle (its translations' rows differ in phase only) and sB one per 64
// orientations, so a block's minimum over a particle's rows needs the largest <qa, qb> of each column
// alone: the epilogue is integer maxima, and the rest is a table (k_prune_base) in units of sA sB.
#include "t2x_kernels.h"
#include <algorithm>
#include <climits>

namespace t2x {

typedef int v4i __attribute__((ext_vector_type(4)));

// Base table values: unscored and padding columns, the clamp of scored ones (upwards conservative,
// downwards marked: a block at or below PB_LOW is always computed), and "no row yet" of a maximum.
// Differences stay within 32 bits: PB_BIG - PB_NONE = 2^31 - 1, and |<qa, qb>| <= 127^2 K8 < 2.7e8.
#define PB_BIG ((1 << 30) - 1)
#define PB_CLAMP 1000000000
#define PB_LOW (-700000000)
#define PB_NONE (-(1 << 30))

__device__ __forceinline__ float prune_unit(float sa, float sb)
{
    const float u = sa * sb;
    return u > 0.f ? u : 1.f;
}

__device__ __forceinline__ float wave_sum(float v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ float wave_max(float v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// Row weights of the low pixels: w = (mean |F|^2 over 4,096 to 8,191 orientations, or all)^(1/4), at least
// 1e-3 of the largest (any positive weights give valid bounds; these level the rows). The sums of
// one of PP_PARTS parts of the orientations for 64 pixels a workgroup; k_prune_weights adds the parts
// and turns them into w and 1 / w.
#define PP_PARTS 32
__global__ __launch_bounds__(256) void k_prune_power(const float* __restrict__ B2, long long ldb2, long long O_all,
                                                     int n_low, float* __restrict__ g)
{
    __shared__ float s[4][64];
    const int p = blockIdx.x * 64 + (threadIdx.x & 63), part = threadIdx.x >> 6;
    const long long step = O_all > 4096 ? O_all / 4096 : 1;
    float a = 0.f;
    if (p < n_low)
        for (long long n = (part * PP_PARTS + blockIdx.y) * step; n < O_all; n += 4 * PP_PARTS * step) a += B2[n * ldb2 + p];
    s[part][threadIdx.x & 63] = a;
    __syncthreads();
    if (part == 0 && p < n_low) {
        const int c = threadIdx.x;
        g[(size_t)blockIdx.y * n_low + p] = s[0][c] + s[1][c] + s[2][c] + s[3][c];
    }
}

__global__ __launch_bounds__(1024) void k_prune_weights(int n_low, const float* __restrict__ g, float* __restrict__ w,
                                                        float* __restrict__ iw)
{
    __shared__ float red[16];
    float mx = 0.f;
    for (int p = threadIdx.x; p < n_low; p += 1024) {
        float a = 0.f;
        for (int k = 0; k < PP_PARTS; k++) a += g[(size_t)k * n_low + p];
        w[p] = a;
        mx = fmaxf(mx, a);
    }
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    for (int k = 0; k < 16; k++) mx = fmaxf(mx, red[k]);
    const bool ok = mx > 0.f && mx < 3.0e38f;
    for (int p = threadIdx.x; p < n_low; p += 1024) {
        const float v = ok ? sqrtf(sqrtf(fmaxf(w[p] / mx, 1e-12f))) : 1.f;
        w[p] = v;
        iw[p] = 1.f / v;
    }
}

// The references' side: one workgroup per 64 orientations, which share the scale. Rows of K8 bytes
// (zero beyond 2 n_low and for orientations >= O_all), |dB| and |B'| of each row (rounded up).
__global__ __launch_bounds__(1024) void k_prune_quant_b(const float* __restrict__ Bm, long long ldb, long long O_all,
                                                       int n_low, int K8, const float* __restrict__ iw,
                                                       signed char* __restrict__ q8, float* __restrict__ sb,
                                                       float2* __restrict__ nb)
{
    __shared__ float red[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long n0 = (long long)blockIdx.x * 64;
    float mx = 0.f;
    for (int r = wave; r < 64; r += 16) {
        const long long n = n0 + r;
        if (n >= O_all) continue;
        const float2* row = reinterpret_cast<const float2*>(Bm + n * ldb);
        for (int p = lane; p < n_low; p += 64) {
            const float2 f = row[p];
            mx = fmaxf(mx, fmaxf(fabsf(f.x), fabsf(f.y)) * iw[p]);
        }
    }
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    for (int k = 0; k < 16; k++) mx = fmaxf(mx, red[k]);
    const float s = mx / 127.f, inv = s > 0.f ? 1.f / s : 0.f;
    if (threadIdx.x == 0) sb[blockIdx.x] = s;
    for (int r = wave; r < 64; r += 16) {
        const long long n = n0 + r;
        const bool valid = n < O_all;
        const float2* row = reinterpret_cast<const float2*>(Bm + (valid ? n : 0) * ldb);
        char2* out = reinterpret_cast<char2*>(q8 + n * K8);
        float e = 0.f, t = 0.f;
        for (int p = lane; p < K8 / 2; p += 64) {
            char2 q = make_char2(0, 0);
            if (valid && p < n_low) {
                const float2 f = row[p];
                const float a = f.x * iw[p], b = f.y * iw[p];
                const float qa = fminf(fmaxf(rintf(a * inv), -127.f), 127.f), qb = fminf(fmaxf(rintf(b * inv), -127.f), 127.f);
                const float da = a - qa * s, db = b - qb * s;
                e += da * da + db * db;
                t += a * a + b * b;
                q = make_char2((signed char)qa, (signed char)qb);
            }
            out[p] = q;
        }
        e = wave_sum(e);
        t = wave_sum(t);
        if (lane == 0) nb[n] = make_float2(sqrtf(e) * 1.0001f, sqrtf(t) * 1.0001f);
    }
}

// What a particle's bounds lose: the factors of sqrt(N1h) (the high set) and sqrt(N1) (the margin).
// 2^-7: the BF16 rounding of N1h's operands and, in the high set, the full pass's own; 2^-9: the margin.
__device__ __forceinline__ float2 prune_factors(const PartScalars& s)
{
    const float ch = (float)fmax(s.C_coarse - s.C_low, 0.) * 1.00001f;
    const float cl = (float)fmax(s.C_low - s.highres_Xi2 / 2., 0.) * 1.00001f;
    return make_float2(2.f * (1.f + 1.f / 128.f) * sqrtf(ch), 2.f / 512.f * sqrtf(cl));
}

// Particles whose bounds lose more than 10 (the cut is 61) by the high set, over 32 orientations on
// average: a larger low set helps them. One workgroup per particle, one wave per orientation.
__global__ __launch_bounds__(256) void k_prune_high(const PartScalars* __restrict__ ps, int stride,
                                                    const float* __restrict__ A1, long long lda1,
                                                    const float* __restrict__ B2, long long ldb2, long long O_all,
                                                    int n_low, int npix, const double* __restrict__ prior_o,
                                                    unsigned* __restrict__ count)
{
    __shared__ float sh[4], sn[4];
    const long long b = (long long)blockIdx.x * stride;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float c0 = prune_factors(ps[b]).x;
    float high = 0.f, cnt = 0.f;
    for (int q = wave; q < 32; q += 4) {
        const long long n = (long long)((q + 0.5) * (double)O_all / 32.);
        if (n >= O_all || !(prior_o[n] > 0.)) continue;
        float h = 0.f;
        for (int p = n_low + lane; p < npix; p += 64) h += A1[b * lda1 + p] * B2[n * ldb2 + p];
        high += c0 * sqrtf(fmaxf(wave_sum(h), 0.f));
        cnt += 1.f;
    }
    if (lane == 0) { sh[wave] = high; sn[wave] = cnt; }
    __syncthreads();
    if (threadIdx.x == 0 && sh[0] + sh[1] + sh[2] + sh[3] > 10.f * (sn[0] + sn[1] + sn[2] + sn[3])) atomicAdd(count, 1u);
}

// The images' side: one workgroup per particle, its T rows minv ctf X_t w in whole numbers with one
// scale; pa[b] = (scale, largest |Aq| of its rows, largest |dA|, 0). The particle's weighted image
// stays in LDS, each wave turns it by one translation's phases at a time. A sample's few particles leave most
// of the chip idle, so they take 16 waves each instead of 4 (10 particles of 49 translations: 58 -> 21 us).
__global__ __launch_bounds__(1024) void k_prune_quant_a(const float2* __restrict__ Fimg, const float* __restrict__ Fctf,
                                                       int Pw, const int* __restrict__ win,
                                                       const float* __restrict__ minv, int npix,
                                                       const PartScalars* __restrict__ ps, int stride,
                                                       const float2* __restrict__ ab, int T, int n_low, int K8,
                                                       const float* __restrict__ w, signed char* __restrict__ q8,
                                                       float4* __restrict__ pa)
{
    extern __shared__ float2 y[];   // [n_low]
    __shared__ float red[16][2];
    const int b = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const size_t bs = (size_t)b * stride;
    const float* mv = minv + (size_t)ps[bs].og * npix;
    float mx = 0.f;
    for (int p = threadIdx.x; p < n_low; p += blockDim.x) {
        const size_t q = bs * Pw + win[p];
        const float2 x = Fimg[q];
        const float s = mv[p] * Fctf[q] * w[p];
        const float2 v = make_float2(s * x.x, s * x.y);
        y[p] = v;
        mx = fmaxf(mx, v.x * v.x + v.y * v.y);
    }
    mx = wave_max(mx);
    if (lane == 0) red[wave][0] = mx;
    __syncthreads();
    for (int k = 0; k < nw; k++) mx = fmaxf(mx, red[k][0]);
    __syncthreads();
    const float s = sqrtf(mx) / 127.f, inv = s > 0.f ? 1.f / s : 0.f;
    float emax = 0.f, tmax = 0.f;
    for (int t = wave; t < T; t += nw) {
        char2* out = reinterpret_cast<char2*>(q8 + ((size_t)b * T + t) * K8);
        float e = 0.f, n = 0.f;
        for (int p = lane; p < K8 / 2; p += 64) {
            char2 q = make_char2(0, 0);
            if (p < n_low) {
                const float2 v = y[p], sh = ab[(size_t)t * npix + p];
                const float a = v.x * sh.x - v.y * sh.y, c = v.x * sh.y + v.y * sh.x;
                const float qa = fminf(fmaxf(rintf(a * inv), -127.f), 127.f), qc = fminf(fmaxf(rintf(c * inv), -127.f), 127.f);
                const float da = a - qa * s, dc = c - qc * s;
                e += da * da + dc * dc;
                n += qa * qa + qc * qc;
                q = make_char2((signed char)qa, (signed char)qc);
            }
            out[p] = q;
        }
        emax = fmaxf(emax, wave_sum(e));
        tmax = fmaxf(tmax, wave_sum(n));
    }
    if (lane == 0) { red[wave][0] = emax; red[wave][1] = tmax; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < nw; k++) { emax = fmaxf(emax, red[k][0]); tmax = fmaxf(tmax, red[k][1]); }
        pa[b] = make_float4(s, sqrtf(tmax) * s * 1.0001f, sqrtf(emax) * 1.0001f, 0.f);
    }
}

// N1 less everything that bounds the cross term's error, rounded down.
// (v_sqrt_f32 alone, 1 ulp: the last term covers it.)
__device__ __forceinline__ float prune_base_value(float n1, float n1h, float2 pf, float4 pa, float2 nb)
{
    const float lose = pf.x * __builtin_amdgcn_sqrtf(fmaxf(n1h, 0.f)) + pf.y * __builtin_amdgcn_sqrtf(fmaxf(n1, 0.f)) +
                       pa.z * nb.y + pa.y * nb.x;
    return n1 - lose - 4e-6f * (fabsf(n1) + lose);
}

// The base table: N1 less the error bounds in units of sA sB, rounded down to whole numbers, for every
// (particle, orientation). N1h = sum over the high pixels of A1 |F|^2 on the matrix cores, its
// non-negative operands rounded to BF16 as they are staged in LDS (their 2^-8 is in c0). 128x128 tiles
// of 4 waves, K step 32; bound by the N1 read and the table's write.
#define PB_PAD 8
__global__ __launch_bounds__(256) void k_prune_base(const PartScalars* __restrict__ ps, int B, int stride,
                                                    const float* __restrict__ N1, long long ldn,
                                                    const float* __restrict__ A1, long long lda1,
                                                    const float* __restrict__ B2, long long ldb2, long long O_all,
                                                    int n_low, int Kn, const float4* __restrict__ pa,
                                                    const float* __restrict__ sb, const float2* __restrict__ nb,
                                                    const double* __restrict__ prior_o, int tiles_m,
                                                    int* __restrict__ base)
{
    typedef Vec8<__bf16>::type v8;
    __shared__ __attribute__((aligned(16))) __bf16 As[128][32 + PB_PAD];
    __shared__ __attribute__((aligned(16))) __bf16 Bs[128][32 + PB_PAD];
    __shared__ float4 spa[128];
    __shared__ float2 spf[128];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = (int)(blockIdx.x % (unsigned)tiles_m) * 128;
    const long long n0 = (long long)(blockIdx.x / (unsigned)tiles_m) * 128;
    floatx4 acc[4][4];
    for (int i = 0; i < 4; i++)
        for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (tid < 128) {
        const int b = min(m0 + tid, B - 1);
        spa[tid] = pa[b];
        spf[tid] = prune_factors(ps[(long long)b * stride]);
    }
    // loader: thread -> (row tid / 2, 16 columns), one K step ahead; rows beyond B read the last particle's
    const int lrow = tid >> 1, lc = (tid & 1) * 16;
    const float* ap = A1 + (long long)min(m0 + lrow, B - 1) * stride * lda1 + lc;
    const float* bp = B2 + (n0 + lrow) * ldb2 + lc;
    const int kb = n_low & ~31;
    float a[16], b[16];
#define PB_LOAD(k0)                                                                          \
    do {                                                                                     \
        _Pragma("unroll") for (int q = 0; q < 4; q++) {                                      \
            *reinterpret_cast<float4*>(&a[4 * q]) = *reinterpret_cast<const float4*>(ap + (k0) + 4 * q); \
            *reinterpret_cast<float4*>(&b[4 * q]) = *reinterpret_cast<const float4*>(bp + (k0) + 4 * q); \
        }                                                                                    \
    } while (0)
    if (kb < Kn) PB_LOAD(kb);
    for (int k0 = kb; k0 < Kn; k0 += 32) {
        v8 va[2], vb[2];
#pragma unroll
        for (int q = 0; q < 16; q++) {   // pixels of the low set count nothing
            va[q >> 3][q & 7] = (__bf16)(k0 + lc + q >= n_low ? a[q] : 0.f);
            vb[q >> 3][q & 7] = (__bf16)b[q];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; q++) {
            *reinterpret_cast<v8*>(&As[lrow][lc + 8 * q]) = va[q];
            *reinterpret_cast<v8*>(&Bs[lrow][lc + 8 * q]) = vb[q];
        }
        __syncthreads();
        if (k0 + 32 < Kn) PB_LOAD(k0 + 32);
        const int kc = (lane >> 4) * 8;
        v8 fa[4], fb[4];
#pragma unroll
        for (int i = 0; i < 4; i++) fa[i] = *reinterpret_cast<const v8*>(&As[wm * 64 + i * 16 + (lane & 15)][kc]);
#pragma unroll
        for (int j = 0; j < 4; j++) fb[j] = *reinterpret_cast<const v8*>(&Bs[wn * 64 + j * 16 + (lane & 15)][kc]);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
#undef PB_LOAD
    __syncthreads();   // spa, spf (where there is no high set the loop has no barrier)
    float2 nbj[4];
    bool sc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const long long n = n0 + wn * 64 + j * 16 + (lane & 15);
        sc[j] = n < O_all && prior_o[n] > 0.;
        nbj[j] = sc[j] ? nb[n] : make_float2(0.f, 0.f);
    }
    const float sbk = sb[(n0 + wn * 64) / 64];
    const long long nl = n0 + wn * 64 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r0 = wm * 64 + i * 16 + (lane >> 4) * 4;
        float n1[4][4];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) n1[r][j] = N1[(long long)min(m0 + r0 + r, B - 1) * stride * ldn + nl + j * 16];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int bb = m0 + r0 + r;
            const float4 pab = spa[r0 + r];
            const float2 pfb = spf[r0 + r];
            const float inv = 1.f / prune_unit(pab.x, sbk);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float x = floorf(prune_base_value(n1[r][j], acc[i][j][r], pfb, pab, nbj[j]) * inv);
                int v = x >= (float)PB_CLAMP ? PB_CLAMP : (x > -(float)PB_CLAMP ? (int)x : -PB_CLAMP);
                v = sc[j] ? v : PB_BIG;
                if (bb < B) base[(long long)bb * ldn + nl + j * 16] = v;
            }
        }
    }
}

// Walk of the bounds GEMM's tiles: groups of 32 tile rows, inside them blocks of 32 x 8 tiles, of which
// the 8 XCDs (workgroup index & 7) take an 8 x 4 part each, the next block of the group keeping the rows.
// A part's 8 + 4 operand tiles are 3 KB a byte of row: up to 1,300 bytes of row they fit one L2 (4 MB)
// whole; longer rows are walked in step, 64 bytes at a time, so that what the parts' tiles share is in
// the L2 together too. Measured at rows of 1,152 bytes only. Partial blocks are walked rows first.
#define PW_ROWS 32
#define PW_COLS 8
__device__ __forceinline__ void bounds_tile(int t, int tiles_m, int tiles_n, int& tm, int& tn)
{
    const int per_group = PW_ROWS * tiles_n;
    const int g = t / per_group;
    const int gs = min(tiles_m - g * PW_ROWS, PW_ROWS);
    const int q = t - g * per_group;
    const int cb = q / (gs * PW_COLS), r = q - cb * gs * PW_COLS;
    const int cw = min(tiles_n - cb * PW_COLS, PW_COLS);
    if (gs == PW_ROWS && cw == PW_COLS) {
        const int x = r & 7, l = r >> 3;   // XCD, and 0 .. 31 inside its part
        tm = g * PW_ROWS + (x >> 1) * 8 + (l & 7);
        tn = cb * PW_COLS + (x & 1) * 4 + (l >> 3);
    } else {
        tm = g * PW_ROWS + r % gs;
        tn = cb * PW_COLS + r / gs;
    }
}

__device__ __forceinline__ int min_row16(int v)
{
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, false));
    v = min(v, __builtin_amdgcn_mov_dpp(v, 0x140, 0xF, 0xF, false));
    return v;
}

typedef const void __attribute__((address_space(1)))* gptr_t;
typedef void __attribute__((address_space(3)))* lptr_t;

struct BoundsParams {
    const signed char* A;   // [tiles_m * 256][K8]
    const signed char* B;   // [tiles_n * 256][K8]
    int K8, M, T, tiles_m, tiles_n;
    const int* base;        // [particles][ldb]
    long long ldb;
    int* lbs;               // [tiles_m * 2][S][nblk]
    int nblk, S, nb_part;   // particles
    int stride;             // particle b is the batch's particle b stride
};

// The INT8 bounds GEMM. lbs[h][z][blk]: over rows [128 h, 128 h + 128) of the z-th particle among them
// and columns [64 blk, 64 blk + 64), the minimum of base - <qa, qb>: lower bounds of diff2 - C_b in
// units of the particle's and the block's scales. K8 a multiple of 128.
//
// One persistent workgroup per compute unit, 256x256 tiles, 8 waves of 128x64 on
// v_mfma_i32_16x16x64_i8. A K step is 64 bytes of every row (32 KB); a ring of four steps in LDS,
// filled by global_load_lds three steps ahead and running on over the tiles of the workgroup, so that
// no tile waits for its first operands; a step's fragments are read while the step before it
// multiplies. The barrier of a step says that its stage is complete and that the stage before it has
// been read by all. Maxima over a particle's rows come first (integers, in registers), then one
// subtraction per column, so the epilogue is a few hundred instructions for 128 MFMA results a lane.
// Measured at 39,200 x 147,456 x 1,152: 6.0 ms (2,200 TOP/s); the same tile as one workgroup per tile
// with an FP32 epilogue per element 7.9 ms; its MFMAs alone would take 2.7 ms at 2.4 GHz and its
// operand moves alone 3.6 ms. The FP16 form over the same pixels (two K chunks a stage, one workgroup
// per tile) took 14.2 ms.
// SB: base rows a wave stages per tile (8 SB particles a tile); 0: the epilogue reads them from memory.
template <int SB>
__global__ __launch_bounds__(512, 2) void k_gemm_i8_bounds(BoundsParams p)
{
    __shared__ __attribute__((aligned(16))) signed char s0[32768], s1[32768], s2[32768], s3[32768];
    __shared__ __attribute__((aligned(16))) int sbase[(SB ? SB : 1) * 8 * 256];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave & 1, wn = wave >> 1;
    const int ntiles = p.tiles_m * p.tiles_n, T = p.T;
    int t = blockIdx.x;
    if (t >= ntiles) return;
    int tm, tn;
    bounds_tile(t, p.tiles_m, p.tiles_n, tm, tn);

    // loader: wave w moves rows [32 w, 32 w + 32) of both operands, 16 rows x 64 bytes an instruction:
    // lane l writes 16-byte chunk l & 3 of row l >> 2 and fetches chunk (l & 3) ^ ((row >> 1) & 3)
    const int lr = lane >> 2, lch = (lane & 3) ^ ((lr >> 1) & 3);
    const unsigned r16 = 16u * p.K8, lo = (unsigned)((wave * 32 + lr) * p.K8 + lch * 16);
    const int nk = p.K8 / 64;
    // the load cursor runs three steps ahead, over this workgroup's tiles (past the last one it
    // reads the current tile again, into stages nobody uses)
    int lt = t, lk = 0;
    const signed char* pa = p.A + (long long)tm * 256 * p.K8;
    const signed char* pb = p.B + (long long)tn * 256 * p.K8;
#define I8_LOAD(S)                                                                                                  \
    do {                                                                                                            \
        _Pragma("unroll") for (int q = 0; q < 2; q++) {                                                             \
            __builtin_amdgcn_global_load_lds((gptr_t)(pa + lo + q * r16), (lptr_t)&S[(wave * 2 + q) * 1024], 16, 0, 0); \
            __builtin_amdgcn_global_load_lds((gptr_t)(pb + lo + q * r16), (lptr_t)&S[16384 + (wave * 2 + q) * 1024], 16, 0, 0); \
        }                                                                                                           \
        pa += 64;                                                                                                   \
        pb += 64;                                                                                                   \
        if (++lk == nk) {                                                                                           \
            lk = 0;                                                                                                 \
            lt += gridDim.x;                                                                                        \
            int am, an;                                                                                             \
            bounds_tile(lt < ntiles ? lt : t, p.tiles_m, p.tiles_n, am, an);                                        \
            pa = p.A + (long long)am * 256 * p.K8;                                                                  \
            pb = p.B + (long long)an * 256 * p.K8;                                                                  \
        }                                                                                                           \
    } while (0)
    const int fr = lane & 15, fc = lane >> 4;
    const int oa = (wm * 128 + fr) * 64 + ((fc ^ ((fr >> 1) & 3)) << 4);
    const int ob = 16384 + (wn * 64 + fr) * 64 + ((fc ^ ((fr >> 1) & 3)) << 4);
#define I8_READ(S, FA, FB)                                                                                         \
    do {                                                                                                            \
        _Pragma("unroll") for (int j = 0; j < 4; j++) FB[j] = *reinterpret_cast<const v4i*>(&S[ob + j * 1024]);     \
        _Pragma("unroll") for (int i = 0; i < 8; i++) FA[i] = *reinterpret_cast<const v4i*>(&S[oa + i * 1024]);     \
    } while (0)
    v4i acc[8][4];
    // s_waitcnt immediates: vmcnt(4) (the last step's four loads may be in flight), lgkmcnt(0)
#define I8_VM4 (0x0070 | (0xF << 8) | 4)
#define I8_VM8 (0x0070 | (0xF << 8) | 8)
#define I8_LGKM0 0xC07F
#define I8_STEP(FA, FB, GA, GB, FREE, NXT, FIRST)                                                                   \
    do {                                                                                                            \
        __builtin_amdgcn_s_waitcnt(I8_VM4);                                                                         \
        __builtin_amdgcn_s_waitcnt(I8_LGKM0);                                                                       \
        __builtin_amdgcn_s_barrier();                                                                               \
        if (FIRST) {                                                                                                \
            _Pragma("unroll") for (int q = 0; q < SB; q++) {                                                        \
                const long long z = min((tm * 256) / T + wave * SB + q, p.nb_part - 1);                             \
                __builtin_amdgcn_global_load_lds((gptr_t)(p.base + z * p.ldb + tn * 256 + lane * 4),                \
                                                 (lptr_t)&sbase[(wave * SB + q) * 256], 16, 0, 0);                  \
            }                                                                                                       \
        }                                                                                                           \
        I8_LOAD(FREE);                                                                                              \
        I8_READ(NXT, GA, GB);                                                                                       \
        _Pragma("unroll") for (int i = 0; i < 8; i++)                                                               \
            _Pragma("unroll") for (int j = 0; j < 4; j++)                                                           \
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(FA[i], FB[j], (FIRST) ? (v4i{0, 0, 0, 0}) : acc[i][j], 0, 0, 0); \
    } while (0)

    // The wave's minima: rows in order, the running maximum of each of its 4 columns a lane; where a
    // particle ends (T rows) the maxima become one bound.
    auto epilogue = [&]() __attribute__((always_inline)) {
        const int mr = tm * 256 + wm * 128, mend = min(mr + 128, p.M);
        const int pt = (tm * 256) / T, pw = mr / T, blk = tn * 4 + wn;
        int z = pw, zend = (pw + 1) * T;
        int mx[4] = {PB_NONE, PB_NONE, PB_NONE, PB_NONE};
        auto flush = [&]() __attribute__((always_inline)) {
            int v;
            if (SB) {
                const int* bz = &sbase[(z - pt) * 256 + wn * 64 + fr];
                v = min(min(bz[0] - mx[0], bz[16] - mx[1]), min(bz[32] - mx[2], bz[48] - mx[3]));
            } else {
                const int* bz = p.base + (long long)z * p.ldb + tn * 256 + wn * 64 + fr;
                v = min(min(bz[0] - mx[0], bz[16] - mx[1]), min(bz[32] - mx[2], bz[48] - mx[3]));
            }
            v = min_row16(v);
            v = min(v, __shfl_xor(v, 16));
            v = min(v, __shfl_xor(v, 32));
            if (lane == 0) p.lbs[((long long)(mr >> 7) * p.S + (z - pw)) * p.nblk + blk] = v;
        };
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int r0 = mr + i * 16;
            if (r0 < mend) {
                if (r0 + 16 <= zend && r0 + 16 <= mend) {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        mx[j] = max(max(max(mx[j], acc[i][j][0]), acc[i][j][1]), max(acc[i][j][2], acc[i][j][3]));
                } else {   // a particle ends inside these 16 rows, or the rows do
                    const int rl = r0 + (lane >> 4) * 4, re = min(r0 + 16, mend);
                    int rs = r0;
                    while (true) {
                        const int rt = min(re, zend);   // rows [rs, rt) are particle z's
#pragma unroll
                        for (int j = 0; j < 4; j++)
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                mx[j] = max(mx[j], (rl + r >= rs && rl + r < rt) ? acc[i][j][r] : PB_NONE);
                        rs = rt;
                        if (rs >= re) break;
                        flush();
                        mx[0] = mx[1] = mx[2] = mx[3] = PB_NONE;
                        z++;
                        zend += T;
                    }
                }
            }
            if (r0 + 16 == zend && r0 + 16 < mend) {   // a particle ends with these rows
                flush();
                mx[0] = mx[1] = mx[2] = mx[3] = PB_NONE;
                z++;
                zend += T;
            }
        }
        if (mr < mend) flush();
    };
#define I8_TILE_END()                                                                                              \
    do {                                                                                                            \
        epilogue();                                                                                                 \
        t += gridDim.x;                                                                                             \
        if (t >= ntiles) {                                                                                          \
            __builtin_amdgcn_s_waitcnt(0);   /* no load into LDS outlives the workgroup */                          \
            return;                                                                                                 \
        }                                                                                                           \
        bounds_tile(t, p.tiles_m, p.tiles_n, tm, tn);                                                               \
        s = 0;                                                                                                      \
    } while (0)

    I8_LOAD(s0);
    I8_LOAD(s1);
    I8_LOAD(s2);
    v4i fa0[8], fb0[4], fa1[8], fb1[4];
    __builtin_amdgcn_s_waitcnt(I8_VM8);   // stage 0
    __builtin_amdgcn_s_barrier();
    I8_READ(s0, fa0, fb0);
    int s = 0;   // even: a tile has an even number of steps, so one begins at ring position 0 or 2
    for (;;) {
        if (s == 0) I8_STEP(fa0, fb0, fa1, fb1, s3, s1, 1);
        else I8_STEP(fa0, fb0, fa1, fb1, s3, s1, 0);
        I8_STEP(fa1, fb1, fa0, fb0, s0, s2, 0);
        s += 2;
        if (s == nk) I8_TILE_END();
        if (s == 0) I8_STEP(fa0, fb0, fa1, fb1, s1, s3, 1);
        else I8_STEP(fa0, fb0, fa1, fb1, s1, s3, 0);
        I8_STEP(fa1, fb1, fa0, fb0, s2, s0, 0);
        s += 2;
        if (s == nk) I8_TILE_END();
    }
#undef I8_LOAD
#undef I8_READ
#undef I8_STEP
#undef I8_TILE_END
}

// Per particle an upper bound of its coarse minimum diff2 (one workgroup per particle): the (row half
// tile, block) with the smallest bound, in it the row with the smallest base - <qa, qb> (computed
// again), and of that row the full diff2 of the 64 columns, from the pass's own
// operands in FP32 (the GEMM's products and scales, summed in another order, so plus 1 + 1e-4 |d|);
// +inf where the particle has no scored column. It seeds the pruning test and the lazy stores' running
// minima. H: the split operands' type (bl null under FP16X2), or float: the FP32 pass's rows.
template <class H> struct Vec16 { typedef H type __attribute__((ext_vector_type(16 / sizeof(H)))); };
// A row . 4 consecutive B rows over K elements (a multiple of 16 bytes), one wave, 16 bytes a lane; the
// sums are in every lane.
template <class H>
__device__ __forceinline__ void seed_dot(const H* ah, const H* al, const H* bh, const H* bl, long long ld, int K, int lane,
                                         float (&out)[4])
{
    typedef typename Vec16<H>::type v16;
    constexpr int E = 16 / sizeof(H);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k = lane; k < K / E; k += 64) {
        const v16 a = reinterpret_cast<const v16*>(ah)[k], c = al ? reinterpret_cast<const v16*>(al)[k] : v16{};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const v16 b = reinterpret_cast<const v16*>(bh + q * ld)[k];
            const v16 d = bl ? reinterpret_cast<const v16*>(bl + q * ld)[k] : v16{};
#pragma unroll
            for (int e = 0; e < E; e++) acc[q] += ((float)a[e] + (float)c[e]) * ((float)b[e] + (float)d[e]);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) out[q] = wave_sum(acc[q]);
}

template <class H>
__global__ __launch_bounds__(256) void k_prune_seed(BoundsParams p, const float4* __restrict__ pa,
                                                    const float* __restrict__ sb, const H* __restrict__ Ah,
                                                    const H* __restrict__ Al, const float* __restrict__ As,
                                                    const H* __restrict__ Bh, const H* __restrict__ Bl,
                                                    const float* __restrict__ Bs, long long ld, int K,
                                                    const double* __restrict__ Cb, const float* __restrict__ N1,
                                                    long long ldn, const double* __restrict__ prior_o, long long N,
                                                    float* __restrict__ seed, unsigned int* __restrict__ pmin)
{
    __shared__ float sv[256];
    __shared__ int si[256];
    __shared__ float sd[64];
    const int b = blockIdx.x, tid = threadIdx.x, T = p.T, lane = tid & 63;
    const long long bs = (long long)b * p.stride;   // in the batch
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h0 = b * T >> 7, nh = ((b * T + T - 1) >> 7) - h0 + 1;
    const int nscan = (int)((N + 63) / 64);   // blocks with a valid column
    const float sa = pa[b].x;
    float best = 3.0e38f;
    int bi = -1;
    for (int q = tid; q < nh * nscan; q += 256) {
        const int h = h0 + q / nscan, blk = q % nscan;
        const int v = p.lbs[((long long)h * p.S + (b - (h * 128) / T)) * p.nblk + blk];
        const float x = v <= PB_LOW ? -3.0e38f : (float)v * prune_unit(sa, sb[blk]);
        if (x < best) { best = x; bi = q; }
    }
    auto reduce = [&]() {   // the smallest (sv, si) of the workgroup, the first of equals
        __syncthreads();
        sv[tid] = best;
        si[tid] = bi;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (tid < w && (sv[tid + w] < sv[tid] || (sv[tid + w] == sv[tid] && si[tid + w] >= 0 && (si[tid] < 0 || si[tid + w] < si[tid])))) {
                sv[tid] = sv[tid + w];
                si[tid] = si[tid + w];
            }
            __syncthreads();
        }
    };
    reduce();
    const int q0 = si[0];
    float m = 3.0e38f;
    if (q0 >= 0) {
        const int h = h0 + q0 / nscan, blk = q0 % nscan;
        const int ra = max(b * T, h * 128), rb = min(b * T + T, h * 128 + 128);   // at most 128 rows
        // wave w: columns [16 w, 16 w + 16) of the block, fragments straight from memory
        const int fr = lane & 15, fc = lane >> 4;
        const long long n = (long long)blk * 64 + wave * 16 + fr;
        const int bz = p.base[(long long)b * p.ldb + n];
        const v4i* bp = reinterpret_cast<const v4i*>(p.B + n * p.K8) + fc;
        best = 3.0e38f;
        bi = -1;
        for (int r0 = ra; r0 < rb; r0 += 64) {
            v4i acc[4];
            const v4i* ap[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                acc[i] = v4i{0, 0, 0, 0};
                ap[i] = reinterpret_cast<const v4i*>(p.A + (long long)min(r0 + i * 16 + fr, rb - 1) * p.K8) + fc;
            }
#pragma unroll 4
            for (int k = 0; k < p.K8 / 64; k++) {
                const v4i bv = bp[4 * k];
#pragma unroll
                for (int i = 0; i < 4; i++) acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ap[i][4 * k], bv, acc[i], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int r = r0 + i * 16 + fc * 4 + e;
                    const float x = (float)(bz - acc[i][e]);
                    if (r < rb && x < best) { best = x; bi = r; }
                }
        }
        reduce();
        const long long r = max(si[0], ra) + (bs - b) * T;   // the batch's row
        for (int c0 = wave * 16; c0 < wave * 16 + 16; c0 += 4) {   // (rows beyond N are zero, in memory)
            const long long n0 = (long long)blk * 64 + c0;
            float acc[4];
            seed_dot<H>(Ah + r * ld, Al ? Al + r * ld : nullptr, Bh + n0 * ld, Bl ? Bl + n0 * ld : nullptr, ld, K, lane, acc);
            if (lane < 4) {
                const long long nc = n0 + lane;
                const float dot = lane == 0 ? acc[0] : (lane == 1 ? acc[1] : (lane == 2 ? acc[2] : acc[3]));
                float d = 3.0e38f;
                if (nc < N && prior_o[nc] > 0.) {
                    const float v = dot * (As ? As[r] : 1.f) * (Bs ? Bs[nc] : 1.f);
                    d = (float)(Cb[bs] + (double)N1[bs * ldn + nc] - (double)v);
                }
                sd[c0 + lane] = d;
            }
        }
        __syncthreads();
        if (tid == 0)
            for (int k = 0; k < 64; k++) m = fminf(m, sd[k]);
    }
    if (tid == 0) {
        const float sdv = m < 3.0e38f ? m + 1.f + 1e-4f * fabsf(m) : __builtin_inff();
        seed[b] = sdv;
        pmin[bs] = float_to_ordered(sdv);
    }
}

// The tiles of the full GEMM that have to be computed: those with a (particle, block) whose bound is
// not more than the negligible-weight cut (60, plus 1 for rounding) above the particle's seed. Appended to list (indices tm * tiles_n + tn) in about
// the order of the GEMM's tile walk (groups of 64 tile rows). One thread per tile.
__global__ __launch_bounds__(256) void k_prune_plan(BoundsParams p, const float4* __restrict__ pa,
                                                    const float* __restrict__ sb, const double* __restrict__ Cb,
                                                    const float* __restrict__ seed, int tiles_m, int tiles_n,
                                                    unsigned* __restrict__ list, unsigned* __restrict__ count)
{
    static_assert(PRUNED_TILE == 128, "a tile holds one row half tile of the bounds and two blocks");
    const unsigned q = blockIdx.x * 256u + threadIdx.x;
    const unsigned nt = (unsigned)tiles_m * (unsigned)tiles_n;
    bool keep = q < nt;
    unsigned tile = 0;
    if (keep) {
        const unsigned pg = 64u * (unsigned)tiles_n, g = q / pg, r = q - g * pg;
        const unsigned gs = min((unsigned)tiles_m - g * 64u, 64u);
        const int tm = (int)(g * 64u + r % gs), tn = (int)(r / gs);
        tile = (unsigned)tm * (unsigned)tiles_n + (unsigned)tn;
        keep = false;
        const int r0 = tm * 128, r1 = min(r0 + 128, p.M);
        const int z0 = r0 / p.T, z1 = r0 < r1 ? (r1 - 1) / p.T : z0 - 1;
        for (int z = z0; z <= z1 && !keep; z++) {
            const double lim = (double)seed[z] + 61. - Cb[(long long)z * p.stride];
            const float sa = pa[z].x;
            const int* v = p.lbs + ((long long)tm * p.S + (z - z0)) * p.nblk + tn * 2;
#pragma unroll
            for (int k = 0; k < 2; k++)
                if (v[k] <= PB_LOW || !((double)v[k] * (double)prune_unit(sa, sb[tn * 2 + k]) > lim)) keep = true;
        }
    }
    const unsigned long long mask = __ballot(keep);
    if (mask == 0ull) return;
    const int lane = threadIdx.x & 63;
    unsigned base = 0;
    if (lane == 0) base = atomicAdd(count, (unsigned)__popcll(mask));
    base = __shfl(base, 0);
    if (keep) list[base + __popcll(mask & ((1ull << lane) - 1ull))] = tile;
}

// ------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------

int prune_prepare_refs(Device* d, long long O_all, long long O_pad, int Kc, int Kn, int n_low, int K8, hipStream_t st)
{
    PruneBufs& q = d->prune;
    T2X_TRY(q.w.ensure(sizeof(float) * (2 + PP_PARTS) * n_low));
    T2X_TRY(q.B8.ensure((size_t)O_pad * K8));
    T2X_TRY(q.sb.ensure(sizeof(float) * (O_pad / 64)));
    T2X_TRY(q.nb.ensure(sizeof(float2) * O_pad));
    float* w = q.w.as<float>();
    float* parts = w + 2 * n_low;
    k_prune_power<<<dim3((unsigned)((n_low + 63) / 64), PP_PARTS), 256, 0, st>>>(d->coarse_B2.as<float>(), Kn, O_all, n_low,
                                                                                parts);
    k_prune_weights<<<1, 1024, 0, st>>>(n_low, parts, w, w + n_low);
    k_prune_quant_b<<<(unsigned)(O_pad / 64), 1024, 0, st>>>(d->coarse_B.as<float>(), Kc, O_all, n_low, K8, w + n_low,
                                                           q.B8.as<signed char>(), q.sb.as<float>(), q.nb.as<float2>());
    T2X_HIP(hipGetLastError());
    return T2X_OK;
}

int prune_high(Device* d, const PruneCall& c, const PartScalars* d_ps, const PassTables& tc, hipStream_t st)
{
    k_prune_high<<<(unsigned)c.B, 256, 0, st>>>(d_ps, c.stride, d->A1.as<float>(), c.Kn, d->coarse_B2.as<float>(), c.Kn,
                                               c.O_all, c.n_low, tc.npix, d->prior_o.as<double>(),
                                               d->prune.cnt.as<unsigned>() + 1);
    T2X_HIP(hipGetLastError());
    return T2X_OK;
}

int prune_bounds(Device* d, const PruneCall& c, const PartScalars* d_ps, const PassTables& tc, int Pw, hipStream_t st)
{
    PruneBufs& q = d->prune;
    const int nblk = (int)(c.O_pad / 64), S = 127 / c.T + 2;
    const long long M = (long long)c.B * c.T;
    if (c.K8 % 128 != 0 || c.M_pad % 256 != 0 || c.O_pad % 256 != 0 || c.n_low * 2 > c.K8 || c.K8 > 16384) {
        set_error("prune: operands not padded to tile multiples");
        return T2X_EINVAL;
    }
    const int tm = (int)(c.M_pad / 256), tn = (int)(c.O_pad / 256);
    if ((long long)tm * tn > 0x3fffffffLL || c.M_pad > 0x7fffffffLL) { set_error("prune: grid too large"); return T2X_EINVAL; }
    T2X_TRY(q.A8.ensure((size_t)c.M_pad * c.K8));
    T2X_TRY(q.pa.ensure(sizeof(float4) * c.B));
    T2X_TRY(q.base.ensure(sizeof(int) * c.B * c.O_pad));
    T2X_TRY(q.lbs.ensure(sizeof(int) * (c.M_pad / 128) * S * nblk));
    T2X_TRY(q.seed.ensure(sizeof(float) * c.B));
    float* w = q.w.as<float>();
    k_prune_quant_a<<<(unsigned)c.B, c.B < d->n_cu ? 1024 : 256, sizeof(float2) * c.n_low, st>>>(
        d->Fimg_cur.as<float2>(), d->Fctf_cur.as<float>(), Pw, tc.d_win.as<int>(), tc.d_minv.as<float>(), tc.npix, d_ps,
        c.stride, d->ab_coarse.as<float2>(), c.T, c.n_low, c.K8, w, q.A8.as<signed char>(), q.pa.as<float4>());
    const int bm = (c.B + 127) / 128;
    k_prune_base<<<(unsigned)(bm * (c.O_pad / 128)), 256, 0, st>>>(
        d_ps, c.B, c.stride, d->N1.as<float>(), c.O_pad, d->A1.as<float>(), c.Kn, d->coarse_B2.as<float>(), c.Kn, c.O_all,
        c.n_low, c.Kn, q.pa.as<float4>(), q.sb.as<float>(), q.nb.as<float2>(), d->prior_o.as<double>(), bm, q.base.as<int>());
    BoundsParams p{};
    p.A = q.A8.as<signed char>();
    p.B = q.B8.as<signed char>();
    p.K8 = c.K8;
    p.M = (int)M;
    p.T = c.T;
    p.tiles_m = tm;
    p.tiles_n = tn;
    p.base = q.base.as<int>();
    p.ldb = c.O_pad;
    p.lbs = q.lbs.as<int>();
    p.nblk = nblk;
    p.S = S;
    p.nb_part = c.B;
    p.stride = c.stride;
    const unsigned grid = (unsigned)std::min<long long>(d->n_cu, (long long)tm * tn);
    // particles a 256-row tile can hold: ceil(255 / T) + 1
    const int slots = (254 + c.T) / c.T + 1;
    if (slots <= 8) k_gemm_i8_bounds<1><<<grid, 512, 0, st>>>(p);
    else if (slots <= 24) k_gemm_i8_bounds<3><<<grid, 512, 0, st>>>(p);
    else k_gemm_i8_bounds<0><<<grid, 512, 0, st>>>(p);
    T2X_HIP(hipGetLastError());
    // seeds, then the full GEMM's tiles
    const double* Cb = c.Cb;
    const int Kc = 2 * c.Kn;
    if (c.prec == T2X_PREC_FP32)
        k_prune_seed<float><<<(unsigned)c.B, 256, 0, st>>>(
            p, q.pa.as<float4>(), q.sb.as<float>(), d->A.as<float>(), nullptr, nullptr, d->coarse_B.as<float>(), nullptr,
            nullptr, Kc, Kc, Cb, d->N1.as<float>(), c.O_pad, d->prior_o.as<double>(), c.O_all, q.seed.as<float>(),
            d->pmin.as<unsigned>());
    else if (c.prec == T2X_PREC_BF16X3)
        k_prune_seed<__bf16><<<(unsigned)c.B, 256, 0, st>>>(
            p, q.pa.as<float4>(), q.sb.as<float>(), (const __bf16*)d->Ah.ptr, (const __bf16*)d->Al.ptr, d->As.as<float>(),
            (const __bf16*)d->coarse_Bh.ptr, (const __bf16*)d->coarse_Bl.ptr, d->coarse_Bs.as<float>(), Kc, Kc, Cb,
            d->N1.as<float>(), c.O_pad, d->prior_o.as<double>(), c.O_all, q.seed.as<float>(), d->pmin.as<unsigned>());
    else
        k_prune_seed<_Float16><<<(unsigned)c.B, 256, 0, st>>>(
            p, q.pa.as<float4>(), q.sb.as<float>(), (const _Float16*)d->Ah.ptr, (const _Float16*)d->Al.ptr,
            d->As.as<float>(), (const _Float16*)d->coarse_Bh.ptr,
            c.prec == T2X_PREC_FP16X2 ? nullptr : (const _Float16*)d->coarse_Bl.ptr, d->coarse_Bs.as<float>(), Kc, Kc, Cb,
            d->N1.as<float>(), c.O_pad, d->prior_o.as<double>(), c.O_all, q.seed.as<float>(), d->pmin.as<unsigned>());
    const int ptm = (int)(c.M_pad / PRUNED_TILE), ptn = (int)(c.O_pad / PRUNED_TILE);
    T2X_TRY(q.list.ensure(sizeof(unsigned) * (size_t)ptm * ptn));
    k_prune_plan<<<(unsigned)(((long long)ptm * ptn + 255) / 256), 256, 0, st>>>(
        p, q.pa.as<float4>(), q.sb.as<float>(), Cb, q.seed.as<float>(), ptm, ptn, q.list.as<unsigned>(),
        q.cnt.as<unsigned>());
    T2X_HIP(hipGetLastError());
    return T2X_OK;
}

}  // namespace t2x
