// surf.hip -- SURF descriptors of given keypoints on gfx950 (the reference computes them with
// OpenCV's cv::cuda::SURF_CUDA on the BIMP keypoints, bimp.cpp:32-59 and :188-199, with
// useProvidedKeypoints, upright off, 64 dimensions).
//
// Restated from the published method (Bay, Ess, Tuytelaars, Van Gool, "Speeded-Up Robust
// Features (SURF)", CVIU 110(3), 2008), not from OpenCV's code; byte parity with OpenCV is
// not pinned.  For a keypoint (x, y, size) the scale is s = 1.2 * size / 9:
//   - Haar wavelet responses come from the integral image: for a half side h, dx is the sum of
//     the h x 2h box right of the sample minus the one left of it, dy the box below minus the
//     box above (pixels outside the frame count as 0);
//   - orientation: samples at (round(x + i*s), round(y + j*s)) for integers i^2 + j^2 <= 36,
//     Haar half side max(1, round(2s)), Gaussian weight exp(-(i^2 + j^2) / 8); the weighted
//     response vectors whose angle falls in a window of pi/3 are summed for 72 window starts
//     (5 degree steps), and the longest sum gives the angle (the first on ties);
//   - descriptor: a 20s x 20s square rotated to that angle, 20 x 20 samples at offsets
//     ((u + 0.5)s, (v + 0.5)s), u, v in [-10, 10), Haar half side max(1, round(s)), responses
//     rotated into the keypoint's frame and weighted by exp(-((u+0.5)^2 + (v+0.5)^2) / 21.78)
//     (sigma 3.3s); each of the 4 x 4 subregions (5 x 5 samples) sums dx, dy, |dx|, |dy|; the
//     64 values are scaled to unit length.
// Rounding of sample positions is half away from zero, evaluated in FP32.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/bimp_hip.h"

namespace {

constexpr int kOriSamples = 113;  // integer (i, j) with i^2 + j^2 <= 36
constexpr int kWindows = 72;
constexpr float kPi = 3.14159265358979323846f;

// ------------------------------------------------------------------ integral image
// II has (H+1) x (W+1) uint32 entries, II[0][*] = II[*][0] = 0, and no workspace beside it, so
// the frame is cut into bands of kBand rows and three launches meet in II itself:
//   k_integral_bands  each band's own integral of its last row, into that row of II;
//   k_integral_scan   those rows summed down the bands: every band's last row is final;
//   k_integral_rows   the other rows, from the last row of the band above.
// The pixels are read twice (they stay in L2) and II written once.  Bound by the launches and
// the chain of loads, scan and store in each (the bytes take 2 us): 18 us at 1920 x 1080, 12 us
// at 640 x 480.  A wavefront per row with a scan per 64 pixels and one thread per column
// walking its 1080 rows on 8 workgroups took 73 us.  Bands of 8 rows took 17 and 13 us.
constexpr int kBand = 4;
constexpr int kIntThreads = 512, kIntPix = 4, kIntChunk = kIntThreads * kIntPix;

// Four pixels of a row from x on, zero past the end; words: rows start 4-byte aligned and hold
// whole words (the pitch's), so that one load takes them.
__device__ __forceinline__ void load4(const uint8_t* __restrict__ row, int x, int W, bool words,
                                      unsigned (&v)[kIntPix]) {
    if (words && x + kIntPix <= W) {
        const unsigned w = *reinterpret_cast<const unsigned*>(row + x);
#pragma unroll
        for (int i = 0; i < kIntPix; ++i) v[i] = (w >> (8 * i)) & 255u;
    } else {
#pragma unroll
        for (int i = 0; i < kIntPix; ++i) v[i] = x + i < W ? row[x + i] : 0u;
    }
}

// Four sums of a row (whose start is only 4-byte aligned) in one store where all are inside.
struct __attribute__((packed, aligned(4))) Sums4 {
    unsigned v[kIntPix];
};
__device__ __forceinline__ void store4(unsigned* __restrict__ row, int x, int W,
                                       const unsigned (&v)[kIntPix]) {
    if (x + kIntPix <= W) {
        Sums4 s;
#pragma unroll
        for (int i = 0; i < kIntPix; ++i) s.v[i] = v[i];
        *reinterpret_cast<Sums4*>(row + x) = s;
    } else {
#pragma unroll
        for (int i = 0; i < kIntPix; ++i)
            if (x + i < W) row[x + i] = v[i];
    }
}

// Inclusive sums along x of ROWS rows of kIntChunk values (v[r]: a thread's four consecutive
// ones), `carry` the sums of the chunks before; all threads of the workgroup call it.
template <int ROWS>
__device__ __forceinline__ void scan_rows(unsigned (&v)[ROWS][kIntPix], unsigned (&carry)[ROWS],
                                          unsigned (*__restrict__ tot)[kIntThreads / 64]) {
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    unsigned t[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
#pragma unroll
        for (int i = 1; i < kIntPix; ++i) v[r][i] += v[r][i - 1];
        t[r] = v[r][kIntPix - 1];
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const unsigned u = __shfl_up(t[r], d, 64);
            if (lane >= d) t[r] += u;
        }
    }
    __syncthreads();  // the chunk before has been read
    if (lane == 63) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) tot[r][wave] = t[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        unsigned before = carry[r] + t[r] - v[r][kIntPix - 1];
#pragma unroll
        for (int w = 0; w < kIntThreads / 64; ++w) {
            if (w < wave) before += tot[r][w];
            carry[r] += tot[r][w];
        }
#pragma unroll
        for (int i = 0; i < kIntPix; ++i) v[r][i] += before;
    }
}

// One workgroup per band: rows b*kBand .. of the frame, the sums into II's last row of the band.
__global__ void __launch_bounds__(kIntThreads) k_integral_bands(const uint8_t* __restrict__ img,
                                                                size_t pitch, int W, int H,
                                                                int words,
                                                                unsigned* __restrict__ ii) {
    __shared__ unsigned tot[1][kIntThreads / 64];
    const int y0 = blockIdx.x * kBand, y1 = min(H, y0 + kBand);
    unsigned* out = ii + (size_t)y1 * (W + 1) + 1;
    unsigned carry[1] = {0};
    for (int x0 = 0; x0 < W; x0 += kIntChunk) {
        const int x = x0 + threadIdx.x * kIntPix;
        unsigned p[kBand][kIntPix], v[1][kIntPix] = {};
#pragma unroll
        for (int r = 0; r < kBand; ++r)
            load4(img + (size_t)min(y0 + r, H - 1) * pitch, x, W, words != 0, p[r]);
#pragma unroll
        for (int r = 0; r < kBand; ++r)
#pragma unroll
            for (int i = 0; i < kIntPix; ++i) v[0][i] += y0 + r < y1 ? p[r][i] : 0u;
        scan_rows<1>(v, carry, tot);
        store4(out, x, W, v[0]);
    }
}

// The bands' last rows summed down the frame, in place: 32 columns by 32 runs of bands per
// workgroup.
__global__ void __launch_bounds__(1024) k_integral_scan(unsigned* __restrict__ ii, int W, int H) {
    __shared__ unsigned part[32][33];
    const int cx = threadIdx.x % 32, seg = threadIdx.x / 32;
    const int x = blockIdx.x * 32 + cx;
    const int nb = (H + kBand - 1) / kBand, per = (nb + 31) / 32;
    const int b0 = min(nb, seg * per), b1 = min(nb, b0 + per);
    const size_t ld = (size_t)W + 1;
    auto at = [&](int b) { return (size_t)min(H, (b + 1) * kBand) * ld + x; };
    unsigned sum = 0;
    if (x <= W && x > 0)
        for (int b = b0; b < b1; ++b) sum += ii[at(b)];
    part[seg][cx] = sum;
    __syncthreads();
    unsigned acc = 0;
    for (int s = 0; s < seg; ++s) acc += part[s][cx];
    if (x > W) return;
    for (int b = b0; b < b1; ++b) {
        acc = x > 0 ? acc + ii[at(b)] : 0u;
        ii[at(b)] = acc;
    }
}

// The other rows of each band (and row 0 of II): sums of the band's rows down to each, along x,
// on top of the last row of the band above.
__global__ void __launch_bounds__(kIntThreads) k_integral_rows(const uint8_t* __restrict__ img,
                                                               size_t pitch, int W, int H,
                                                               int words,
                                                               unsigned* __restrict__ ii) {
    constexpr int R = kBand - 1;
    __shared__ unsigned tot[R][kIntThreads / 64];
    const int band = blockIdx.x, y0 = band * kBand;
    const int rows = min(H, y0 + kBand) - y0 - 1;  // rows of this launch: all but the last
    const size_t ld = (size_t)W + 1;
    const unsigned* top = ii + (size_t)y0 * ld + 1;
    unsigned* out = ii + (size_t)(y0 + 1) * ld + 1;
    if (band == 0)
        for (int x = threadIdx.x; x <= W; x += kIntThreads) ii[x] = 0u;
    if ((int)threadIdx.x < rows) out[(size_t)threadIdx.x * ld - 1] = 0u;
    unsigned carry[R] = {};
    for (int x0 = 0; x0 < W; x0 += kIntChunk) {
        const int x = x0 + threadIdx.x * kIntPix;
        unsigned v[R][kIntPix], t[kIntPix];
#pragma unroll
        for (int r = 0; r < R; ++r)
            load4(img + (size_t)min(y0 + r, H - 1) * pitch, x, W, words != 0, v[r]);
#pragma unroll
        for (int i = 0; i < kIntPix; ++i) t[i] = band > 0 && x + i < W ? top[x + i] : 0u;
#pragma unroll
        for (int r = 1; r < R; ++r)
#pragma unroll
            for (int i = 0; i < kIntPix; ++i) v[r][i] += v[r - 1][i];
        scan_rows<R>(v, carry, tot);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r >= rows) break;
#pragma unroll
            for (int i = 0; i < kIntPix; ++i) v[r][i] += t[i];
            store4(out + (size_t)r * ld, x, W, v[r]);
        }
    }
}

__device__ __forceinline__ int round_away(float v) { return (int)roundf(v); }

// Haar responses of half side h at (px, py): dx = the h x 2h box right of the sample minus the
// one left of it, dy = the box below minus the box above, boxes clipped to the frame.  The four
// boxes share the eight outer points of a 3 x 3 grid (an empty clipped box sums to 0 by itself; so
// that the boxes of a position beyond the integers are empty ones too, the sums saturate).
// OFF: byte offsets from the uniform base, 32 bits for an integral of up to 2^30 entries (all that
// bimp_integral_image makes; a caller's own may be larger).
template <class OFF>
__device__ __forceinline__ void haar(const unsigned* __restrict__ ii, int W, int H, int px, int py,
                                     int h, float* dx, float* dy) {
    auto clip = [](int v, int n) { return min(max(v, 0), n); };
    auto at = [&](OFF o) {
        return *reinterpret_cast<const unsigned*>(reinterpret_cast<const char*>(ii) + o);
    };
    auto lo = [&](int p) { return __builtin_elementwise_sub_sat(p, h); };
    auto hi = [&](int p) { return __builtin_elementwise_add_sat(p, h); };
    const OFF ld = 4 * ((OFF)W + 1);
    const OFF c0 = (OFF)4 * clip(lo(px), W), c1 = (OFF)4 * clip(px, W), c2 = (OFF)4 * clip(hi(px), W);
    const OFF r0 = clip(lo(py), H) * ld, r1 = clip(py, H) * ld, r2 = clip(hi(py), H) * ld;
    const unsigned a00 = at(r0 + c0), a01 = at(r0 + c1), a02 = at(r0 + c2);
    const unsigned a10 = at(r1 + c0), a12 = at(r1 + c2);
    const unsigned a20 = at(r2 + c0), a21 = at(r2 + c1), a22 = at(r2 + c2);
    const int right = (int)(a22 - a02 - a21 + a01), left = (int)(a21 - a01 - a20 + a00);
    const int below = (int)(a22 - a12 - a20 + a10), above = (int)(a12 - a02 - a10 + a00);
    *dx = (float)(right - left);
    *dy = (float)(below - above);
}

// Column counts of the disc's rows: row j = -6 .. 6 holds i = -w .. w.
__device__ __forceinline__ void disc_point(int t, int* i, int* j) {
    constexpr int w[13] = {0, 3, 4, 5, 5, 5, 6, 5, 5, 5, 4, 3, 0};
    int cnt = t, jj = 0;
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        const int n = 2 * w[k] + 1;
        if (jj == k && cnt >= n) {
            cnt -= n;
            jj = k + 1;
        }
    }
    int wj = 0;
#pragma unroll
    for (int k = 0; k < 13; ++k) wj = jj == k ? w[k] : wj;
    *i = cnt - wj;
    *j = jj - 6;
}

// A workgroup describes a few keypoints: their 113 orientation samples each, 72 windows, 400
// descriptor samples and 64 feature sums are dealt to all its threads, and the Gaussian weights,
// the same for every keypoint, are evaluated once.  Bound by VALU work, most of it the windows'
// sums (kept in sample order) and the samples' positions, with the gathers from the integral
// image beside it: 46 us for 8000 keypoints.  One wavefront per keypoint, with the disc's points
// found by a loop of square roots, the windows in one full and one mostly idle round, sixteen
// gathers per sample and an arctangent per improvement of the best window, took 121 us.
template <int KP, int THREADS, int WIN, int HELD, class OFF = unsigned>
struct SurfCfg {
    using off = OFF;
    static constexpr int kp = KP, threads = THREADS;
    static constexpr int win = WIN, per = kWindows / WIN;  // windows per thread, threads
    static constexpr int held = HELD;  // keypoints whose descriptor samples are held at once
    static_assert(KP * per <= THREADS && kWindows % WIN == 0 && KP % HELD == 0, "split");
    static constexpr int buf() {
        const int a = KP * kOriSamples * (int)sizeof(float4), b = HELD * 400 * (int)sizeof(float2);
        return (a > b ? a : b) / (int)sizeof(float4);
    }
};

// An angle lies in a window when its offset d from the window's start, plus 2 pi if negative,
// is below pi/3, all in FP32.  Rounding is monotone, so the negative offsets that pass are those
// up to one value, found here; a non-negative one passes when its bits are below pi/3's.
constexpr float kWindow = kPi / 3.f;
constexpr float last_wrapped() {
    unsigned b = __builtin_bit_cast(unsigned, kWindow - 2.f * kPi) - 64u;  // closer to zero
    while (!(__builtin_bit_cast(float, b) + 2.f * kPi < kWindow)) ++b;     // away from zero
    return __builtin_bit_cast(float, b);
}
constexpr float kWrapped = last_wrapped();
static_assert(kWrapped + 2.f * kPi < kWindow && kWrapped < 0.f, "wrapped offsets");
static_assert(!(__builtin_bit_cast(float, __builtin_bit_cast(unsigned, kWrapped) - 1u) + 2.f * kPi <
                kWindow), "the last one");
__device__ __forceinline__ bool in_window(float d) {
    return __float_as_uint(d) < __builtin_bit_cast(unsigned, kWindow) || d <= kWrapped;
}

template <class S>
__global__ void __launch_bounds__(S::threads) k_surf(const unsigned* __restrict__ ii, int W,
                                                       int H, const float* __restrict__ kp, int ld,
                                                       int n, int upright,
                                                       float* __restrict__ desc, int desc_ld,
                                                       float* __restrict__ angle_out) {
    constexpr int kSamples = 400, kSurfKp = S::kp, kSurfThreads = S::threads;
    constexpr int kWin = S::win, kPer = S::per, kHeld = S::held;
    // orientation samples (weighted response, angle), then the descriptor's (two responses)
    __shared__ float4 buf[S::buf()];
    __shared__ float gd[kSamples];
    __shared__ float4 ori[kOriSamples];  // i, j, weight
    __shared__ float kx[kSurfKp], ky[kSurfKp], ks[kSurfKp], kco[kSurfKp], ksi[kSurfKp], kth[kSurfKp];
    __shared__ unsigned long long best[kSurfKp];
    __shared__ float win[kSurfKp][kWindows][2];
    const int tid = threadIdx.x, k0 = blockIdx.x * kSurfKp;
    if (tid < kSurfKp) {
        const int k = min(k0 + tid, n - 1);
        kx[tid] = kp[k];
        ky[tid] = kp[(size_t)ld + k];
        ks[tid] = 1.2f * kp[4 * (size_t)ld + k] / 9.f;
        best[tid] = 0;
        kth[tid] = 0.f;
    }
    for (int t = tid; t < kSamples; t += kSurfThreads) {
        const int u = t % 20 - 10, v = t / 20 - 10;
        gd[t] = expf(-((u + 0.5f) * (u + 0.5f) + (v + 0.5f) * (v + 0.5f)) / (2.f * 3.3f * 3.3f));
    }
    if (!upright && tid < kOriSamples) {
        int i, j;
        disc_point(tid, &i, &j);
        ori[tid] = make_float4((float)i, (float)j, expf(-(float)(i * i + j * j) / 8.f), 0.f);
    }
    __syncthreads();
    if (!upright) {
        for (int e = tid; e < kSurfKp * kOriSamples; e += kSurfThreads) {
            const int k = e / kOriSamples, t = e - k * kOriSamples;
            const float4 q = ori[t];
            const float s = ks[k];
            float dx, dy;
            haar<typename S::off>(ii, W, H, round_away(kx[k] + q.x * s),
                                  round_away(ky[k] + q.y * s), max(1, round_away(2.f * s)), &dx,
                                  &dy);
            float a = atan2f(dy, dx);
            if (a < 0) a += 2.f * kPi;
            buf[e] = make_float4(q.z * dx, q.z * dy, a, 0.f);
        }
        __syncthreads();
        if (tid < kSurfKp * kPer) {
            const int k = tid / kPer, w0 = tid % kPer;
            float sx[kWin] = {}, sy[kWin] = {}, a0[kWin];
#pragma unroll
            for (int w = 0; w < kWin; ++w)
                a0[w] = (w0 + kPer * w) * (2.f * kPi / kWindows);
            const float4* sm = buf + k * kOriSamples;
#pragma unroll 4
            for (int t = 0; t < kOriSamples; ++t) {
                const float4 q = sm[t];
#pragma unroll
                for (int w = 0; w < kWin; ++w) {
                    const bool in = in_window(q.z - a0[w]);
                    sx[w] += in ? q.x : 0.f;
                    sy[w] += in ? q.y : 0.f;
                }
            }
            // the longest window sum, the first of equal ones (lengths are non-negative, so
            // their bits order them)
            unsigned long long key = 0;
#pragma unroll
            for (int w = 0; w < kWin; ++w) {
                const int wv = w0 + kPer * w;
                win[k][wv][0] = sx[w];
                win[k][wv][1] = sy[w];
                const float m = sx[w] * sx[w] + sy[w] * sy[w];
                const unsigned long long c =
                    ((unsigned long long)__float_as_uint(m) << 32) | (unsigned)(kWindows - wv);
                key = c > key ? c : key;
            }
            atomicMax(&best[k], key);
        }
        __syncthreads();
        if (tid < kSurfKp) {
            const int w = kWindows - (int)(unsigned)best[tid];
            kth[tid] = atan2f(win[tid][w][1], win[tid][w][0]);
        }
        __syncthreads();
    }
    if (tid < kSurfKp) {
        kco[tid] = cosf(kth[tid]);
        ksi[tid] = sinf(kth[tid]);
    }
    __syncthreads();
    float2* smp = reinterpret_cast<float2*>(buf);
#pragma unroll 1
    for (int h0 = 0; h0 < kSurfKp; h0 += kHeld) {
        for (int e = tid; e < kHeld * kSamples; e += kSurfThreads) {
            const int kl = e / kSamples, t = e - kl * kSamples, k = h0 + kl;
            const int u = t % 20 - 10, v = t / 20 - 10;
            const float s = ks[k], co = kco[k], si = ksi[k];
            const float ou = (u + 0.5f) * s, ov = (v + 0.5f) * s;
            const int px = round_away(kx[k] + co * ou - si * ov);
            const int py = round_away(ky[k] + si * ou + co * ov);
            float dx, dy;
            haar<typename S::off>(ii, W, H, px, py, max(1, round_away(s)), &dx, &dy);
            const float g = gd[t];
            smp[e] = make_float2(g * (dx * co + dy * si), g * (-dx * si + dy * co));
        }
        __syncthreads();
        // one wavefront per keypoint: lane l holds feature l % 4 (dx, dy, |dx|, |dy|) of subregion
        // l / 4 (4 x 4, row-major), summed over its 5 x 5 samples in row-major order
        const int lane = tid % 64;
        const int r = lane / 4, q = lane % 4;
        const int u0 = (r % 4) * 5, v0 = (r / 4) * 5;
        for (int kl = tid / 64; kl < kHeld && k0 + h0 + kl < n; kl += kSurfThreads / 64) {
            const int k = h0 + kl;
            const float* f = reinterpret_cast<const float*>(smp + kl * kSamples) + (q & 1);
            float val = 0.f;
#pragma unroll
            for (int vv = 0; vv < 5; ++vv)
#pragma unroll
                for (int uu = 0; uu < 5; ++uu) {
                    const float x = f[2 * ((v0 + vv) * 20 + u0 + uu)];
                    val += q < 2 ? x : fabsf(x);
                }
            float sq = val * val;
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) sq += __shfl_xor(sq, d, 64);
            const float inv = sq > 0.f ? 1.f / sqrtf(sq) : 0.f;
            desc[(size_t)(k0 + k) * desc_ld + lane] = val * inv;
            if (angle_out && lane == 0) angle_out[k0 + k] = kth[k];
        }
        __syncthreads();  // the next keypoints' samples take their place
    }
}

template <class S>
void launch_surf(const unsigned* ii, int W, int H, const float* kp, int ld, int n, int upright,
                 float* desc, int desc_ld, float* angle, hipStream_t s) {
    k_surf<S><<<(n + S::kp - 1) / S::kp, S::threads, 0, s>>>(ii, W, H, kp, ld, n, upright, desc,
                                                             desc_ld, angle);
}

}  // namespace

extern "C" {

int bimp_integral_image(const uint8_t* d_img, size_t pitch, int width, int height,
                        unsigned* d_integral, bimp_stream_t stream) {
    if (!d_img || !d_integral || width <= 0 || height <= 0 || pitch < (size_t)width ||
        (size_t)width * height * 255u > 0x7fffffffu)
        return BIMP_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const int words = ((uintptr_t)d_img | pitch) % 4 == 0 ? 1 : 0;
    const int bands = (height + kBand - 1) / kBand;
    k_integral_bands<<<bands, kIntThreads, 0, s>>>(d_img, pitch, width, height, words, d_integral);
    k_integral_scan<<<(width + 1 + 31) / 32, 1024, 0, s>>>(d_integral, width, height);
    k_integral_rows<<<bands, kIntThreads, 0, s>>>(d_img, pitch, width, height, words, d_integral);
    return hipGetLastError() == hipSuccess ? BIMP_OK : BIMP_E_DEVICE;
}

int bimp_surf_descriptors(const unsigned* d_integral, int width, int height, const float* d_kp,
                          int ld, int n, int upright, float* d_desc, int desc_ld, float* d_angle,
                          bimp_stream_t stream) {
    if (n < 0 || (n > 0 && (!d_integral || !d_kp || !d_desc)) || ld < n || desc_ld < 64 ||
        width <= 0 || height <= 0)
        return BIMP_E_ARG;
    if (n == 0) return BIMP_OK;
    // Long lists share more per workgroup (two windows per thread and one read of a sample for
    // both); short ones need the shorter chain of a workgroup with half the keypoints: 8000
    // keypoints 46 against 51 us, 4000 29.7 against 27.9, 1500 21.7 against 16.6, 60 17.4
    // against 11.9.
    if ((size_t)(width + 1) * (height + 1) > (size_t(1) << 30))
        launch_surf<SurfCfg<2, 256, 1, 2, size_t>>(d_integral, width, height, d_kp, ld, n, upright,
                                                   d_desc, desc_ld, d_angle, (hipStream_t)stream);
    else if (n >= 6000)
        launch_surf<SurfCfg<4, 256, 2, 4>>(d_integral, width, height, d_kp, ld, n, upright, d_desc,
                                           desc_ld, d_angle, (hipStream_t)stream);
    else
        launch_surf<SurfCfg<2, 256, 1, 2>>(d_integral, width, height, d_kp, ld, n, upright, d_desc,
                                           desc_ld, d_angle, (hipStream_t)stream);
    return hipGetLastError() == hipSuccess ? BIMP_OK : BIMP_E_DEVICE;
}

}  // extern "C"
