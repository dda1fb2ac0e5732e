// diff.hip -- differentiation form: the filter / complex-cell / end-stop / inhibition chain
// on float images, and its hand-written adjoint.
//
// Forward (per scale, per image; FP32): level image L (float pyramid), padded image
//   Pd = s * pad(L)                                 (clamp padding, convolutionFFT2D.cuh:56-85)
//   Z_o = IFFT(FFT(Pd) * Qhat_o) / N,  Qhat_o = FFT(pad(Ke_o + i*Ko_o))   (cuda_bimp.cu:486-507)
//   C_o = |Z_o|,  D = end-stop - inhibition          (cuda_bimp.cuh:436-517)
// Adjoint, for an upstream gradient gD of D:
//   gC_o from the stencil masks (two deterministic passes, no atomics),
//   gZ_o = gC_o * Z_o / |Z_o|,  Ghat_o = FFT(gZ_o),
//   gPd  = Re IFFT(sum_o conj(Qhat_o) * Ghat_o) / N,
//   Y_o  = IFFT(Ghat_o * conj(FFT(Pd))) / N = dL/dKe_o + i dL/dKo_o at the tap positions,
//   then gL = s * pad^T(gPd) and the float-pyramid adjoint down to the image.
// All transforms are full complex 2D FFTs.  The backward keeps spectra kx-major (a column's FH
// values contiguous), so that column transforms read D and Q straight into registers, and what
// passes between row and column transforms in blocks of kb columns (kb * rows contiguous).
// Everything elementwise rides in a transform's load or store: eight launches per group of
// scales and images (k_pad_rows .. k_img_rows), besides the tap rows and their sums.
#include <hip/hip_runtime.h>

#include <utility>

#include "diff.hpp"
#include "fft_device.hpp"

namespace bimpk {

namespace {

using bimpdev::FFTCfg;
using bimpdev::in_index;
using bimpdev::out_index;

constexpr int kRowThreads = 256;

// A thread's group of TPV lanes in its workgroup: one wavefront or two share it from 64 lanes
// on, so it (and every row index and pointer made from it) stays in scalar registers there.
template <int TPV>
__device__ __forceinline__ int group_of(int tid) {
    return TPV >= 64 ? __builtin_amdgcn_readfirstlane(tid / TPV) : tid / TPV;
}

// A transform's results made opaque: what is done with them next would otherwise change how the
// compiler contracts the transform's last additions, and with that the bits of a spectrum.
template <int E>
__device__ __forceinline__ void pin(float2 (&v)[E]) {
#pragma unroll
    for (int e = 0; e < E; ++e) asm volatile("" : "+v"(v[e].x), "+v"(v[e].y));
}

// Column kernels: a workgroup owns CB adjacent columns, one group of TPV lanes each; a column
// stages through LDS with stride S (2 (mod 16) complex spreads the staging accesses).
template <int N>
struct ACfg {
    static constexpr int TPV = FFTCfg<N>::TPV, E = FFTCfg<N>::E;
    static constexpr int CB = diff_block_columns(N);
    static constexpr int THREADS = CB * TPV;
    static constexpr int S = N + 2;
    static constexpr int LDS = CB * S * (int)sizeof(float2);
};

// Columns of `maps` row-major maps of H x W into kx-major spectra of FH x W: row y of the
// transform reads row y of the map, rows [H, H+k) its last row and later ones row 0 (the clamp
// padding).  One entry of `k` per scale of the group.
template <int N>
__global__ void __launch_bounds__(ACfg<N>::THREADS) k_cols_kx(const float2* __restrict__ in, int H,
                                                               int W, AdjInts k, int nscales,
                                                               float2* __restrict__ out,
                                                               const float2* __restrict__ tw) {
    using A = ACfg<N>;
    extern __shared__ float2 lds2[];
    const int map = blockIdx.y, kX = k.v[map % nscales];
    const float2* src = in + (size_t)map * H * W;
    const int c0 = blockIdx.x * A::CB, b = threadIdx.x % A::CB, y0 = threadIdx.x / A::CB;
    float2 v[A::E];
#pragma unroll
    for (int i = 0; i < A::E; ++i) {
        const int y = y0 + i * A::TPV;
        const int ry = y < H ? y : (y < H + kX ? H - 1 : 0);
        v[i] = src[(size_t)ry * W + c0 + b];
    }
#pragma unroll
    for (int i = 0; i < A::E; ++i) lds2[b * A::S + y0 + i * A::TPV] = v[i];
    __syncthreads();
    const int g = group_of<A::TPV>(threadIdx.x), lane = threadIdx.x % A::TPV;
    float2* my = lds2 + (size_t)g * A::S;
#pragma unroll
    for (int e = 0; e < A::E; ++e) v[e] = my[in_index<N>(e, lane)];
    bimpdev::stage_sync<A::TPV>();
    bimpdev::fft<N, false>(v, reinterpret_cast<float*>(my), lane, tw);
    float2* dst = out + ((size_t)map * W + c0 + g) * N;
#pragma unroll
    for (int e = 0; e < A::E; ++e) dst[out_index<N>(e, lane)] = v[e];
}

__device__ __forceinline__ int reflect101(int t, int n) {
    if (t < 0) t = -t;
    if (t >= n) t = 2 * (n - 1) - t;
    return t;
}

// Float pyramid level (the 5x5 binomial / 256 of pyrDown with reflect-101 borders, no rounding).
// blockIdx.z: image of the batch (levels of one size back to back)
__global__ void k_pyr_down_f(const float* __restrict__ src, int sw, int sh,
                             float* __restrict__ dst, int dw, int dh) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (x >= dw) return;
    src += (size_t)blockIdx.z * sw * sh;
    dst += (size_t)blockIdx.z * dw * dh;
    const float k[5] = {1.f, 4.f, 6.f, 4.f, 1.f};
    float acc = 0.f;
    for (int i = -2; i <= 2; ++i) {
        const float* row = src + (size_t)reflect101(2 * y + i, sh) * sw;
        float r = 0.f;
        for (int j = -2; j <= 2; ++j) r += k[j + 2] * row[reflect101(2 * x + j, sw)];
        acc += k[i + 2] * r;
    }
    dst[(size_t)y * dw + x] = acc * (1.f / 256.f);
}

// Weights of the pyramid's 1D stencil seen from source index p: every (d, w) with
// src index p receiving weight w/16 from destination d.  Preimages of p under reflect-101
// are p, -p (p > 0) and 2(n-1) - p (p < n-1).
__device__ __forceinline__ int pyr_taps(int p, int n, int dn, int* d, float* w) {
    const float k[5] = {1.f, 4.f, 6.f, 4.f, 1.f};
    int cnt = 0;
    int pre[3], np = 0;
    pre[np++] = p;
    if (p > 0) pre[np++] = -p;
    if (p < n - 1) pre[np++] = 2 * (n - 1) - p;
    for (int a = 0; a < np; ++a) {
        const int t = pre[a];
        for (int i = -2; i <= 2; ++i) {
            const int q = t - i;
            if (q & 1) continue;
            const int dd = q / 2;
            if (dd < 0 || dd >= dn) continue;
            d[cnt] = dd;
            w[cnt] = k[i + 2] * (1.f / 16.f);
            ++cnt;
        }
    }
    return cnt;
}

// gsrc += pyrDown^T(gdst)
__global__ void k_pyr_down_adj(const float* __restrict__ gdst, int dw, int dh,
                               float* __restrict__ gsrc, int sw, int sh) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y;
    if (x >= sw) return;
    gdst += (size_t)blockIdx.z * dw * dh;
    gsrc += (size_t)blockIdx.z * sw * sh;
    int dy[9], dx[9];
    float wy[9], wx[9];
    const int ny = pyr_taps(y, sh, dh, dy, wy);
    const int nx = pyr_taps(x, sw, dw, dx, wx);
    float acc = 0.f;
    for (int a = 0; a < ny; ++a) {
        float r = 0.f;
        for (int b = 0; b < nx; ++b) r += wx[b] * gdst[(size_t)dy[a] * dw + dx[b]];
        acc += wy[a] * r;
    }
    gsrc[(size_t)y * sw + x] += acc;
}

// ---------------------------------------------------------------- bank of the parameters
// Taps of the quadrature kernels and their derivatives for one (scale, orientation) per
// workgroup, by the formulas of the detection path's FP32 taps (cuda_bimp.cu:304-331: FP32
// expressions around FP64 exp and cos, a sequential FP32 sum of the even taps) and their FP64
// derivatives, operation for operation as the host evaluates them, with no contraction.  The
// three sums run in tap order, each on a wavefront of its own over the chunk in LDS.  Bound by
// FP64 exp and cos; on one host thread the taps of eight scales took 4 ms per parameter change.
struct TapVals {
    float e, ko;             // even tap before its DC offset, odd tap
    double der, deg, dor, dog;  // derivatives by sigma ratio and gamma (even: before their DC)
};
__device__ TapVals tap_at(const TapScale& t, const TapTrig& g, int o, float gamma, int row,
                          int col) {
#pragma clang fp contract(off)
    const float phi = (float)(-3.1415926535897932384626433832795 / 2);
    const int x = col - t.kX, y = row - t.kX;
    const float xr = (float)x * g.ct[o] + (float)y * g.st[o];
    const float yr = (float)y * g.ct[o] - (float)x * g.st[o];
    const float q = xr * xr + gamma * yr * yr;
    const float env = (float)exp((double)(t.negInv * q));
    const double f = 2 * 3.1415926535897932384626433832795 * (double)xr / (double)t.lambda;
    TapVals v;
    v.e = (float)((double)env * cos(f));
    v.ko = (float)((double)env * cos(f + (double)phi));
    const double xd = x, yd = y;
    const double xrd = xd * g.ctd[o] + yd * g.std[o], yrd = yd * g.ctd[o] - xd * g.std[o];
    const double qd = xrd * xrd + (double)gamma * yrd * yrd;
    const double sg = t.sigma;
    const double envd = exp(-qd / (2 * sg * sg));
    const double fd = 2 * 3.1415926535897932384626433832795 * xrd / (double)t.lambda;
    const double phid = -3.1415926535897932384626433832795 / 2;
    const double dr = envd * qd * (double)t.lambda / (sg * sg * sg);
    const double dg = -envd * yrd * yrd / (2 * sg * sg);
    const double ce = cos(fd), co = cos(fd + phid);
    v.der = dr * ce;
    v.deg = dg * ce;
    v.dor = dr * co;
    v.dog = dg * co;
    return v;
}

constexpr int kTapThreads = 1024;
__global__ void __launch_bounds__(kTapThreads) k_taps(TapSet set, TapTrig trig, float gamma,
                                                      float2* __restrict__ taps, size_t stride) {
#pragma clang fp contract(off)
    __shared__ float ce[kTapThreads];
    __shared__ double cr[kTapThreads], cg[kTapThreads];
    __shared__ double sums[3];
    const int o = blockIdx.x, j = blockIdx.y, tid = threadIdx.x;
    const TapScale& t = set.s[j];
    const int kk = t.kW * t.kW;
    const size_t n = (size_t)kNumOri * kk;
    float2* out = taps + (size_t)j * stride + (size_t)o * kk;
    float* dK = t.dK + (size_t)o * kk;
    float es = 0.f;
    double ds = 0.0;
    for (int m0 = 0; m0 < kk; m0 += kTapThreads) {
        const int m = m0 + tid;
        if (m < kk) {
            const TapVals v = tap_at(t, trig, o, gamma, m / t.kW, m % t.kW);
            out[m] = make_float2(v.e, v.ko);
            dK[1 * n + m] = (float)v.dor;
            dK[3 * n + m] = (float)v.dog;
            ce[tid] = v.e;
            cr[tid] = v.der;
            cg[tid] = v.deg;
        }
        __syncthreads();
        const int c = min(kTapThreads, kk - m0);
        if (tid == 0)
            for (int i = 0; i < c; ++i) es += ce[i];
        else if (tid == 64)
            for (int i = 0; i < c; ++i) ds += cr[i];
        else if (tid == 128)
            for (int i = 0; i < c; ++i) ds += cg[i];
        __syncthreads();
    }
    if (tid == 0) sums[0] = (double)(es / (t.fs * t.fs));
    if (tid == 64) sums[1] = ds / ((double)t.fs * (double)t.fs);
    if (tid == 128) sums[2] = ds / ((double)t.fs * (double)t.fs);
    __syncthreads();
    const float dc = (float)sums[0];
    for (int m = tid; m < kk; m += kTapThreads) {
        const TapVals v = tap_at(t, trig, o, gamma, m / t.kW, m % t.kW);
        out[m].x = v.e - dc;
        dK[0 * n + m] = (float)(v.der - sums[1]);
        dK[2 * n + m] = (float)(v.deg - sums[2]);
    }
}

// Row transforms of the kernels placed on the torus, tap (r, c) at ((r-kX) mod FH,
// (c-kX) mod FW): the kW rows that hold taps (requires kW <= FH, FW).
template <int N>
__global__ void __launch_bounds__(kRowThreads) k_bank_rows(const float2* __restrict__ taps,
                                                           size_t stride, TapSet set, int kwmax,
                                                           int rows, float2* __restrict__ out,
                                                           const float2* __restrict__ tw) {
    using C = FFTCfg<N>;
    constexpr int GPB = kRowThreads / C::TPV;
    extern __shared__ float lds[];
    const int grp = group_of<C::TPV>(threadIdx.x), lane = threadIdx.x % C::TPV;
    const int row = blockIdx.x * GPB + grp;
    const int rr = row < rows ? row : 0, map = rr / kwmax, r = rr % kwmax;
    const TapScale& t = set.s[map / kNumOri];
    const bool act = row < rows && r < t.kW;
    const float2* src = taps + (size_t)(map / kNumOri) * stride +
                        ((size_t)(map % kNumOri) * t.kW + (act ? r : 0)) * t.kW;
    float2 v[C::E];
#pragma unroll
    for (int e = 0; e < C::E; ++e) {
        int c = in_index<N>(e, lane) + t.kX;
        if (c >= N) c -= N;
        v[e] = c < t.kW ? src[c] : make_float2(0.f, 0.f);
    }
    bimpdev::fft<N, false>(v, lds + grp * bimpdev::fft_lds_floats<N>(), lane, tw);
    if (act) {
        float2* p = out + (size_t)row * N;
#pragma unroll
        for (int e = 0; e < C::E; ++e) p[out_index<N>(e, lane)] = v[e];
    }
}

// Column transforms of those rows (zero elsewhere): the spectra Q_o and, for o = 0..4, the
// quadrature bank G_o = Re Q_o / (FH*FW) of the detection path's inverse column pass, both
// kx-major.  blockIdx.x: column block, .y: scale * 8 + orientation.
template <int N>
__global__ void __launch_bounds__(ACfg<N>::THREADS) k_bank_cols(const float2* __restrict__ in,
                                                                TapSet set, int W, int kwmax,
                                                                float invN,
                                                                const float2* __restrict__ tw) {
    using A = ACfg<N>;
    extern __shared__ float2 lds2[];
    const int j = blockIdx.y / kNumOri, o = blockIdx.y % kNumOri;
    const TapScale& t = set.s[j];
    const float2* src = in + (size_t)blockIdx.y * kwmax * W;
    const int c0 = blockIdx.x * A::CB, b = threadIdx.x % A::CB, y0 = threadIdx.x / A::CB;
    float2 v[A::E];
#pragma unroll
    for (int i = 0; i < A::E; ++i) {
        int r = y0 + i * A::TPV + t.kX;
        if (r >= N) r -= N;
        v[i] = r < t.kW ? src[(size_t)r * W + c0 + b] : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int i = 0; i < A::E; ++i) lds2[b * A::S + y0 + i * A::TPV] = v[i];
    __syncthreads();
    const int g = group_of<A::TPV>(threadIdx.x), lane = threadIdx.x % A::TPV;
    float2* my = lds2 + (size_t)g * A::S;
#pragma unroll
    for (int e = 0; e < A::E; ++e) v[e] = my[in_index<N>(e, lane)];
    bimpdev::stage_sync<A::TPV>();
    bimpdev::fft<N, false>(v, reinterpret_cast<float*>(my), lane, tw);
    pin<A::E>(v);
    const size_t at = ((size_t)o * W + c0 + g) * N;
#pragma unroll
    for (int e = 0; e < A::E; ++e) {
        const int ky = out_index<N>(e, lane);
        t.Q[at + ky] = v[e];
        if (o < kUniqueOri) t.G[at + ky] = v[e].x * invN;
    }
}

// ---------------------------------------------------------------- backward pipeline
// The launches below cover the entries of a group, scales of one level and transform size by
// images: entry k = image * nscales + scale (AdjSet), each with its own buffers.

// A product that rounds once: the compiler must not contract it into the additions that the
// following transform starts with, so that a value is the same wherever it is computed.
__device__ __forceinline__ float mul1(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}
__device__ __forceinline__ float2 scale1(float2 a, float s) {
    return make_float2(mul1(a.x, s), mul1(a.y, s));
}
// |z|^2, in the same operations everywhere
__device__ __forceinline__ float norm1(float2 z) { return fmaf(z.x, z.x, mul1(z.y, z.y)); }

__device__ __forceinline__ int clamp_src(int y, int H, int k) { return y < H ? y : (y < H + k ? H - 1 : 0); }

// Row transforms of the padded image's distinct rows y < H: Pd = s * pad(L) as complex, L the
// top-left H x W region of a level image (`pitch` floats per row, images lstride apart).
template <int N>
__global__ void __launch_bounds__(kRowThreads) k_pad_rows(const float* __restrict__ L, int pitch,
                                                          size_t lstride, int H, int W, AdjInts k,
                                                          int nscales, float s, int rows,
                                                          float2* __restrict__ out,
                                                          const float2* __restrict__ tw) {
    using C = FFTCfg<N>;
    constexpr int GPB = kRowThreads / C::TPV;
    extern __shared__ float lds[];
    const int grp = group_of<C::TPV>(threadIdx.x), lane = threadIdx.x % C::TPV;
    // every group transforms (a spare one row 0, unstored): a 128-lane group's stages take
    // the workgroup barrier
    const int row = blockIdx.x * GPB + grp;
    const bool act = row < rows;
    const int r = act ? row : 0, entry = r / H, y = r % H;
    const int kX = k.v[entry % nscales];
    const float* src = L + (entry / nscales) * lstride + (size_t)y * pitch;
    float zero = 0.f;
    asm volatile("" : "+v"(zero));  // a runtime zero: the transform's arithmetic stays general
    float2 v[C::E];
#pragma unroll
    for (int e = 0; e < C::E; ++e)
        v[e] = make_float2(mul1(s, src[clamp_src(in_index<N>(e, lane), W, kX)]), zero);
    bimpdev::fft<N, false>(v, lds + grp * bimpdev::fft_lds_floats<N>(), lane, tw);
    if (act) {
        float2* p = out + (size_t)row * N;
#pragma unroll
        for (int e = 0; e < C::E; ++e) p[out_index<N>(e, lane)] = v[e];
    }
}

// Z_o's columns: inverse column transforms of D * Q_o / (FH*FW), rows y < Hc into the block
// layout of T.  Workgroups are dealt round-robin to the eight XCDs; the numbering gives each
// XCD every eighth column block, its eight orientations back to back (D's columns from L2 after
// the first), then the images of one scale (that XCD's share of Q stays in its L2), then the
// scales: 194 us for 32 entries of 512 x 512 (208 when first measured, against 224 with each
// orientation on one XCD).
template <int N>
__global__ void __launch_bounds__(ACfg<N>::THREADS) k_z_cols(const float2* __restrict__ D,
                                                             AdjSet set, int nb, int W, int Hc,
                                                             float invN, float2* __restrict__ T,
                                                             const float2* __restrict__ tw) {
    using A = ACfg<N>;
    extern __shared__ float2 lds2[];
    const int nblk = W / A::CB, per = (nblk + 7) / 8;
    int i = blockIdx.x / 8;
    const int o = i % kNumOri;
    i /= kNumOri;
    const int blk = (i % per) * 8 + blockIdx.x % 8;
    i /= per;
    if (blk >= nblk) return;  // uniform
    const int entry = (i % nb) * set.n + i / nb;
    const int g = group_of<A::TPV>(threadIdx.x), lane = threadIdx.x % A::TPV;
    const int kx = blk * A::CB + g;
    const float2* d = D + ((size_t)entry * W + kx) * N;
    const float2* q = set.Q[entry % set.n] + ((size_t)o * W + kx) * N;
    float2 v[A::E];
#pragma unroll
    for (int e = 0; e < A::E; ++e) {
        const int i = in_index<N>(e, lane);
        const float2 dv = d[i], qv = q[i];
        v[e] = scale1(make_float2(fmaf(dv.x, qv.x, -mul1(dv.y, qv.y)),
                                  fmaf(dv.y, qv.x, mul1(dv.x, qv.y))), invN);
    }
    float2* my = lds2 + (size_t)g * A::S;
    bimpdev::fft<N, true>(v, reinterpret_cast<float*>(my), lane, tw);
#pragma unroll
    for (int e = 0; e < A::E; ++e) my[out_index<N>(e, lane)] = v[e];
    __syncthreads();
    float2* t = T + (((size_t)entry * kNumOri + o) * W + (size_t)blk * A::CB) * Hc;
    const int b = threadIdx.x % A::CB, y0 = threadIdx.x / A::CB;
#pragma unroll
    for (int i = 0; i < A::E; ++i) {
        const int y = y0 + i * A::TPV;
        if (y < Hc) t[(size_t)y * A::CB + b] = lds2[b * A::S + y];
    }
}

// Element x of row y in the block layout with kb = 2^sh columns per block.
__device__ __forceinline__ size_t blk_at(int x, int y, int rows, int sh) {
    return ((size_t)(x >> sh) * rows + y) << sh | (x & ((1 << sh) - 1));
}

// Inverse row transforms of T's rows: Z (row-major) and C = |Z|.
template <int N>
__global__ void __launch_bounds__(kRowThreads) k_z_rows(const float2* __restrict__ T, int Hc,
                                                        int sh, int rows, float2* __restrict__ Z,
                                                        float* __restrict__ Cm,
                                                        const float2* __restrict__ tw) {
    using C = FFTCfg<N>;
    constexpr int GPB = kRowThreads / C::TPV;
    extern __shared__ float lds[];
    const int grp = group_of<C::TPV>(threadIdx.x), lane = threadIdx.x % C::TPV;
    const int row = blockIdx.x * GPB + grp;
    const bool act = row < rows;
    const int r = act ? row : 0, map = r / Hc, y = r % Hc;
    const float2* t = T + (size_t)map * Hc * N;
    float2 v[C::E];
#pragma unroll
    for (int e = 0; e < C::E; ++e) v[e] = t[blk_at(in_index<N>(e, lane), y, Hc, sh)];
    bimpdev::fft<N, true>(v, lds + grp * bimpdev::fft_lds_floats<N>(), lane, tw);
    pin<C::E>(v);
    if (act) {
        float2* z = Z + (size_t)row * N;
        float* c = Cm + (size_t)row * N;
#pragma unroll
        for (int e = 0; e < C::E; ++e) {
            const int x = out_index<N>(e, lane);
            z[x] = v[e];
            c[x] = sqrtf(norm1(v[e]));
        }
    }
}

__device__ __forceinline__ bool valid(int x, int y, int a, int b, int W, int H) {
    const int aa = a < 0 ? -a : a, bb = b < 0 ? -b : b;
    return 2 * bb <= x && x <= W - 2 * bb && 2 * aa <= y && y <= H - 2 * aa;
}

// Pass 1 of the stencil adjoint: per pixel and orientation, which branches of the forward
// (cuda_bimp.cuh:436-502) are active where the upstream gradient g is nonzero:
//   bit o: ds > 0, bit 8 + o: tangential > 0, bit 16 + o: v2 > 0 and v1 > 0, bit 24 + o: v2 > 0
// stored with g as one 8-byte pair per pixel of H x FW (zero right of the data).  Four
// float masks per pixel and orientation took 16 times the bytes: 92 us to write and 96 us to
// gather from per scale of eight 512 x 512 images, against 55 us here.
// EDGE: pixels near the frame's edge test each orientation's reach and wrap their reads; a
// wavefront whose 64 pixels lie inside every reach does neither.  Bound by instructions: 32
// entries of 512 x 512 and 32 of 256 x 256 took 254 us with the tests everywhere, 212 so.
template <bool EDGE>
__device__ __forceinline__ unsigned branch_bits(const float* __restrict__ C, size_t mp, int P,
                                                int FW, int H, int W, const CellParams& p, int x,
                                                int y) {
    const int g0 = y * FW + x;
    auto cat = [&](const float* m, int idx) {
        if (EDGE) {
            if (idx >= P) idx -= P;
            if (idx < 0) idx += P;
        }
        return m[(unsigned)idx];
    };
    unsigned bits = 0;
#pragma unroll
    for (int o = 0; o < kNumOri; ++o) {
        const float* Co = C + o * mp;
        const float* C2 = C + ((o + kNumOri / 2) % kNumOri) * mp;
        const float c = Co[(unsigned)g0];
        const int a = p.ea[o], b = p.eb[o];
        if (!EDGE || valid(x, y, a, b, W, H)) {
            const int d1 = 2 * b - 2 * a * FW;
            const float v = (float)((double)c - 0.5 * (double)cat(Co, g0 + d1) -
                                    0.5 * (double)cat(Co, g0 - d1));
            if (v > 0.f) bits |= 1u << o;
        }
        const int ia = p.ia[o], ib = p.ib[o];
        if (!EDGE || valid(x, y, ia, ib, W, H)) {
            const float vt = cat(Co, g0 - ia * FW - ib) - c;
            if (vt > 0.f) bits |= 1u << (8 + o);
            const int rr = p.ra[o] * FW + p.rb[o];
            float v1 = c - 16.f * cat(C2, g0 + rr);
            const bool m1 = v1 > 0.f;
            v1 = m1 ? v1 : 0.f;
            const float v2 = v1 + c - 16.f * cat(C2, g0 - rr);
            if (v2 > 0.f) bits |= (1u << (24 + o)) | (m1 ? 1u << (16 + o) : 0u);
        }
    }
    return bits;
}

// blockIdx.z: entry.
__global__ void __launch_bounds__(256) k_branch_bits(const float* __restrict__ C, int Hc, int FH,
                                                     int FW, int H, int W, AdjSet set,
                                                     const float* __restrict__ gD, size_t gstride,
                                                     uint2* __restrict__ out) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, entry = blockIdx.z;
    if (x >= FW) return;
    const int j = entry % set.n;
    const CellParams& p = set.cp[j];
    // complex-cell maps are read with the reference's linear index y*FW + x over the FH x FW
    // array, wrapping past the end (the forward stencil's semantics); they hold Hc rows, which
    // is all that valid pixels reach
    const int P = FH * FW;
    const size_t mp = (size_t)Hc * FW;
    C += (size_t)entry * kNumOri * mp;
    gD += (size_t)(entry / set.n) * gstride + set.resp[j];
    int ra = 0, rb = 0;  // the widest reach (the r taps lie inside the i taps')
#pragma unroll
    for (int o = 0; o < kNumOri; ++o) {
        ra = max(ra, max(abs(p.ea[o]), abs(p.ia[o])));
        rb = max(rb, max(abs(p.eb[o]), abs(p.ib[o])));
    }
    const int xw = __builtin_amdgcn_readfirstlane(x);  // the wavefront's first pixel
    // reads stay in rows 0..H-1 and columns 0..W-1 (a valid pixel may reach row H or column W,
    // one past the data, which wraps where the data fills the padded array)
    const bool inside =
            valid(xw, y, ra, rb, W - 1, H - 1) && valid(xw + 63, y, ra, rb, W - 1, H - 1);
    const float g = x < W ? gD[(size_t)y * W + x] : 0.f;
    unsigned bits = 0;
    if (inside)
        bits = branch_bits<false>(C, mp, P, FW, H, W, p, x, y);
    else if (g != 0.f)
        bits = branch_bits<true>(C, mp, P, FW, H, W, p, x, y);
    out[(size_t)entry * H * FW + y * FW + x] = make_uint2(__float_as_uint(g), g != 0.f ? bits : 0u);
}

// Pass 2, in the load of gZ's row transforms: gathers, for a map position q and orientation o,
// every forward read of C_o(q):
//   D = sum_o relu(C(x) - C(x+d1)/2 - C(x+d2)/2) - sum_o [relu(C(x+t) - C(x)) + R_o(x)],
//   R_o(x) = relu(relu(C_o(x) - 16 C_o'(x+r)) + C_o(x) - 16 C_o'(x-r)), o' = o+4,
// then gZ = gC * Z / |Z| (zero where |Z| = 0) and the forward row transform into T's layout.
// Bound by HBM (Z in, T out: 212 us at the copy rate for four scales of eight 512 x 512 images);
// takes 392 us, of which the gather is about 160.
struct Gather {
    const uint2* gm;  // (g, branch bits), H rows of FW
    int P, HF;        // FH*FW, H*FW
    template <bool CHECK>
    __device__ __forceinline__ uint2 at(int idx) const {
        if (!CHECK) return gm[(unsigned)idx];
        if (idx >= P) idx -= P;
        if (idx < 0) idx += P;
        return idx < HF ? gm[(unsigned)idx] : make_uint2(0u, 0u);
    }
};
__device__ __forceinline__ float pick(uint2 v, int bit) {
    return (v.y >> bit) & 1u ? __uint_as_float(v.x) : 0.f;
}
struct Taps {
    int d1, t, rr, o, op;
};
template <bool CHECK>
__device__ __forceinline__ float gather_gc(const Gather& m, const Taps& k, int q) {
    const uint2 c = m.at<CHECK>(q);
    float acc = pick(c, k.o) - 0.5f * pick(m.at<CHECK>(q - k.d1), k.o) -
                0.5f * pick(m.at<CHECK>(q + k.d1), k.o);
    acc += pick(c, 8 + k.o) - pick(m.at<CHECK>(q - k.t), 8 + k.o);
    acc -= pick(c, 16 + k.o) + pick(c, 24 + k.o);
    // partner terms: C_o is the second map of orientation o' = o + 4 (mod 8)
    acc += 16.f * pick(m.at<CHECK>(q - k.rr), 16 + k.op) +
           16.f * pick(m.at<CHECK>(q + k.rr), 24 + k.op);
    return acc;
}

template <int N>
__global__ void __launch_bounds__(kRowThreads) k_gz_rows(const uint2* __restrict__ gm, int FH,
                                                         int H, int Hc, int sh, AdjSet set,
                                                         int rows, const float2* __restrict__ Z,
                                                         float2* __restrict__ T,
                                                         const float2* __restrict__ tw) {
    using C = FFTCfg<N>;
    constexpr int GPB = kRowThreads / C::TPV;
    extern __shared__ float lds[];
    const int grp = group_of<C::TPV>(threadIdx.x), lane = threadIdx.x % C::TPV;
    const int row = blockIdx.x * GPB + grp;
    const bool act = row < rows;
    const int r = act ? row : 0, map = r / Hc, y = r % Hc;
    const int o = map % kNumOri, entry = map / kNumOri;
    const CellParams& p = set.cp[entry % set.n];
    Taps k;
    k.o = o;
    k.op = (o + kNumOri / 2) % kNumOri;
    k.d1 = -2 * p.ea[o] * N + 2 * p.eb[o];
    k.t = -p.ia[o] * N - p.ib[o];
    k.rr = p.ra[k.op] * N + p.rb[k.op];
    const Gather m{gm + (size_t)entry * H * N, FH * N, H * N};
    const int reach = max(max(abs(k.d1), abs(k.t)), abs(k.rr));
    const float2* z = Z + (size_t)r * N;
    float2 v[C::E];
#pragma unroll
    for (int e = 0; e < C::E; ++e) v[e] = z[in_index<N>(e, lane)];
    auto scale = [&](float2& a, float gc) {
        const float mag = sqrtf(norm1(a));
        a = scale1(a, mag > 0.f ? gc / mag : 0.f);
    };
    // (at most two elements' gathers in flight: all of them would take every register at the
    // longer lengths; 640 x 480: 1160 us with four, 1085 with two)
    if (y * N >= reach && (y + 1) * N + reach <= m.HF) {
#pragma unroll
        for (int e = 0; e < C::E; ++e) {
            if (e % 2 == 0) __builtin_amdgcn_sched_barrier(0);
            scale(v[e], gather_gc<false>(m, k, y * N + in_index<N>(e, lane)));
        }
    } else {
#pragma unroll
        for (int e = 0; e < C::E; ++e) {
            if (e % 2 == 0) __builtin_amdgcn_sched_barrier(0);
            scale(v[e], gather_gc<true>(m, k, y * N + in_index<N>(e, lane)));
        }
    }
    bimpdev::fft<N, false>(v, lds + grp * bimpdev::fft_lds_floats<N>(), lane, tw);
    if (act) {
        float2* t = T + (size_t)map * Hc * N;
#pragma unroll
        for (int e = 0; e < C::E; ++e) t[blk_at(out_index<N>(e, lane), y, Hc, sh)] = v[e];
    }
}

// Register order of a forward transform's result -> order of an inverse transform's input.
template <int N>
__device__ __forceinline__ void to_input_order(float2 (&v)[FFTCfg<N>::E], float2* my, int lane) {
    using R = bimpdev::RadInfo<typename FFTCfg<N>::Rad>;
    if constexpr (R::first != R::last) {
#pragma unroll
        for (int e = 0; e < FFTCfg<N>::E; ++e) my[out_index<N>(e, lane)] = v[e];
        bimpdev::stage_sync<FFTCfg<N>::TPV>();
#pragma unroll
        for (int e = 0; e < FFTCfg<N>::E; ++e) v[e] = my[in_index<N>(e, lane)];
        bimpdev::stage_sync<FFTCfg<N>::TPV>();
    }
}

// All that happens to the gradient spectra Ghat_o of one column block, which never leave the
// chip: for each orientation the columns of T (rows [0, Hc), zero below) are transformed;
// conj(Q_o) Ghat_o adds to the image's spectrum, and Ghat_o conj(D) / (FH*FW) is transformed
// back for its kW tap rows (r - kX) mod FH, the only ones the parameter sums read, into Yc.
// Then the image's columns go back, and the rows the clamp padding repeated fold onto rows
// 0 and H-1 (pad^T in y), so that only H rows remain for the row pass, in block layout in A.
// Bound by the transforms' VALU work and the read of T; 300 us for four scales of eight
// 512 x 512 images.  As separate passes over the eight maps the two transforms, the sum and
// the product took 4 x 142 us.  blockIdx.x: column block.
template <int N>
__global__ void __launch_bounds__(ACfg<N>::THREADS) k_adj_cols(const float2* __restrict__ T,
                                                               const float2* __restrict__ D,
                                                               AdjSet set, int nb, int W, int H,
                                                               int Hc, float invN, int kwmax,
                                                               float2* __restrict__ Yc,
                                                               float2* __restrict__ Aimg,
                                                               float2* __restrict__ sums,
                                                               const float2* __restrict__ tw) {
    using A = ACfg<N>;
    extern __shared__ float2 lds2[];
    // the images of one scale run together and share Q in the L2s
    const int blk = blockIdx.x, j = blockIdx.y / nb, entry = (int)(blockIdx.y % nb) * set.n + j;
    const int kW = set.kW[j], kX = set.kX[j];
    const int g = group_of<A::TPV>(threadIdx.x), lane = threadIdx.x % A::TPV;
    const int b = threadIdx.x % A::CB, y0 = threadIdx.x / A::CB;
    const int kx = blk * A::CB + g;
    const float2* d = D + ((size_t)entry * W + kx) * N;
    float2* my = lds2 + (size_t)g * A::S;
    // The running sum over orientations: in registers up to 16 values per lane; above, in
    // memory (each lane its own elements), since both arrays no longer fit (1536 points: 170
    // registers spilled).
    constexpr bool kRegs = A::E <= 16;
    float2* const sum = sums + ((size_t)entry * W + kx) * N;
    float2 acc[A::E];
#pragma unroll
    for (int e = 0; e < A::E; ++e) acc[e] = make_float2(0.f, 0.f);
#pragma unroll 1
    for (int o = 0; o < kNumOri; ++o) {
        const float2* t = T + (((size_t)entry * kNumOri + o) * W + (size_t)blk * A::CB) * Hc;
        float2 v[A::E];
#pragma unroll
        for (int i = 0; i < A::E; ++i) {
            const int y = y0 + i * A::TPV;
            v[i] = y < Hc ? t[(size_t)y * A::CB + b] : make_float2(0.f, 0.f);
        }
        __syncthreads();  // the tap rows of the orientation before have left the staging region
#pragma unroll
        for (int i = 0; i < A::E; ++i) lds2[b * A::S + y0 + i * A::TPV] = v[i];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < A::E; ++e) v[e] = my[in_index<N>(e, lane)];
        bimpdev::stage_sync<A::TPV>();
        bimpdev::fft<N, false>(v, reinterpret_cast<float*>(my), lane, tw);
        pin<A::E>(v);
        const float2* q = set.Q[j] + ((size_t)o * W + kx) * N;
#pragma unroll
        for (int e = 0; e < A::E; ++e) {
            if (e % 8 == 0) __builtin_amdgcn_sched_barrier(0);  // at most eight loads ahead
            const int i = out_index<N>(e, lane);
            const float2 qv = q[i], dv = d[i], gv = v[e];
            if constexpr (kRegs) {
                acc[e].x += qv.x * gv.x + qv.y * gv.y;
                acc[e].y += qv.x * gv.y - qv.y * gv.x;
            } else {
                float2 a = o ? sum[i] : make_float2(0.f, 0.f);
                a.x += qv.x * gv.x + qv.y * gv.y;
                a.y += qv.x * gv.y - qv.y * gv.x;
                sum[i] = a;
            }
            v[e] = scale1(make_float2(fmaf(gv.x, dv.x, mul1(gv.y, dv.y)),
                                      fmaf(gv.y, dv.x, -mul1(gv.x, dv.y))), invN);
        }
        to_input_order<N>(v, my, lane);
        bimpdev::fft<N, true>(v, reinterpret_cast<float*>(my), lane, tw);
#pragma unroll
        for (int e = 0; e < A::E; ++e) my[out_index<N>(e, lane)] = v[e];
        __syncthreads();
        float2* yc = Yc + ((size_t)entry * kNumOri + o) * kwmax * W + (size_t)blk * A::CB + b;
        for (int r = y0; r < kW; r += A::TPV) {
            const int y = r < kX ? r - kX + N : r - kX;
            yc[(size_t)r * W] = lds2[b * A::S + y];
        }
    }
#pragma unroll
    for (int e = 0; e < A::E; ++e) {
        if constexpr (!kRegs) acc[e] = sum[out_index<N>(e, lane)];
        acc[e] = scale1(acc[e], invN);
    }
    __syncthreads();
    to_input_order<N>(acc, my, lane);
    bimpdev::fft<N, true>(acc, reinterpret_cast<float*>(my), lane, tw);
    // fold: rows [H, H + kX) onto H - 1, rows [H + kX, N) onto 0, summed over the group's lanes
    float2 last = make_float2(0.f, 0.f), first = make_float2(0.f, 0.f);
#pragma unroll
    for (int e = 0; e < A::E; ++e) {
        const int y = out_index<N>(e, lane);
        my[y] = acc[e];
        if (y >= H && y < H + kX) last = bimpdev::cadd(last, acc[e]);
        if (y >= H + kX) first = bimpdev::cadd(first, acc[e]);
    }
    if (H < N) {
        constexpr int WL = A::TPV < 64 ? A::TPV : 64;
#pragma unroll
        for (int sh = WL / 2; sh >= 1; sh >>= 1) {
            last.x += __shfl_xor(last.x, sh, WL);
            last.y += __shfl_xor(last.y, sh, WL);
            first.x += __shfl_xor(first.x, sh, WL);
            first.y += __shfl_xor(first.y, sh, WL);
        }
        // one lane per wavefront of the group adds its share, one wavefront after the other
        for (int wv = 0; wv < A::TPV / WL; ++wv) {
            bimpdev::stage_sync<A::TPV>();
            if (lane == wv * WL) {
                my[H - 1] = bimpdev::cadd(my[H - 1], last);
                my[0] = bimpdev::cadd(my[0], first);
            }
        }
    }
    __syncthreads();
    float2* out = Aimg + ((size_t)entry * W + (size_t)blk * A::CB) * H;
#pragma unroll
    for (int i = 0; i < A::E; ++i) {
        const int y = y0 + i * A::TPV;
        if (y < H) out[(size_t)y * A::CB + b] = lds2[b * A::S + y];
    }
}

// Image gradient of one level row: for each scale of the group the inverse row transform of
// A's row, its real part with the padded columns folded onto columns 0 and W-1 (pad^T in x),
// scaled and added in the scales' order to the level's gradient (`pitch` floats per row, images
// lstride apart), which starts at zero with `fresh`; the columns and rows of the level outside
// the H x W data are then cleared as well.  One group of lanes per (image, row).
template <int N>
__global__ void __launch_bounds__(kRowThreads) k_img_rows(const float2* __restrict__ Aimg, int H,
                                                          int W, int sh, AdjInts k, int nscales,
                                                          int rows, float s, int fresh,
                                                          float* __restrict__ gL, int pitch,
                                                          int lrows, size_t lstride,
                                                          const float2* __restrict__ tw) {
    using C = FFTCfg<N>;
    constexpr int GPB = kRowThreads / C::TPV;
    constexpr int WL = C::TPV < 64 ? C::TPV : 64;
    extern __shared__ float lds[];
    __shared__ float2 part[GPB][2];
    const int grp = group_of<C::TPV>(threadIdx.x), lane = threadIdx.x % C::TPV;
    const int row = blockIdx.x * GPB + grp;
    const bool act = row < rows;
    const int r = act ? row : 0, img = r / H, y = r % H;
    float* g = gL + img * lstride + (size_t)y * pitch;
    float sum[C::E];
#pragma unroll
    for (int e = 0; e < C::E; ++e) {
        const int x = out_index<N>(e, lane);
        sum[e] = !fresh && x < W ? g[x] : 0.f;
    }
#pragma unroll 1
    for (int j = 0; j < nscales; ++j) {
        const float2* a = Aimg + (size_t)(img * nscales + j) * H * N;
        const int kX = k.v[j];
        float2 v[C::E];
#pragma unroll
        for (int e = 0; e < C::E; ++e) v[e] = a[blk_at(in_index<N>(e, lane), y, H, sh)];
        bimpdev::fft<N, true>(v, lds + grp * bimpdev::fft_lds_floats<N>(), lane, tw);
        float last = 0.f, first = 0.f;
        if (W < N) {
#pragma unroll
            for (int e = 0; e < C::E; ++e) {
                const int x = out_index<N>(e, lane);
                if (x >= W && x < W + kX) last += v[e].x;
                if (x >= W + kX) first += v[e].x;
            }
#pragma unroll
            for (int d = WL / 2; d >= 1; d >>= 1) {
                last += __shfl_xor(last, d, WL);
                first += __shfl_xor(first, d, WL);
            }
            if constexpr (C::TPV > 64) {
                __syncthreads();
                if (lane % 64 == 0) part[grp][lane / 64] = make_float2(last, first);
                __syncthreads();
                last = part[grp][0].x + part[grp][1].x;
                first = part[grp][0].y + part[grp][1].y;
            }
        }
#pragma unroll
        for (int e = 0; e < C::E; ++e) {
            const int x = out_index<N>(e, lane);
            float t = v[e].x;
            if (x == W - 1) t += last;
            if (x == 0) t += first;
            sum[e] += s * t;
        }
    }
    if (!act) return;
#pragma unroll
    for (int e = 0; e < C::E; ++e) {
        const int x = out_index<N>(e, lane);
        if (x < W) g[x] = sum[e];
    }
    if (fresh) {
        for (int x = W + lane; x < pitch; x += C::TPV) g[x] = 0.f;
        if (y == H - 1)
            for (int i = lane; i < (lrows - H) * pitch; i += C::TPV) g[pitch + i] = 0.f;
    }
}

// Row transforms of the tap rows: rows r < kW of the 8 x kwmax rows of each entry, in place.
template <int N>
__global__ void __launch_bounds__(kRowThreads) k_tap_rows(float2* __restrict__ Yc, AdjInts kW,
                                                          int nscales, int kwmax, int rows,
                                                          const float2* __restrict__ tw) {
    using C = FFTCfg<N>;
    constexpr int GPB = kRowThreads / C::TPV;
    extern __shared__ float lds[];
    const int grp = group_of<C::TPV>(threadIdx.x), lane = threadIdx.x % C::TPV;
    const int row = blockIdx.x * GPB + grp;
    const int r = row < rows ? row : 0;
    const int entry = r / (kNumOri * kwmax);
    // (a 128-lane group's stages take the workgroup barrier: unused rows are transformed too)
    const bool act = row < rows && r % kwmax < kW.v[entry % nscales];
    float2* p = Yc + (size_t)r * N;
    float2 v[C::E];
#pragma unroll
    for (int e = 0; e < C::E; ++e)
        v[e] = act ? p[in_index<N>(e, lane)] : make_float2(0.f, 0.f);
    bimpdev::fft<N, true>(v, lds + grp * bimpdev::fft_lds_floats<N>(), lane, tw);
    if (act) {
#pragma unroll
        for (int e = 0; e < C::E; ++e) p[out_index<N>(e, lane)] = v[e];
    }
}

// Parameter gradient partials: sum over orientations and taps of
//   Re Y_o(tap) dKe/dtheta + Im Y_o(tap) dKo/dtheta  for theta = (sigma ratio, gamma),
// with Y_o's tap rows in Yc; one pair of partial sums per block (fixed-order tree), summed on
// the host in block order.  blockIdx.y: entry; scale j's partials start at j * jstride.
__global__ void __launch_bounds__(256) k_param_partials(const float2* __restrict__ Yc, AdjSet set,
                                                        int kwmax, int FW,
                                                        float* __restrict__ partials,
                                                        size_t pstride, int jstride) {
    __shared__ float sr[256], sg[256];
    const int entry = blockIdx.y, j = entry % set.n;
    const int kW = set.kW[j], kX = set.kX[j];
    const float* dK = set.dK[j];
    const int n = kNumOri * kW * kW;
    if ((int)blockIdx.x * 256 >= n) return;
    const int i = blockIdx.x * 256 + threadIdx.x;
    Yc += (size_t)entry * kNumOri * kwmax * FW;
    partials += (size_t)(entry / set.n) * pstride + (size_t)j * jstride;
    float vr = 0.f, vg = 0.f;
    if (i < n) {
        const int o = i / (kW * kW), m = i % (kW * kW), r = m / kW, c = m % kW;
        const int x = (c - kX + FW) % FW;
        const float2 v = Yc[((size_t)o * kwmax + r) * FW + x];
        const size_t stride = (size_t)n;
        vr = v.x * dK[0 * stride + i] + v.y * dK[1 * stride + i];
        vg = v.x * dK[2 * stride + i] + v.y * dK[3 * stride + i];
    }
    sr[threadIdx.x] = vr;
    sg[threadIdx.x] = vg;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            sr[threadIdx.x] += sr[threadIdx.x + h];
            sg[threadIdx.x] += sg[threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = sr[0];
        partials[2 * blockIdx.x + 1] = sg[0];
    }
}

__global__ void k_fill(float* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}

inline dim3 ew(size_t n) { return dim3((unsigned)((n + 255) / 256)); }

}  // namespace

// Dynamic LDS of the row kernels (kRowThreads / TPV exchange regions) and column kernels.
template <int N>
constexpr int row_lds() {
    return (kRowThreads / FFTCfg<N>::TPV) * bimpdev::fft_lds_floats<N>() * (int)sizeof(float);
}
template <int N>
int row_blocks(int rows) {
    constexpr int GPB = kRowThreads / FFTCfg<N>::TPV;
    return (rows + GPB - 1) / GPB;
}
int block_shift(int n) {
    int sh = 0;
    while ((1 << sh) < diff_block_columns(n)) ++sh;
    return sh;
}

hipError_t diff_prepare(int n) {
#define X(N)                                                                                 \
    if (n == N) {                                                                            \
        const std::pair<const void*, int> f[] = {                                            \
            {(const void*)k_bank_rows<N>, row_lds<N>()},                                     \
            {(const void*)k_bank_cols<N>, ACfg<N>::LDS},                                     \
            {(const void*)k_pad_rows<N>, row_lds<N>()},                                      \
            {(const void*)k_z_rows<N>, row_lds<N>()},                                        \
            {(const void*)k_gz_rows<N>, row_lds<N>()},                                       \
            {(const void*)k_img_rows<N>, row_lds<N>()},                                      \
            {(const void*)k_tap_rows<N>, row_lds<N>()},                                      \
            {(const void*)k_cols_kx<N>, ACfg<N>::LDS},                                       \
            {(const void*)k_z_cols<N>, ACfg<N>::LDS},                                        \
            {(const void*)k_adj_cols<N>, ACfg<N>::LDS}};                                     \
        hipError_t e = hipSuccess;                                                           \
        for (const auto& k : f)                                                              \
            if (e == hipSuccess)                                                             \
                e = hipFuncSetAttribute(k.first, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                        k.second);                                           \
        return e;                                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_taps(const TapSet& set, const TapTrig& trig, float gamma, float2* taps,
                     size_t stride, hipStream_t s) {
    k_taps<<<dim3(kNumOri, set.n), kTapThreads, 0, s>>>(set, trig, gamma, taps, stride);
    return hipGetLastError();
}

hipError_t diff_bank_rows(const TapSet& set, const float2* taps, size_t stride, int kwmax, int FW,
                          float2* out, const float2* tw, hipStream_t s) {
    const int rows = set.n * kNumOri * kwmax;
#define X(N)                                                                                 \
    if (FW == N) {                                                                           \
        k_bank_rows<N><<<row_blocks<N>(rows), kRowThreads, row_lds<N>(), s>>>(               \
            taps, stride, set, kwmax, rows, out, tw);                                        \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_bank_cols(const TapSet& set, const float2* in, int kwmax, int FH, int FW,
                          float invN, const float2* tw, hipStream_t s) {
#define X(N)                                                                                 \
    if (FH == N) {                                                                           \
        using A = ACfg<N>;                                                                   \
        if (FW % A::CB) return hipErrorInvalidValue;                                         \
        k_bank_cols<N><<<dim3(FW / A::CB, set.n * kNumOri), A::THREADS, A::LDS, s>>>(        \
            in, set, FW, kwmax, invN, tw);                                                   \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_cols_kx(const float2* in, int H, int FH, int W, const AdjInts& k, int nscales,
                        int maps, float2* out, const float2* tw, hipStream_t s) {
#define X(N)                                                                                 \
    if (FH == N) {                                                                           \
        using A = ACfg<N>;                                                                   \
        if (W % A::CB) return hipErrorInvalidValue;                                          \
        k_cols_kx<N><<<dim3(W / A::CB, maps), A::THREADS, A::LDS, s>>>(in, H, W, k, nscales, \
                                                                        out, tw);            \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_pyr_down(const float* src, int sw, int sh, float* dst, int dw, int dh, int nb,
                         hipStream_t s) {
    k_pyr_down_f<<<dim3((dw + 127) / 128, dh, nb), 128, 0, s>>>(src, sw, sh, dst, dw, dh);
    return hipGetLastError();
}

hipError_t diff_pyr_down_adj(const float* gdst, int dw, int dh, float* gsrc, int sw, int sh,
                             int nb, hipStream_t s) {
    k_pyr_down_adj<<<dim3((sw + 127) / 128, sh, nb), 128, 0, s>>>(gdst, dw, dh, gsrc, sw, sh);
    return hipGetLastError();
}

hipError_t diff_backward_rows(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B,
                              const float2* tw, hipStream_t s) {
    const int entries = set.n * L.nb;
    const int prows = entries * L.H;
#define X(N)                                                                                 \
    if (L.FW == N) {                                                                         \
        k_pad_rows<N><<<row_blocks<N>(prows), kRowThreads, row_lds<N>(), s>>>(               \
            L.img, L.pitch, L.lstride, L.H, L.W, set.ints(set.kX), set.n, L.gain, prows, B.T, tw); \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_z_cols(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B, const float2* tw,
                       hipStream_t s) {
#define X(N)                                                                                 \
    if (L.FH == N) {                                                                         \
        using A = ACfg<N>;                                                                   \
        const int per = (L.FW / A::CB + 7) / 8;                                              \
        k_z_cols<N><<<8 * kNumOri * per * set.n * L.nb, A::THREADS, A::LDS, s>>>(            \
            B.D, set, L.nb, L.FW, L.Hc, L.invN, B.T, tw);                                    \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_cells_grad(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B,
                           const float* gD, size_t gstride, const float2* tw, hipStream_t s) {
    const int entries = set.n * L.nb, rows = entries * kNumOri * L.Hc;
    const int sh = block_shift(L.FH);
#define X(N)                                                                                 \
    if (L.FW == N) {                                                                         \
        k_z_rows<N><<<row_blocks<N>(rows), kRowThreads, row_lds<N>(), s>>>(B.T, L.Hc, sh, rows, \
                                                                           B.Z, B.C, tw);    \
        k_branch_bits<<<dim3((N + 255) / 256, L.H, entries), 256, 0, s>>>(                   \
            B.C, L.Hc, L.FH, N, L.H, L.W, set, gD, gstride, B.gm);                           \
        k_gz_rows<N><<<row_blocks<N>(rows), kRowThreads, row_lds<N>(), s>>>(                 \
            B.gm, L.FH, L.H, L.Hc, sh, set, rows, B.Z, B.T, tw);                             \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_adj_cols(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B, int kwmax,
                         const float2* tw, hipStream_t s) {
#define X(N)                                                                                 \
    if (L.FH == N) {                                                                         \
        using A = ACfg<N>;                                                                   \
        k_adj_cols<N><<<dim3(L.FW / A::CB, set.n * L.nb), A::THREADS, A::LDS, s>>>(          \
            B.T, B.D, set, L.nb, L.FW, L.H, L.Hc, L.invN, kwmax, B.Yc, B.A, B.Z, tw);        \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t diff_adj_rows(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B, int kwmax,
                         bool fresh, float* glev, int lrows, float* partials, size_t pstride,
                         int jstride, const float2* tw, hipStream_t s) {
    const int entries = set.n * L.nb, rows = L.nb * L.H, trows = entries * kNumOri * kwmax;
    const int sh = block_shift(L.FH);
#define X(N)                                                                                 \
    if (L.FW == N) {                                                                         \
        k_img_rows<N><<<row_blocks<N>(rows), kRowThreads, row_lds<N>(), s>>>(                \
            B.A, L.H, L.W, sh, set.ints(set.kX), set.n, rows, L.gain, fresh ? 1 : 0, glev,   \
            L.pitch, lrows, L.lstride, tw);                                                  \
        k_tap_rows<N><<<row_blocks<N>(trows), kRowThreads, row_lds<N>(), s>>>(               \
            B.Yc, set.ints(set.kW), set.n, kwmax, trows, tw);                                \
        k_param_partials<<<dim3(diff_param_blocks(kwmax), entries), 256, 0, s>>>(            \
            B.Yc, set, kwmax, N, partials, pstride, jstride);                                \
        return hipGetLastError();                                                            \
    }
    BIMP_FOR_SIZES(X)
#undef X
    return hipErrorInvalidValue;
}

int diff_param_blocks(int kW) { return (kNumOri * kW * kW + 255) / 256; }

hipError_t diff_fill(float* p, size_t n, hipStream_t s) {
    k_fill<<<ew(n), 256, 0, s>>>(p, n);
    return hipGetLastError();
}

}  // namespace bimpk
