// features.hip -- the keypoints' downstream consumers on gfx950: the colour histogram
// descriptor and brute-force two-nearest-neighbour matching with the ratio test.
//
// Reference: Context::getDescriptors (bimp/src/bimp.cpp:32-59) appends a 24-float colour
// histogram (addColorFeatures_kernel, bimp/include/detection/cuda_bimp.cuh:8-71) to each
// keypoint's descriptor; matchContexts / downloadMatches (bimp.cpp:188-240) match two
// descriptor sets with OpenCV's CUDA brute-force matcher (L2, k = 2) and keep a match when
// the best distance is below 0.6 x the second best.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "../../include/bimp_hip.h"

namespace {

// ------------------------------------------------------------------ colour histogram
// One thread per keypoint and channel (a window holds at most (2p)^2 pixels, p =
// (int)(log2(size)/2)).  The histogram arithmetic is the reference's: a channel byte is a signed
// char v, bin k collects 31.875*k < v < 31.875*(k+1), so only bytes 1..127 count (bins 0..3); the
// counts are scaled by 0.5 / (3 * pixels) in double.  Pixels outside the image are skipped (the
// reference's inclusive bounds also read column `width` and row `height`).  Bound by the latency
// of one thread's chain (logarithm, pixels, divisions): 4.9 us for 8000 keypoints, 7.0 us with
// one thread for the three channels.
__global__ void __launch_bounds__(64) k_color_features(const float* __restrict__ kp, int ld, int n,
                                                       const uint8_t* __restrict__ bgr,
                                                       size_t pitch, int width, int height,
                                                       float* __restrict__ desc, int desc_ld) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = e / 3, ch = e - 3 * i;
    if (i >= n) return;
    const float x = kp[i], y = kp[(size_t)ld + i], size = kp[4 * (size_t)ld + i];
    const int cx = (int)x, cy = (int)y;
    const int p = (int)(log2((double)size) / 2.0);
    unsigned cnt[4] = {0};  // bins 0..3 (bins 4..7 cannot be reached)
    int found = 0;
    for (int iy = cy - p; iy < cy + p; ++iy) {
        if (iy < 0 || iy >= height) continue;
        const uint8_t* row = bgr + (size_t)iy * pitch + ch;
        for (int ix = cx - p; ix < cx + p; ++ix) {
            if (ix < 0 || ix >= width) continue;
            found += 3;
            const int v = row[3 * ix];
            // 31.875*k < v < 31.875*(k+1) for integer v in 1..127 is k = (8*v) / 255
            const int bin = v >= 1 && v <= 127 ? (8 * v) / 255 : 4;
#pragma unroll
            for (int k = 0; k < 4; ++k) cnt[k] += bin == k ? 1u : 0u;
        }
    }
    float* d = desc + (size_t)i * desc_ld + 8 * ch;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const double c = k < 4 ? (double)cnt[k < 4 ? k : 0] : 0.0;
        // (0.5 * c) / found, rounded once to float as the reference does
        d[k] = (float)((0.5 * c) / (found * 1.0));
    }
}

// ------------------------------------------------------------------ 2-NN matching
// A workgroup of 16 x 16 threads owns 16R query rows and walks the tiles of 16R train rows of
// its slice of the train set (blockIdx.y); thread (ty, tx) accumulates the R x R squared
// distances of its queries and trains over the dimensions, in order, and keeps the best two
// (distance, index) of each of its queries.  Both tiles pass through LDS kDC dimensions at a
// time, dimension-major, in two buffers: the next piece is loaded into registers while the
// current one is used, one barrier per piece.
//
// Bound: FP32 VALU issue, one subtraction and one fma per query, train and dimension (no packed
// FP32; the matrix cores' |q|^2 + |t|^2 - 2qt would lose the small distances' digits).  A loop of
// nothing but such instructions on registers issues 73 T lanes/s, so 8000 x 8000 x 152 cannot take
// less than 0.27 ms; the kernel's 369 M wavefront instructions would take 0.32 ms and it takes
// 0.43 to 0.46 (boxes differ), with two 16-byte LDS reads per 32 operations beside them.  Before,
// one workgroup walked the whole train set for its 64 queries, in one LDS buffer: 125 workgroups
// for 8000 queries, 3.66 ms; 517 x 433 x 152 took 177 us on 9 workgroups, now 16 us.
constexpr int kDC = 16;

struct Best2 {
    float d0, d1;
    int i0, i1;
};

__device__ __forceinline__ bool before(float d, int i, float e, int j) {
    return d < e || (d == e && (unsigned)i < (unsigned)j);
}

__device__ __forceinline__ void insert(Best2& b, float d, int i) {
    if (before(d, i, b.d0, b.i0)) {
        b.d1 = b.d0;
        b.i1 = b.i0;
        b.d0 = d;
        b.i0 = i;
    } else if (before(d, i, b.d1, b.i1)) {
        b.d1 = d;
        b.i1 = i;
    }
}

// Order-preserving key of a candidate: squared distances are non-negative, so their bits order
// as unsigned integers; the index breaks ties toward the lower one.  No candidate: +inf, ~0.
typedef unsigned long long u64;
constexpr u64 kNoKey = ((u64)0x7f800000u << 32) | 0xffffffffu;
__device__ __forceinline__ u64 key_of(float d, int i) {
    return ((u64)__float_as_uint(d) << 32) | (unsigned)i;
}

// Slices of the train set meet in the outputs: query i's best key sits in its idx2 pair, its
// second best in its dist2 pair (8 bytes each, 8-byte aligned).  The displaced key, or the
// offered one if it does not displace any, goes on to the second slot, so that once all have
// been offered the slots hold the two smallest in any order of arrival.
__device__ __forceinline__ void offer(u64* best, u64* second, u64 k) {
    const u64 old = atomicMin(best, k);
    const u64 rest = old < k ? k : old;
    if (rest < kNoKey) atomicMin(second, rest);
}

__global__ void k_knn2_init(u64* __restrict__ best, u64* __restrict__ second, int nq) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nq) best[i] = second[i] = kNoKey;
}

__global__ void k_knn2_unpack(int* __restrict__ idx2, float* __restrict__ dist2, int nq) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nq) return;
    const u64 a = *reinterpret_cast<const u64*>(idx2 + 2 * (size_t)i);
    const u64 b = *reinterpret_cast<const u64*>(dist2 + 2 * (size_t)i);
    idx2[2 * (size_t)i] = (int)(unsigned)a;
    idx2[2 * (size_t)i + 1] = (int)(unsigned)b;
    dist2[2 * (size_t)i] = sqrtf(__uint_as_float((unsigned)(a >> 32)));
    dist2[2 * (size_t)i + 1] = sqrtf(__uint_as_float((unsigned)(b >> 32)));
}

template <int R>
__device__ __forceinline__ void read_rows(const float* __restrict__ row, int t, float (&v)[R]) {
    if constexpr (R == 2) {
        const float2 a = *reinterpret_cast<const float2*>(row + 2 * t);
        v[0] = a.x;
        v[1] = a.y;
    } else {
        const float4 a = *reinterpret_cast<const float4*>(row + 4 * t);
        v[0] = a.x;
        v[1] = a.y;
        v[2] = a.z;
        v[3] = a.w;
    }
}

// VEC: rows are 16-byte aligned (base and stride), so four dimensions load at once.
// ATOMIC: several slices per query (gridDim.y > 1) meet in the outputs' key slots.
template <int R, bool VEC, bool ATOMIC>
__global__ void __launch_bounds__(256) k_knn2(const float* __restrict__ q, int nq, int qld,
                                              const float* __restrict__ t, int nt, int tld,
                                              int dim, int tiles_per_slice,
                                              int* __restrict__ idx2, float* __restrict__ dist2) {
    constexpr int K = 16 * R, PAD = K + 4;         // PAD = 4 (mod 16) words: the transposing
    constexpr int NV = K * kDC / 4;                // stores spread over the banks
    constexpr int PER = (NV + 255) / 256;          // float4 a thread stages per operand
    __shared__ __align__(16) float qs[2][kDC][PAD];
    __shared__ __align__(16) float ts[2][kDC][PAD];
    const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
    const int q0 = blockIdx.x * K;
    const int ntiles = (nt + K - 1) / K;
    const int tile0 = blockIdx.y * tiles_per_slice;
    const int tile1 = min(ntiles, tile0 + tiles_per_slice);
    const int nc = (dim + kDC - 1) / kDC;
    Best2 b[R];
#pragma unroll
    for (int r = 0; r < R; ++r) b[r] = Best2{INFINITY, INFINITY, -1, -1};

    float4 pq[PER], pt[PER];
    auto load = [&](const float* __restrict__ base, int row, int rows, int ld, int d) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < rows && d < dim) {
            const float* p = base + (size_t)row * ld + d;
            if (VEC && d + 4 <= dim) {
                v = *reinterpret_cast<const float4*>(p);
            } else {
                v.x = p[0];
                if (d + 1 < dim) v.y = p[1];
                if (d + 2 < dim) v.z = p[2];
                if (d + 3 < dim) v.w = p[3];
            }
        }
        return v;
    };
    auto fetch = [&](int tile, int c) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int e = tid + 256 * k, r = e / (kDC / 4), d = c * kDC + 4 * (e % (kDC / 4));
            if (NV % 256 == 0 || e < NV) {
                pq[k] = load(q, q0 + r, nq, qld, d);
                pt[k] = load(t, tile * K + r, nt, tld, d);
            }
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int e = tid + 256 * k, r = e / (kDC / 4), d = 4 * (e % (kDC / 4));
            if (NV % 256 == 0 || e < NV) {
                qs[buf][d][r] = pq[k].x;
                qs[buf][d + 1][r] = pq[k].y;
                qs[buf][d + 2][r] = pq[k].z;
                qs[buf][d + 3][r] = pq[k].w;
                ts[buf][d][r] = pt[k].x;
                ts[buf][d + 1][r] = pt[k].y;
                ts[buf][d + 2][r] = pt[k].z;
                ts[buf][d + 3][r] = pt[k].w;
            }
        }
    };

    float acc[R][R];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < R; ++c) acc[r][c] = 0.f;
    auto step = [&](int buf, int d) {
        float qv[R], tv[R];
        read_rows<R>(qs[buf][d], ty, qv);
        read_rows<R>(ts[buf][d], tx, tv);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < R; ++c) {
                const float df = qv[r] - tv[c];
                acc[r][c] = fmaf(df, df, acc[r][c]);
            }
    };

    if (tile0 < tile1) {
        fetch(tile0, 0);
        put(0);
    }
    __syncthreads();
    int buf = 0;
    for (int tile = tile0; tile < tile1; ++tile) {
        for (int c = 0; c < nc; ++c) {
            const bool more = c + 1 < nc || tile + 1 < tile1;
            if (more) fetch(c + 1 < nc ? tile : tile + 1, c + 1 < nc ? c + 1 : 0);
            if ((c + 1) * kDC <= dim) {
#pragma unroll 4
                for (int d = 0; d < kDC; ++d) step(buf, d);
            } else {
                for (int d = 0; d < dim - c * kDC; ++d) step(buf, d);
            }
            if (more) put(buf ^ 1);  // its readers passed the barrier of the piece before
            __syncthreads();
            buf ^= 1;
        }
#pragma unroll
        for (int c = 0; c < R; ++c) {
            const int ti = tile * K + R * tx + c;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (ti < nt) insert(b[r], acc[r][c], ti);
                acc[r][c] = 0.f;
            }
        }
    }
    // the 16 threads of a query row merge their pairs across lanes (a row's threads are 16
    // consecutive lanes); lane tx = 0 holds the result
#pragma unroll
    for (int r = 0; r < R; ++r) {
        Best2 m = b[r];
#pragma unroll
        for (int sh = 8; sh >= 1; sh >>= 1) {
            const float d0 = __shfl_xor(m.d0, sh, 16), d1 = __shfl_xor(m.d1, sh, 16);
            const int i0 = __shfl_xor(m.i0, sh, 16), i1 = __shfl_xor(m.i1, sh, 16);
            insert(m, d0, i0);
            insert(m, d1, i1);
        }
        const int qi = q0 + R * ty + r;
        if (tx == 0 && qi < nq) {
            int* const oi = idx2 + 2 * (size_t)qi;
            float* const od = dist2 + 2 * (size_t)qi;
            if constexpr (ATOMIC) {
                u64* const best = reinterpret_cast<u64*>(oi);
                u64* const second = reinterpret_cast<u64*>(od);
                if (m.i0 >= 0) offer(best, second, key_of(m.d0, m.i0));
                if (m.i1 >= 0) offer(best, second, key_of(m.d1, m.i1));
            } else {
                oi[0] = m.i0;
                oi[1] = m.i1;
                od[0] = sqrtf(m.d0);
                od[1] = sqrtf(m.d1);
            }
        }
    }
}

// Whether 64-bit minima work on p: memory of the current device.  Host memory that the device can
// write takes plain stores but no such atomics (PCIe carries only add, swap and compare-and-swap),
// and managed or another device's memory is not relied on either.
bool device_atomics(const void* p) {
    int dev = -1;
    hipPointerAttribute_t a{};
    if (hipGetDevice(&dev) != hipSuccess || hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();  // not an address that the runtime knows
        return false;
    }
    return a.type == hipMemoryTypeDevice && !a.isManaged && a.device == dev;
}

template <int R, bool VEC>
void launch_knn2(const float* q, int nq, int qld, const float* t, int nt, int tld, int dim,
                 int* idx2, float* dist2, hipStream_t s) {
    constexpr int K = 16 * R;
    const int ntiles = (nt + K - 1) / K, nqt = (nq + K - 1) / K;
    // One tile per workgroup up to 4096 workgroups, then slices of several tiles (8000 x 8000:
    // 32 slices 465 us, 16 477, 8 519, one 2436; 4000 x 4000: 63 slices 128 us, 8 slices 167;
    // 517 x 433: 14 slices 16 us, one 118).  The outputs hold the slices' keys only where they are
    // 8-byte aligned and in this device's memory; otherwise a query has one slice.
    const bool keys = ntiles > 1 && ((uintptr_t)idx2 | (uintptr_t)dist2) % 8 == 0 &&
                      device_atomics(idx2) && device_atomics(dist2);
    int per = std::max(1, ntiles);
    if (keys) per = std::max(1, (int)(((long)ntiles * nqt + 4095) / 4096));
    // (a grid's y extent is limited to 65535)
    per = std::max(per, (ntiles + 65534) / 65535);
    const dim3 grid(nqt, std::max(1, (ntiles + per - 1) / per));
    if (grid.y > 1) {
        u64 *best = reinterpret_cast<u64*>(idx2), *second = reinterpret_cast<u64*>(dist2);
        k_knn2_init<<<(nq + 255) / 256, 256, 0, s>>>(best, second, nq);
        k_knn2<R, VEC, true><<<grid, 256, 0, s>>>(q, nq, qld, t, nt, tld, dim, per, idx2, dist2);
        k_knn2_unpack<<<(nq + 255) / 256, 256, 0, s>>>(idx2, dist2, nq);
    } else {
        k_knn2<R, VEC, false><<<grid, 256, 0, s>>>(q, nq, qld, t, nt, tld, dim, per, idx2, dist2);
    }
}

template <bool VEC>
void dispatch_knn2(const float* q, int nq, int qld, const float* t, int nt, int tld, int dim,
                   int* idx2, float* dist2, hipStream_t s) {
    // R = 4 where its tiles fill the chip's 256 CUs a few times over (it runs six workgroups
    // per CU), else R = 2, whose tiles are four times as many: 2000 x 2000 x 152 (1024 tiles of
    // 64 x 64) 43 us against 52 us with R = 2, 1000 x 1000 (256 tiles) 30 against 21 us.  R = 8
    // took a tenth longer than R = 4 at 8000 x 8000 (211 VGPRs, two wavefronts per SIMD).
    const long tiles4 = (long)((nq + 63) / 64) * ((nt + 63) / 64);
    if (tiles4 >= 768)
        launch_knn2<4, VEC>(q, nq, qld, t, nt, tld, dim, idx2, dist2, s);
    else
        launch_knn2<2, VEC>(q, nq, qld, t, nt, tld, dim, idx2, dist2, s);
}

}  // namespace

extern "C" {

int bimp_color_features(const float* d_kp, int ld, int n, const uint8_t* d_bgr, size_t bgr_pitch,
                        int width, int height, float* d_desc, int desc_ld, bimp_stream_t stream) {
    if (n < 0 || (n > 0 && (!d_kp || !d_bgr || !d_desc)) || ld < n || desc_ld < BIMP_COLOR_DIMENSIONS ||
        width <= 0 || height <= 0 || bgr_pitch < (size_t)3 * width)
        return BIMP_E_ARG;
    if (n == 0) return BIMP_OK;
    const unsigned blocks = (unsigned)((3 * (long long)n + 63) / 64);
    k_color_features<<<blocks, 64, 0, (hipStream_t)stream>>>(d_kp, ld, n, d_bgr, bgr_pitch, width,
                                                             height, d_desc, desc_ld);
    return hipGetLastError() == hipSuccess ? BIMP_OK : BIMP_E_DEVICE;
}

int bimp_match_knn2(const float* d_query, int nq, int q_ld, const float* d_train, int nt,
                    int t_ld, int dim, int* d_idx2, float* d_dist2, bimp_stream_t stream) {
    if (nq < 0 || nt < 0 || dim <= 0 || q_ld < dim || t_ld < dim ||
        (nq > 0 && (!d_query || !d_idx2 || !d_dist2)) || (nt > 0 && !d_train))
        return BIMP_E_ARG;
    if (nq == 0) return BIMP_OK;
    const bool vec = q_ld % 4 == 0 && t_ld % 4 == 0 &&
                     ((uintptr_t)d_query | (uintptr_t)d_train) % 16 == 0;
    if (vec)
        dispatch_knn2<true>(d_query, nq, q_ld, d_train, nt, t_ld, dim, d_idx2, d_dist2,
                            (hipStream_t)stream);
    else
        dispatch_knn2<false>(d_query, nq, q_ld, d_train, nt, t_ld, dim, d_idx2, d_dist2,
                             (hipStream_t)stream);
    return hipGetLastError() == hipSuccess ? BIMP_OK : BIMP_E_DEVICE;
}

int bimp_ratio_matches(const int* idx2, const float* dist2, int nq, double ratio,
                       bimp_match* out, int cap, int* count) {
    if (nq < 0 || !count || (nq > 0 && (!idx2 || !dist2)) || cap < 0 || (cap > 0 && !out))
        return BIMP_E_ARG;
    int n = 0;
    for (int i = 0; i < nq; ++i) {
        const float d1 = dist2[2 * (size_t)i], d2 = dist2[2 * (size_t)i + 1];
        // downloadMatches (bimp.cpp:228): dist1 < 0.6 * dist2, the product in double
        if (idx2[2 * (size_t)i] >= 0 && (double)d1 < ratio * (double)d2) {
            if (n < cap) out[n] = bimp_match{i, idx2[2 * (size_t)i], 0, d1};
            ++n;
        }
    }
    *count = n;
    return n > cap ? BIMP_W_OVERFLOW : BIMP_OK;
}

}  // extern "C"
