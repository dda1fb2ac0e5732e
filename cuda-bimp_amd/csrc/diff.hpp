// diff.hpp -- launch interface of the differentiation form's kernels (diff.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace bimpk {

// Columns per block of the column kernels and of what they exchange with row kernels.
constexpr int diff_block_columns(int n) { return n <= 2048 ? 8 : 4; }

constexpr int kAdjMax = kMaxBatch;  // scales of one backward group

// One int per scale of a group.
struct AdjInts {
    int v[kAdjMax];
};

// The scales of a backward group: one pyramid level and transform size.  Its launches cover
// n scales x nb images; entry = image * n + scale.
struct AdjSet {
    int n;
    int kX[kAdjMax], kW[kAdjMax];
    const float2* Q[kAdjMax];  // bank spectra, 8 x FW x FH (kx-major)
    const float* dK[kAdjMax];  // tap derivatives
    size_t resp[kAdjMax];      // offset of the scale's D map in a response vector
    CellParams cp[kAdjMax];
    static AdjInts ints(const int (&a)[kAdjMax]) {
        AdjInts r;
        for (int i = 0; i < kAdjMax; ++i) r.v[i] = a[i];
        return r;
    }
};

// Geometry of the group's level and the images in hand (nb of them from img on).
struct AdjLevel {
    int H, W, FH, FW, Hc, nb;
    int pitch;       // floats per row of a level image
    size_t lstride;  // floats from one image of the level to the next
    float gain, invN;
    const float* img;
};

// Work buffers, per entry: D FW x FH and A FW x H complex (kx-major / blocks), T and Z 8 x Hc
// x FW complex (T first holds the H x FW row spectra), C the same in floats, gm H x FW pairs,
// Yc 8 x kwmax x FW complex.
struct AdjBuffers {
    float2 *D, *T, *Z, *A, *Yc;
    float* C;
    uint2* gm;
};

// What the taps of a scale follow from, and where its bank goes.
struct TapScale {
    float lambda, fs, negInv;  // negInv: -1 / (2 sigma^2) as the FP32 taps use it
    double sigma;              // FP64 sigma of the derivatives
    int kW, kX;
    float* dK;                 // 4 x 8 x kW x kW: dKe/dr, dKo/dr, dKe/dg, dKo/dg
    float2* Q;                 // 8 x FW x FH
    float* G;                  // 5 x FW x FH
};
struct TapSet {
    int n;
    TapScale s[kAdjMax];
};
// sine and cosine of the orientations, FP32 (of the FP32 angle) and FP64
struct TapTrig {
    float st[kNumOri], ct[kNumOri];
    double std[kNumOri], ctd[kNumOri];
};

hipError_t diff_prepare(int n);
// bank of the current parameters for one group of scales: taps and tap derivatives, row
// transforms of the kwmax x FW tap rows per scale and orientation, then columns into Q and G
hipError_t diff_taps(const TapSet& set, const TapTrig& trig, float gamma, float2* taps,
                     size_t stride, hipStream_t s);
hipError_t diff_bank_rows(const TapSet& set, const float2* taps, size_t stride, int kwmax, int FW,
                          float2* out, const float2* tw, hipStream_t s);
hipError_t diff_bank_cols(const TapSet& set, const float2* in, int kwmax, int FH, int FW,
                          float invN, const float2* tw, hipStream_t s);
// forward column transforms of H x W maps, clamp-padded to FH rows, into kx-major spectra
hipError_t diff_cols_kx(const float2* in, int H, int FH, int W, const AdjInts& k, int nscales,
                        int maps, float2* out, const float2* tw, hipStream_t s);
hipError_t diff_pyr_down(const float* src, int sw, int sh, float* dst, int dw, int dh, int nb,
                         hipStream_t s);
hipError_t diff_pyr_down_adj(const float* gdst, int dw, int dh, float* gsrc, int sw, int sh,
                             int nb, hipStream_t s);
// backward of one group, in order: padded row transforms into T (then diff_cols_kx from T
// into D), Z's columns, Z's rows with the cells adjoint and gZ's rows, gZ's columns, then the
// image rows into the level's gradient and the parameter partials
hipError_t diff_backward_rows(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B,
                              const float2* tw, hipStream_t s);
hipError_t diff_z_cols(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B, const float2* tw,
                       hipStream_t s);
hipError_t diff_cells_grad(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B,
                           const float* gD, size_t gstride, const float2* tw, hipStream_t s);
hipError_t diff_adj_cols(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B, int kwmax,
                         const float2* tw, hipStream_t s);
hipError_t diff_adj_rows(const AdjSet& set, const AdjLevel& L, const AdjBuffers& B, int kwmax,
                         bool fresh, float* glev, int lrows, float* partials, size_t pstride,
                         int jstride, const float2* tw, hipStream_t s);
int diff_param_blocks(int kW);
hipError_t diff_fill(float* p, size_t n, hipStream_t s);

}  // namespace bimpk
