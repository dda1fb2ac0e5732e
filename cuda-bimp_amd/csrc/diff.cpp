// diff.cpp -- host side of the differentiation form (C ABI bimp_diff_*, include/bimp_hip.h).
//
// A diff context holds, per scale, the bank spectra Qhat_o of the current Gabor parameters
// (sigma ratio, gamma), their real quadrature form G_o and the tap derivatives dK/dtheta; per
// frame it recomputes the complex responses instead of storing them (forward and backward
// each run the filter).  The forward takes the detection path's transforms (two image rows
// per complex row FFT, half spectra, inverse columns with the Hermitian partner, G_o for
// o = 0..4 with 5..7 mirrored); the backward needs Z_o, FFT(Pd) and C_o on the whole periodic
// domain and recomputes them with full complex 2D transforms.  Images are FP32, scaled by
// 255 * input_scale before filtering, so an image u8/255 gives the maps of the uint8 path up
// to the pyramid's rounding.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <string>
#include <vector>

#include "../../include/bimp_hip.h"
#include "bank.hpp"
#include "diff.hpp"

namespace {

using bimpk::kNumOri;

struct DScale {
    bimph::ScaleGeom g;
    bimpk::CellParams cp;
    float2* Q = nullptr;   // 8 x FW x FH bank spectra, kx-major
    float* G = nullptr;    // 5 x FW x FH quadrature bank Re(Q_o) / (FH*FW), kx-major
    int Hc = 0, Wc = 0, ldc = 0;  // complex-cell region of the forward (as in detection)
    float2* DT = nullptr;  // forward: (FW/2+1) x FH half spectrum, column-major, per image
    float* Cf = nullptr;   // forward: 8 x Hc x ldc complex-cell maps, per image
    int nbf = 1;           // forward: images per launch of its group (DT, Cf copies)
    float* dK = nullptr;   // 4 x 8 x kW x kW tap derivatives (dKe/dr, dKo/dr, dKe/dg, dKo/dg)
    size_t respOff = 0;    // offset of this scale's D map in a response vector
};

int round_half_away(double v) { return (int)std::round(v); }

}  // namespace

struct bimp_diff {
    int width = 0, height = 0;
    bimp_options opt{};
    float ratio = 0.f, gamma = 0.f;
    std::vector<DScale> sc;
    size_t respSize = 0;
    int maxLevel = 0;
    std::vector<int> lw, lh;
    std::vector<float*> lev, glev;
    std::map<int, float2*> tw;
    // forward: scales of one level and transform size share each launch (first, count)
    std::vector<std::pair<int, int>> groups;
    float2 *R = nullptr, *T = nullptr;  // forward: row spectra and inverse-column output
    float* Sf = nullptr;                // forward: single-stopped maps (scratch)
    size_t rSize = 0, tSize = 0;
    float2* taps = nullptr;             // (Ke, Ko) of a group being set up, per scale
    size_t tapStride = 0;
    unsigned* maxslot = nullptr;
    // backward: work buffers of up to `entries` (scale, image) pairs per launch
    bimpk::AdjBuffers adj{};
    int entries = 1, kwMax = 0;
    float* partials = nullptr;
    int maxBlocks = 0;
    int nbMax = 8;  // images whose pyramids are held at once
    // the end of the last forward on a stream other than the null stream, recorded there: a
    // parameter change waits for it
    hipEvent_t fwdDone = nullptr;
    bool fwdPending = false;   // fwdDone marks a forward that nothing has waited for
    bool fwdCaptured = false;  // a forward sits in a caller's graph, whose replays mark nothing
    std::string err;
};

namespace {

constexpr size_t kForwardTBytes = 160u << 20;  // T of a forward launch, as in detection

int dfail(bimp_diff* d, int code, const std::string& m) {
    if (d) d->err = m;
    return code;
}

#define DCHK(d, expr)                                                                   \
    do {                                                                                \
        hipError_t e_ = (expr);                                                         \
        if (e_ != hipSuccess)                                                           \
            return dfail(d, BIMP_E_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

// Taps, tap derivatives and bank spectra of (ratio, gamma), on the device.  They replace those
// that a forward reads, so the last one ends first: it may still run on a stream that the null
// stream, which all of this goes to, does not wait for.  A backward has ended when its call
// returns.
int set_params(bimp_diff* d, float ratio, float gamma) {
    const hipStream_t s = nullptr;
    if (d->fwdCaptured)
        DCHK(d, hipDeviceSynchronize());
    else if (d->fwdPending)
        DCHK(d, hipStreamWaitEvent(s, d->fwdDone, 0));
    const double pi = 3.1415926535897932384626433832795;
    bimpk::TapTrig trig;
    for (int o = 0; o < kNumOri; ++o) {
        const float theta = (float)(o * pi / 8);
        trig.st[o] = (float)std::sin((double)theta);
        trig.ct[o] = (float)std::cos((double)theta);
        trig.std[o] = std::sin(o * pi / 8);
        trig.ctd[o] = std::cos(o * pi / 8);
    }
    for (const auto& gr : d->groups) {
        // (the tap rows of `entries` scales fit the work buffer they pass through)
        for (int j0 = 0; j0 < gr.second; j0 += d->entries) {
            bimpk::TapSet set{};
            set.n = std::min(gr.second - j0, d->entries);
            for (int j = 0; j < set.n; ++j) {
                const DScale& x = d->sc[gr.first + j0 + j];
                const double sigma = (double)x.g.lambda * (double)ratio;
                const float sf = (float)sigma, sq = sf * sf;
                set.s[j] = bimpk::TapScale{x.g.lambda, x.g.fs, -1.0f / (2 * sq), sigma, x.g.kW,
                                           x.g.kX, x.dK, x.Q, x.G};
            }
            const auto& g = d->sc[gr.first].g;
            DCHK(d, bimpk::diff_taps(set, trig, gamma, d->taps, d->tapStride, s));
            // T is free here: only a backward uses it
            DCHK(d, bimpk::diff_bank_rows(set, d->taps, d->tapStride, d->kwMax, g.FW, d->adj.T,
                                          d->tw[g.FW], s));
            DCHK(d, bimpk::diff_bank_cols(set, d->adj.T, d->kwMax, g.FH, g.FW,
                                          1.0f / ((float)g.FH * (float)g.FW), d->tw[g.FH], s));
        }
    }
    DCHK(d, hipStreamSynchronize(s));
    d->fwdPending = false;
    d->ratio = ratio;
    d->gamma = gamma;
    return BIMP_OK;
}

// Float pyramids of nb consecutive images into d->lev (level l of image b at
// lev[l] + b * lw[l] * lh[l]).
int pyramid(bimp_diff* d, const float* img, int nb, hipStream_t s) {
    DCHK(d, hipMemcpyAsync(d->lev[0], img, (size_t)nb * d->width * d->height * 4,
                           hipMemcpyDeviceToDevice, s));
    for (int l = 1; l <= d->maxLevel; ++l)
        DCHK(d, bimpk::diff_pyr_down(d->lev[l - 1], d->lw[l - 1], d->lh[l - 1], d->lev[l], d->lw[l],
                                     d->lh[l], nb, s));
    return BIMP_OK;
}

// The D maps of scales first..first+n-1 (one pyramid level, one transform size) into the
// response vector `resp` through the detection path's kernels, one launch per stage: real
// row FFTs of the float level (two rows per complex FFT), column FFTs of the half spectra,
// inverse columns with the quadrature bank G, inverse rows with the complex-cell magnitude
// over the Hc x Wc region, then the cells stencil.
int group_forward(bimp_diff* d, int first, int n, int img0, int nb, float* resp, hipStream_t s) {
    // entry k = b * n + j of the launches: image img0 + b of the pyramids in d->lev, scale
    // first + j; its D map goes to resp + b * respSize
    const DScale& x0 = d->sc[first];
    const auto& g = x0.g;
    const size_t dtSize = (size_t)(g.FW / 2 + 1) * g.FH;
    bimpk::ScaleSet ss;
    ss.n = n * nb;
    bimpk::CellScale cs[bimpk::kMaxEntries];
    for (int b = 0; b < nb; ++b)
        for (int j = 0; j < n; ++j) {
            const DScale& x = d->sc[first + j];
            const int k = b * n + j;
            ss.kX[k] = x.g.kX;
            ss.G[k] = x.G;
            ss.DT[k] = x.DT + (size_t)b * dtSize;
            ss.C[k] = x.Cf + (size_t)b * kNumOri * x.Hc * x.ldc;
            cs[k] = bimpk::CellScale{ss.C[k], x.Hc, x.ldc, g.FH, g.FW, g.H, g.W, x.cp,
                                     resp + (size_t)b * d->respSize + x.respOff,
                                     d->Sf + (size_t)b * d->respSize + x.respOff, d->maxslot};
        }
    const int ncols = g.FW / 2 + 1;
    const size_t rstride = (size_t)g.H * ncols;
    const size_t tstride = (size_t)kNumOri * x0.Hc * g.FW;
    const size_t lsz = (size_t)d->lw[g.level] * d->lh[g.level];
    DCHK(d, bimpk::launch_fwd_rows_f32(g.FW, d->lev[g.level] + img0 * lsz, lsz, n,
                                       (size_t)d->lw[g.level], g.H, g.W, ss,
                                       255.0f * d->opt.input_scale, d->R, ncols, rstride,
                                       d->tw[g.FW], s));
    DCHK(d, bimpk::launch_fwd_cols(g.FH, d->R, ncols, rstride, g.H, ss, ncols, d->tw[g.FH], s));
    DCHK(d, bimpk::launch_inv_cols(g.FH, ss, g.FW, x0.Hc, d->T, tstride, d->tw[g.FH], s));
    DCHK(d, bimpk::launch_inv_rows(g.FW, g.FH, ss, d->T, tstride, x0.Hc, x0.Wc, x0.ldc,
                                   d->tw[g.FW], s));
    // as few launches as the job table allows, of about the same size
    const int parts = (n * nb + bimpk::kCellMaxScales - 1) / bimpk::kCellMaxScales;
    for (int q = 0; q < parts; ++q) {
        const int k0 = n * nb * q / parts, k1 = n * nb * (q + 1) / parts;
        DCHK(d, bimpk::launch_cells(cs + k0, k1 - k0, s));
    }
    return BIMP_OK;
}

int forward(bimp_diff* d, const float* img, int nimg, float* resp, hipStream_t s) {
    const size_t isz = (size_t)d->width * d->height;
    // chunks of images whose pyramids fit d->lev; each group takes nbf of them per launch
    for (int b0 = 0; b0 < nimg; b0 += d->nbMax) {
        const int nb = std::min(d->nbMax, nimg - b0);
        int st = pyramid(d, img + b0 * isz, nb, s);
        if (st) return st;
        for (const auto& gr : d->groups) {
            const int nbf = d->sc[gr.first].nbf;
            for (int b = 0; b < nb; b += nbf)
                if ((st = group_forward(d, gr.first, gr.second, b, std::min(nbf, nb - b),
                                        resp + (size_t)(b0 + b) * d->respSize, s)))
                    return st;
        }
    }
    return BIMP_OK;
}

// What a parameter change has to wait for: the work that a forward has put on s.  (Nothing on the
// null stream, where the change itself runs: the marker, a barrier packet, takes 3 us.)
int mark_forward(bimp_diff* d, hipStream_t s) {
    if (!s) return BIMP_OK;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    DCHK(d, hipStreamIsCapturing(s, &capturing));
    if (capturing != hipStreamCaptureStatusNone) {
        d->fwdCaptured = true;
        return BIMP_OK;
    }
    DCHK(d, hipEventRecord(d->fwdDone, s));
    d->fwdPending = true;
    return BIMP_OK;
}

// Backward of scales first..first+n-1 (one level, one transform size) for nb images from img0
// of the pyramids in d->lev: adds to (with `fresh`: sets) their level gradients in d->glev and
// writes their parameter partials.  gD: the upstream gradient of image img0's response vector.
int group_backward(bimp_diff* d, int first, int n, int img0, int nb, const float* gD, bool fresh,
                   size_t pstride, hipStream_t s) {
    const DScale& x0 = d->sc[first];
    const auto& g = x0.g;
    bimpk::AdjSet set{};
    set.n = n;
    for (int j = 0; j < n; ++j) {
        const DScale& x = d->sc[first + j];
        set.kX[j] = x.g.kX;
        set.kW[j] = x.g.kW;
        set.Q[j] = x.Q;
        set.dK[j] = x.dK;
        set.resp[j] = x.respOff;
        set.cp[j] = x.cp;
    }
    const size_t lsz = (size_t)d->lw[g.level] * d->lh[g.level];
    const bimpk::AdjLevel L{g.H, g.W, g.FH, g.FW, x0.Hc, nb, d->lw[g.level], lsz,
                            255.0f * d->opt.input_scale,
                            1.0f / (float)((size_t)g.FH * g.FW), d->lev[g.level] + img0 * lsz};
    const float2 *twH = d->tw[g.FH], *twW = d->tw[g.FW];
    const auto& w = d->adj;
    DCHK(d, bimpk::diff_backward_rows(set, L, w, twW, s));
    DCHK(d, bimpk::diff_cols_kx(w.T, g.H, g.FH, g.FW, set.ints(set.kX), n, n * nb, w.D, twH, s));
    DCHK(d, bimpk::diff_z_cols(set, L, w, twH, s));
    DCHK(d, bimpk::diff_cells_grad(set, L, w, gD, d->respSize, twW, s));
    DCHK(d, bimpk::diff_adj_cols(set, L, w, d->kwMax, twH, s));
    DCHK(d, bimpk::diff_adj_rows(set, L, w, d->kwMax, fresh, d->glev[g.level] + img0 * lsz,
                                 d->lh[g.level],
                                 d->partials + pstride * img0 + 2 * (size_t)d->maxBlocks * first,
                                 pstride, 2 * d->maxBlocks, twW, s));
    return BIMP_OK;
}

}  // namespace

extern "C" {

int bimp_diff_create(int width, int height, const float* lambdas, int n, const bimp_options* opt,
                     bimp_diff** out) {
    if (!out) return BIMP_E_ARG;
    *out = nullptr;
    if (width < 8 || height < 8 || !lambdas || n <= 0 || n > 64) return BIMP_E_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return BIMP_E_DEVICE;
    bimp_diff* d = new bimp_diff;
    d->width = width;
    d->height = height;
    if (opt)
        d->opt = *opt;
    else
        bimp_default_options(&d->opt);
    auto bail = [&](int code) {
        bimp_diff_destroy(d);
        return code;
    };
    std::vector<float> lam(lambdas, lambdas + n);
    std::sort(lam.begin(), lam.end());
    std::vector<int> sizes;
    for (float l : lam) {
        DScale x;
        if (!bimph::derive_scale(l, width, height, d->opt.pyr_threshold, d->opt.support, &x.g) ||
            x.g.lambda < 1.f || x.g.H < 4 || x.g.W < 4)
            return bail(BIMP_E_ARG);
        if (!bimpk::fft_size_supported(x.g.FH) || !bimpk::fft_size_supported(x.g.FW) ||
            x.g.kW > x.g.FH || x.g.kW > x.g.FW)
            return bail(BIMP_E_UNSUPPORTED);
        for (int o = 0; o < kNumOri; ++o) {
            const double theta = (double)(float)(o * 3.1415926535897932384626433832795 / kNumOri);
            x.cp.ea[o] = round_half_away(0.6 * x.g.lambda * std::cos(theta));
            x.cp.eb[o] = round_half_away(0.6 * x.g.lambda * std::sin(theta));
            x.cp.ia[o] = round_half_away(0.6 * x.g.lambda * std::sin(theta));
            x.cp.ib[o] = round_half_away(0.6 * x.g.lambda * std::cos(theta));
            x.cp.ra[o] = round_half_away(0.5 * x.cp.ia[o]);
            x.cp.rb[o] = round_half_away(0.5 * x.cp.ib[o]);
        }
        x.respOff = d->respSize;
        d->respSize += (size_t)x.g.H * x.g.W;
        // the complex-cell region the cells stencil reads (the detection context's rule)
        x.Wc = std::min(x.g.FW, x.g.W + 1);
        x.Hc = std::min(x.g.FH, x.g.H + (x.g.W == x.g.FW ? 2 : 1));
        x.ldc = (x.Wc + 31) / 32 * 32;

        d->maxLevel = std::max(d->maxLevel, x.g.level);
        sizes.push_back(x.g.FH);
        sizes.push_back(x.g.FW);
        d->sc.push_back(x);
    }
    // launch groups: consecutive scales (sorted by wavelength) of one level and transform size
    for (int i = 0; i < (int)d->sc.size();) {
        const auto& g = d->sc[i].g;
        int n = 1;
        while (i + n < (int)d->sc.size() && n < bimpk::kMaxBatch && n < bimpk::kCellMaxScales &&
               d->sc[i + n].g.level == g.level && d->sc[i + n].g.FH == g.FH &&
               d->sc[i + n].g.FW == g.FW)
            ++n;
        d->groups.emplace_back(i, n);
        // The forward takes nbf images of the group per launch: n * nbf entries, at least 8 and
        // up to kMaxEntries while their T stays in the last-level cache (eight entries, and the
        // row pass image by image, took 202 us for three 333 x 251 images against 149, 236
        // against 137 for five of 200 x 130).
        const size_t t1 = (size_t)n * kNumOri * d->sc[i].Hc * g.FW * sizeof(float2);
        const int fit = (int)std::min<size_t>(bimpk::kMaxEntries / n, kForwardTBytes / t1);
        const int nbf = std::min(d->nbMax, std::max({1, bimpk::kMaxBatch / n, fit}));
        for (int j = 0; j < n; ++j) d->sc[i + j].nbf = nbf;
        d->rSize = std::max(d->rSize, (size_t)n * nbf * g.H * (g.FW / 2 + 1));
        d->tSize = std::max(d->tSize, (size_t)n * nbf * kNumOri * d->sc[i].Hc * g.FW);
        i += n;
    }
    d->lw.assign(d->maxLevel + 1, 0);
    d->lh.assign(d->maxLevel + 1, 0);
    d->lw[0] = width;
    d->lh[0] = height;
    for (int l = 1; l <= d->maxLevel; ++l) {
        d->lw[l] = (d->lw[l - 1] + 1) / 2;
        d->lh[l] = (d->lh[l - 1] + 1) / 2;
    }
    // (scale, image) pairs per backward launch: up to 32, while their buffers (two complex maps
    // of the padded size, the gradient's pairs and, per orientation, two complex and one real
    // map) stay within 4 GB.  More pairs mean fewer and longer launches: eight 512 x 512 images
    // took 2277, 2084 and 2017 us with 8, 16 and 32, five 200 x 130 images 616, 479 and 350 us.
    // A launch holds no more than one group's scales of the images held at once.
    size_t pm = 0, kwfw = 0;
    int widest = 0;
    for (const auto& gr : d->groups) widest = std::max(widest, gr.second);
    for (const auto& x : d->sc) {
        pm = std::max(pm, (size_t)x.g.FH * x.g.FW);
        kwfw = std::max(kwfw, (size_t)x.g.FW);
        d->kwMax = std::max(d->kwMax, x.g.kW);
    }
    const size_t per = pm * (2 * sizeof(float2) + sizeof(uint2) +
                             kNumOri * (2 * sizeof(float2) + sizeof(float)));
    const size_t most = std::min<size_t>(32, (size_t)widest * d->nbMax);
    d->entries = (int)std::max<size_t>(1, std::min<size_t>(most, (size_t(4) << 30) / per));
    const size_t NE = (size_t)d->entries;
    const size_t NB = (size_t)d->nbMax;
    d->lev.assign(d->maxLevel + 1, nullptr);
    d->glev.assign(d->maxLevel + 1, nullptr);
    for (int l = 0; l <= d->maxLevel; ++l)
        if (hipMalloc(&d->lev[l], NB * d->lw[l] * d->lh[l] * 4) != hipSuccess ||
            hipMalloc(&d->glev[l], NB * d->lw[l] * d->lh[l] * 4) != hipSuccess)
            return bail(BIMP_E_ALLOC);
    for (auto& x : d->sc) {
        const size_t kk = (size_t)x.g.kW * x.g.kW;
        d->tapStride = std::max(d->tapStride, kNumOri * kk);
        d->maxBlocks = std::max(d->maxBlocks, bimpk::diff_param_blocks(x.g.kW));
        if (hipMalloc(&x.Q, (size_t)kNumOri * x.g.FH * x.g.FW * sizeof(float2)) != hipSuccess ||
            hipMalloc(&x.G, (size_t)bimpk::kUniqueOri * x.g.FH * x.g.FW * sizeof(float)) != hipSuccess ||
            hipMalloc(&x.DT, (size_t)x.nbf * (x.g.FW / 2 + 1) * x.g.FH * sizeof(float2)) != hipSuccess ||
            hipMalloc(&x.Cf, (size_t)x.nbf * kNumOri * x.Hc * x.ldc * sizeof(float)) != hipSuccess ||
            hipMalloc(&x.dK, 4 * kNumOri * kk * sizeof(float)) != hipSuccess)
            return bail(BIMP_E_ALLOC);
    }
    auto& w = d->adj;
    if (hipMalloc(&w.D, NE * pm * sizeof(float2)) != hipSuccess ||
        hipMalloc(&w.A, NE * pm * sizeof(float2)) != hipSuccess ||
        hipMalloc(&w.T, NE * kNumOri * pm * sizeof(float2)) != hipSuccess ||
        hipMalloc(&w.Z, NE * kNumOri * pm * sizeof(float2)) != hipSuccess ||
        hipMalloc(&w.C, NE * kNumOri * pm * sizeof(float)) != hipSuccess ||
        hipMalloc(&w.gm, NE * pm * sizeof(uint2)) != hipSuccess ||
        hipMalloc(&w.Yc, NE * kNumOri * d->kwMax * kwfw * sizeof(float2)) != hipSuccess ||
        hipMalloc(&d->taps, (size_t)bimpk::kAdjMax * d->tapStride * sizeof(float2)) != hipSuccess ||
        hipMalloc(&d->maxslot, sizeof(unsigned)) != hipSuccess ||
        hipMalloc(&d->R, d->rSize * sizeof(float2)) != hipSuccess ||
        hipMalloc(&d->T, d->tSize * sizeof(float2)) != hipSuccess ||
        hipMalloc(&d->Sf, (size_t)d->nbMax * d->respSize * sizeof(float)) != hipSuccess ||
        hipMalloc(&d->partials, NB * 2 * (size_t)d->maxBlocks * d->sc.size() * sizeof(float)) !=
                hipSuccess)
        return bail(BIMP_E_ALLOC);
    std::sort(sizes.begin(), sizes.end());
    sizes.erase(std::unique(sizes.begin(), sizes.end()), sizes.end());
    for (int n2 : sizes) {
        if (bimpk::diff_prepare(n2) != hipSuccess || bimpk::prepare_size(n2) != hipSuccess)
            return bail(BIMP_E_DEVICE);
        std::vector<float2> t;
        if (!bimpk::twiddle_table(n2, t)) return bail(BIMP_E_UNSUPPORTED);
        float2* p = nullptr;
        if (hipMalloc(&p, t.size() * sizeof(float2) + 256) != hipSuccess) return bail(BIMP_E_ALLOC);
        d->tw[n2] = p;
        if (hipMemcpy(p, t.data(), t.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess)
            return bail(BIMP_E_DEVICE);
    }
    // (orders kernels of this device only)
    if (hipEventCreateWithFlags(&d->fwdDone,
                                hipEventDisableTiming | hipEventDisableSystemFence) != hipSuccess)
        return bail(BIMP_E_ALLOC);
    if (bimpk::prepare_common() != hipSuccess) return bail(BIMP_E_DEVICE);
    const int st = set_params(d, d->opt.sigma_ratio, d->opt.gamma);
    if (st) return bail(st);
    *out = d;
    return BIMP_OK;
}

int bimp_diff_destroy(bimp_diff* d) {
    if (!d) return BIMP_E_ARG;
    (void)hipDeviceSynchronize();
    for (auto& x : d->sc) {
        (void)hipFree(x.Q);
        (void)hipFree(x.G);
        (void)hipFree(x.DT);
        (void)hipFree(x.Cf);
        (void)hipFree(x.dK);
    }
    for (auto* p : d->lev) (void)hipFree(p);
    for (auto* p : d->glev) (void)hipFree(p);
    for (auto& kv : d->tw) (void)hipFree(kv.second);
    for (void* p : {(void*)d->adj.D, (void*)d->adj.A, (void*)d->adj.T, (void*)d->adj.Z,
                    (void*)d->adj.C, (void*)d->adj.gm, (void*)d->adj.Yc, (void*)d->taps,
                    (void*)d->maxslot, (void*)d->partials, (void*)d->R, (void*)d->T, (void*)d->Sf})
        (void)hipFree(p);
    if (d->fwdDone) (void)hipEventDestroy(d->fwdDone);
    delete d;
    return BIMP_OK;
}

long long bimp_diff_response_size(const bimp_diff* d) { return d ? (long long)d->respSize : BIMP_E_ARG; }

int bimp_diff_set_params(bimp_diff* d, float sigma_ratio, float gamma) {
    if (!d || !(sigma_ratio > 0.f) || !(gamma > 0.f)) return BIMP_E_ARG;
    if (sigma_ratio == d->ratio && gamma == d->gamma) return BIMP_OK;
    return set_params(d, sigma_ratio, gamma);
}

int bimp_diff_forward(bimp_diff* d, const float* d_img, int nimg, float* d_resp,
                      bimp_stream_t stream) {
    if (!d || !d_img || !d_resp || nimg <= 0) return BIMP_E_ARG;
    const hipStream_t s = (hipStream_t)stream;
    const int st = forward(d, d_img, nimg, d_resp, s);
    const int marked = mark_forward(d, s);  // after a failure too: some of it may be under way
    return st ? st : marked;
}

int bimp_diff_backward(bimp_diff* d, const float* d_img, int nimg, const float* d_grad_resp,
                       float* d_grad_img, double* grad_params, bimp_stream_t stream) {
    if (!d || !d_img || !d_grad_resp || !d_grad_img || nimg <= 0) return BIMP_E_ARG;
    hipStream_t s = (hipStream_t)stream;
    const size_t isz = (size_t)d->width * d->height;
    double gr = 0, gg = 0;
    std::vector<float> part;
    const size_t pstride = 2 * (size_t)d->maxBlocks * d->sc.size();  // partials per image
    // chunks of images whose pyramids are held; each group then takes as many (scale, image)
    // pairs per launch as the work buffers hold
    for (int b0 = 0; b0 < nimg; b0 += d->nbMax) {
        const int nb = std::min(d->nbMax, nimg - b0);
        int st = pyramid(d, d_img + b0 * isz, nb, s);
        if (st) return st;
        std::vector<char> fresh(d->maxLevel + 1, 1);
        for (const auto& gr : d->groups) {
            // (a group holds at most kMaxBatch scales)
            for (int j0 = 0; j0 < gr.second; j0 += d->entries) {
                const int n = std::min(gr.second - j0, d->entries);
                const int nbg = std::max(1, d->entries / n);
                const int level = d->sc[gr.first].g.level;
                for (int b = 0; b < nb; b += nbg)
                    if ((st = group_backward(d, gr.first + j0, n, b, std::min(nbg, nb - b),
                                             d_grad_resp + (size_t)(b0 + b) * d->respSize,
                                             fresh[level] != 0, pstride, s)))
                        return st;
                fresh[level] = 0;
            }
        }
        // (a level no scale uses starts at zero as well)
        for (int l = 0; l <= d->maxLevel; ++l)
            if (fresh[l])
                DCHK(d, bimpk::diff_fill(d->glev[l], (size_t)nb * d->lw[l] * d->lh[l], s));
        for (int l = d->maxLevel; l >= 1; --l)
            DCHK(d, bimpk::diff_pyr_down_adj(d->glev[l], d->lw[l], d->lh[l], d->glev[l - 1],
                                             d->lw[l - 1], d->lh[l - 1], nb, s));
        DCHK(d, hipMemcpyAsync(d_grad_img + b0 * isz, d->glev[0], (size_t)nb * isz * 4,
                               hipMemcpyDeviceToDevice, s));
        part.resize(pstride * nb);
        DCHK(d, hipMemcpyAsync(part.data(), d->partials, part.size() * 4, hipMemcpyDeviceToHost, s));
        DCHK(d, hipStreamSynchronize(s));
        // image by image, scale by scale, block by block: the order of one image at a time
        for (int b = 0; b < nb; ++b)
            for (size_t si = 0; si < d->sc.size(); ++si) {
                const int nbk = bimpk::diff_param_blocks(d->sc[si].g.kW);
                const float* pp = part.data() + pstride * b + 2 * (size_t)d->maxBlocks * si;
                for (int k = 0; k < nbk; ++k) {
                    gr += pp[2 * k];
                    gg += pp[2 * k + 1];
                }
            }
    }
    if (grad_params) {
        grad_params[0] = gr;
        grad_params[1] = gg;
    }
    return BIMP_OK;
}

const char* bimp_diff_last_error(const bimp_diff* d) { return d ? d->err.c_str() : ""; }

}  // extern "C"
