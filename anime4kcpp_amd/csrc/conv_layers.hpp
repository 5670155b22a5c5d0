// The conv3x3 layers of the layer-by-layer networks (ACNet<8>, ArtCNN<F>, FSRCNNX<F>): their
// epilogues (LayerMode), which keep the reference's separately rounded steps after the conv sum
// (Common.hpp:116-164, 227-288, 290-341), and the 16- and 32-channel kernel.  The 8-channel layers
// are conv8_rows.hpp's.
//   kRelu          max(v, 0)                                        ArtCNN body
//   kPrelu         max(v, 0) + a * min(v, 0)                        ACNet<8>, FSRCNNX body
//   kAddFeat       v * 1 + feat                                     ArtCNN's last F -> F
//   kPreluConv1x1  PReLU, then conv1x1 F -> F + bias, * 1 + feat, PReLU
//                                                                   FSRCNNX's last block
//   kShuffle       conv F -> 4, pixel shuffle to 2x                 ArtCNN, FSRCNNX tail
//   kShuffleSrc    the same, + the source pixel                     ACNet<8> final
//   kReluDeconv    ReLU, then the 2x2 stride-2 deconv 8 -> 1 to 2x  ACNetLegacy's last layer
//                  (Common.hpp:344-393), layer by layer
// convf_layer (F = 16 or 32): one launch per layer, reading an F-channel f32 map from HBM (channel
// quads interleaved per pixel: pixel x at float4 index F/4 * x + q, rows of `fp` bytes), and
// writing the next map or, for the last layer, the 2x output image.  v_mfma_f32_16x16x4_f32 with
// M = 16 output channels per tile (F/16 tiles), N = 16 pixels of one row, K = 9 taps x F; lane
// group g supplies input channels g*F/4 .. g*F/4 + F/4 - 1 from channel-quad LDS planes; NI items
// per wave batch share each tap's A operands.  A lane's D registers hold 4 consecutive channels of
// one pixel, which is exactly the B operand a conv1x1 MFMA needs (K step r of lane group g = the
// r-th of them), so the fused conv1x1 costs F/4 x F/16 more MFMAs and no data movement.
#pragma once

#include "acnet_device.hpp"
#include "acnet_kernels.hpp"
#include "acnet_mfma32_item.hpp"   // mma32

namespace achip {

#pragma clang fp contract(off)

enum LayerMode : int { kRelu = 0, kPrelu = 1, kAddFeat = 2, kPreluConv1x1 = 3, kShuffle = 4, kShuffleSrc = 5,
                       kReluDeconv = 6 };

// Arguments of one layer launch; a mode leaves the fields it does not read null.
struct LayerArgs {
    const float* wa;        // this layer's per-lane A operands
    const float* bias;      // F biases (4 for the shuffle modes)
    const float* alpha;     // F PReLU slopes
    const float* w1;        // conv1x1 A operands
    const float* b1;        // conv1x1 biases (F)
    const float* alpha1;    // F PReLU slopes after the skip connection
    const float4* feat;     // skip-connection map, same pitch as the input map
    const float* k2;        // deconv weights k2[c][q] (kReluDeconv)
    const void* src;        // source image (kShuffleSrc)
    long ss;
    void* dst;              // output image (shuffle modes)
    long ds;
};

// PReLU (Common.hpp:42-49): max(v, 0) + alpha * min(v, 0), each step rounded
__device__ inline float prelu(float v, float alpha)
{
    return __fadd_rn(fmaxf(v, 0.0f), __fmul_rn(alpha, fminf(v, 0.0f)));
}

__device__ inline float add_skip(float v, float f) { return __fadd_rn(__fmul_rn(v, 1.0f), f); }

// Stage ROWS x CW pixels of an f32 map (NQ channel quads per pixel, rows of fp bytes) whose
// top-left is image pixel (cx0, ry0), clamped to the image, into LDS: quad q of staged pixel
// (c, r) goes to planes[q][r * PW + c].  Each thread issues all of its loads before its first
// LDS store, so a workgroup waits for one load latency rather than one per pass over the tile.
template <int NT, int CW, int ROWS, int NQ, int PW>
__device__ __forceinline__ void stage_map(const float4* __restrict__ fin, long fp, int W, int H, int cx0, int ry0,
                                          float4* const* planes)
{
    constexpr int N = ROWS * CW, K = (N + NT - 1) / NT;
    float4 v[K][NQ];
#pragma unroll
    for (int k = 0; k < K; k++) {
        // threads past the last pixel load it again (no branch around the loads) and skip the store
        const int e = min(static_cast<int>(threadIdx.x) + k * NT, N - 1);
        const int r = e / CW, c = e - r * CW;
        const int sy = clampi(ry0 + r, 0, H - 1), sx = clampi(cx0 + c, 0, W - 1);
        const float4* px = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(fin) + static_cast<long>(sy) * fp) + NQ * sx;
#pragma unroll
        for (int q = 0; q < NQ; q++) v[k][q] = px[q];
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int e = threadIdx.x + k * NT;
        if (k < K - 1 || e < N) {
            const int r = e / CW, c = e - r * CW;
#pragma unroll
            for (int q = 0; q < NQ; q++) planes[q][r * PW + c] = v[k][q];
        }
    }
}

// ---- F = 16 or 32: channel tiles ----
// TW x 16 output pixels per workgroup of NT threads; NI items per wave batch.  The defaults
// are the fastest of a sweep over 1080p maps on one MI355X: 32 x 16 (F = 16, 55 KB of LDS)
// and 16 x 16 (F = 32, 74 KB) tiles let two workgroups share a CU, so one stages its tile
// while the other computes.
template <int F, int TW_ = (F == 16 ? 32 : 16), int NT_ = 512, int NI_ = (F == 16 ? 4 : 2), int PF_ = 1>
struct ConvTile {
    static constexpr bool PF = PF_;                                     // load tap p + 1's A operands during tap p
    static constexpr int TW = TW_, TH = 16, NT = NT_, NW = NT / 64;
    static constexpr int PW = (TW + 2 + 15) / 16 * 16, PH = TH + 2;    // plane pitch: 16-pixel multiple
    static constexpr int NQ = F / 4;                                    // channel-quad planes
    static constexpr int KQ = F / 4;                                    // K steps per tap (channels per lane group)
    static constexpr int MT = F / 16;                                   // 16-channel output tiles
    static constexpr int NI = NI_;                                      // items per wave batch
    static constexpr int SEGS = TW / 16, ITEMS = SEGS * TH;
    static constexpr int BATCHES = (ITEMS / NW + NI - 1) / NI;
    static_assert(ITEMS % (NW * NI) == 0, "whole batches");
};

template <int F, int MODE, typename TOUT, class C = ConvTile<F>>
__global__ __launch_bounds__(C::NT) void convf_layer(const float4* __restrict__ fin, long fp, int W, int H,
                                                     float4* __restrict__ fout, const LayerArgs la)
{
    static_assert(MODE != kShuffleSrc, "convf_layer epilogues");
    __shared__ float4 planes[C::NQ][C::PH * C::PW];
    const int tiles_x = gridDim.x;
    const int t = xcd_tile(blockIdx.y * tiles_x + blockIdx.x, tiles_x * gridDim.y);
    const int ty = t / tiles_x, tx = t - ty * tiles_x;
    const int x0 = tx * C::TW, y0 = ty * C::TH;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, j = lane & 15;

    // stage rows y0-1 .. y0+TH, columns x0-1 .. x0+TW (replicated at the image edges)
    {
        float4* pl[C::NQ];
#pragma unroll
        for (int q = 0; q < C::NQ; q++) pl[q] = planes[q];
        stage_map<C::NT, C::TW + 2, C::PH, C::NQ, C::PW>(fin, fp, W, H, x0 - 1, y0 - 1, pl);
    }
    // lane (g, j) of output tile h owns channels 16 h + 4 g .. + 3
    f32x4m b0[C::MT];
#pragma unroll
    for (int h = 0; h < C::MT; h++) {
        if constexpr (MODE == kShuffle)   // output channels 0..3 only: rows 0-3 of the first tile
            b0[h] = (h == 0 && g == 0) ? (f32x4m){ la.bias[0], la.bias[1], la.bias[2], la.bias[3] } : (f32x4m){ 0.f, 0.f, 0.f, 0.f };
        else {
            const float* bl = la.bias + 16 * h + 4 * g;
            b0[h] = (f32x4m){ bl[0], bl[1], bl[2], bl[3] };
        }
    }
    // the F -> 4 tail needs only the first output tile (channels 0-3)
    constexpr int MTU = MODE == kShuffle ? 1 : C::MT;
    // slopes and conv1x1 operands of this lane's channels, in registers for the whole tile
    constexpr bool PRELU = MODE == kPrelu || MODE == kPreluConv1x1;
    constexpr int NA = PRELU ? C::MT : 1, N1 = MODE == kPreluConv1x1 ? C::MT : 1;
    float al[NA][4], al1[N1][4], w1[4 * N1][N1];
    f32x4m b1[N1];
    if constexpr (PRELU) {
#pragma unroll
        for (int h = 0; h < C::MT; h++)
#pragma unroll
            for (int r = 0; r < 4; r++) al[h][r] = la.alpha[16 * h + 4 * g + r];
    }
    if constexpr (MODE == kPreluConv1x1) {
#pragma unroll
        for (int h = 0; h < C::MT; h++) {
            const float* bl = la.b1 + 16 * h + 4 * g;
            b1[h] = (f32x4m){ bl[0], bl[1], bl[2], bl[3] };
#pragma unroll
            for (int r = 0; r < 4; r++) {
                al1[h][r] = la.alpha1[16 * h + 4 * g + r];
#pragma unroll
                for (int h2 = 0; h2 < C::MT; h2++) w1[4 * h + r][h2] = la.w1[((4 * h + r) * 64 + lane) * C::MT + h2];
            }
        }
    }
    __syncthreads();

    const int gx1 = min(x0 + C::TW, W), gy1 = min(y0 + C::TH, H);
    for (int batch = 0; batch < C::BATCHES; batch++) {
        f32x4m acc[C::NI][C::MT];
        int base[C::NI];
#pragma unroll
        for (int i = 0; i < C::NI; i++) {
            const int item = wave + C::NW * (batch * C::NI + i);
            const int row = item / C::SEGS, seg = item - row * C::SEGS;
            // item pixels (x0 + 16 seg + j, y0 + row): staged at (16 seg + j + 1, row + 1)
            base[i] = row * C::PW + 16 * seg + j;
#pragma unroll
            for (int h = 0; h < C::MT; h++) acc[i][h] = b0[h];
        }
        // A operands [tap][lane][q * MTU + h]: KQ * MTU floats per tap and lane
        constexpr int AW = C::KQ * MTU;
        float4 an[AW / 4];
        const float4* const ap0 = reinterpret_cast<const float4*>(la.wa + static_cast<long>(lane) * AW);
        constexpr long kTapF4 = 64L * AW / 4;   // float4s per tap
        if constexpr (C::PF) {
#pragma unroll
            for (int v = 0; v < AW / 4; v++) an[v] = ap0[v];
        }
#pragma unroll 1
        for (int p = 0; p < 9; p++) {
            const int dy = p / 3, dx = p - dy * 3;
            float a[AW];
            if constexpr (C::PF) {
#pragma unroll
                for (int v = 0; v < AW / 4; v++) {
                    a[4 * v] = an[v].x; a[4 * v + 1] = an[v].y; a[4 * v + 2] = an[v].z; a[4 * v + 3] = an[v].w;
                }
                if (p < 8) {
#pragma unroll
                    for (int v = 0; v < AW / 4; v++) an[v] = ap0[(p + 1) * kTapF4 + v];
                }
            } else {
#pragma unroll
                for (int v = 0; v < AW / 4; v++) {
                    const float4 f = ap0[p * kTapF4 + v];
                    a[4 * v] = f.x; a[4 * v + 1] = f.y; a[4 * v + 2] = f.z; a[4 * v + 3] = f.w;
                }
            }
            // B operands of every item first, then the MFMAs with the K step outermost, so
            // that consecutive MFMAs update different accumulators (NI x MTU chains)
            float bv[C::NI][C::KQ];
#pragma unroll
            for (int i = 0; i < C::NI; i++) {
                const int off = base[i] + dy * C::PW + dx;
#pragma unroll
                for (int v = 0; v < C::KQ / 4; v++) {
                    const float4 f = planes[(C::KQ / 4) * g + v][off];
                    bv[i][4 * v] = f.x; bv[i][4 * v + 1] = f.y; bv[i][4 * v + 2] = f.z; bv[i][4 * v + 3] = f.w;
                }
            }
#pragma unroll
            for (int q = 0; q < C::KQ; q++)
#pragma unroll
                for (int i = 0; i < C::NI; i++)
#pragma unroll
                    for (int h = 0; h < MTU; h++) acc[i][h] = mma32(a[q * MTU + h], bv[i][q], acc[i][h]);
        }
        if constexpr (MODE == kPreluConv1x1) {
            // PReLU, then conv1x1: K step 4 h + r of lane group g is channel 16 h + 4 g + r,
            // this lane's D register r of tile h; A operands [4 h + r][lane][h2]
#pragma unroll
            for (int i = 0; i < C::NI; i++) {
                f32x4m d[C::MT];
#pragma unroll
                for (int h2 = 0; h2 < C::MT; h2++) d[h2] = b1[h2];
#pragma unroll
                for (int h = 0; h < C::MT; h++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float bv = prelu(acc[i][h][r], al[h][r]);
#pragma unroll
                        for (int h2 = 0; h2 < C::MT; h2++) d[h2] = mma32(w1[4 * h + r][h2], bv, d[h2]);
                    }
#pragma unroll
                for (int h2 = 0; h2 < C::MT; h2++) acc[i][h2] = d[h2];
            }
        }
        // epilogue: lane (g, j) holds output channels 16 h + 4 g .. + 3 of pixel j
#pragma unroll
        for (int i = 0; i < C::NI; i++) {
            const int item = wave + C::NW * (batch * C::NI + i);
            const int row = item / C::SEGS, seg = item - row * C::SEGS;
            const int x = x0 + 16 * seg + j, y = y0 + row;
            if (x >= gx1 || y >= gy1) continue;
            if constexpr (MODE == kShuffle) {
                if (g == 0) {   // the 4 sub-pixels n: output (2x + n % 2, 2y + n / 2)
                    const f32x4m v = acc[i][0];
                    store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y) + 2 * x, v[0], v[1]);
                    store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y + 1) + 2 * x, v[2], v[3]);
                }
            } else {
                const long off = static_cast<long>(y) * fp;
                float4* po = reinterpret_cast<float4*>(reinterpret_cast<char*>(fout) + off) + C::NQ * x;
#pragma unroll
                for (int h = 0; h < C::MT; h++) {
                    const f32x4m v = acc[i][h];
                    float4 o;
                    if constexpr (MODE == kRelu) {
                        o = make_float4(fmaxf(v[0], 0.f), fmaxf(v[1], 0.f), fmaxf(v[2], 0.f), fmaxf(v[3], 0.f));
                    } else if constexpr (MODE == kPrelu) {
                        o = make_float4(prelu(v[0], al[h][0]), prelu(v[1], al[h][1]), prelu(v[2], al[h][2]), prelu(v[3], al[h][3]));
                    } else {   // kAddFeat, kPreluConv1x1: * 1 + feat (then PReLU)
                        const float4 r = *(reinterpret_cast<const float4*>(reinterpret_cast<const char*>(la.feat) + off) + C::NQ * x + 4 * h + g);
                        o = make_float4(add_skip(v[0], r.x), add_skip(v[1], r.y), add_skip(v[2], r.z), add_skip(v[3], r.w));
                        if constexpr (MODE == kPreluConv1x1)
                            o = make_float4(prelu(o.x, al1[h][0]), prelu(o.y, al1[h][1]), prelu(o.z, al1[h][2]), prelu(o.w, al1[h][3]));
                    }
                    po[4 * h + g] = o;
                }
            }
        }
    }
}

// Grid for a W x H map.
template <int F, class C = ConvTile<F>>
inline dim3 convf_grid(int W, int H) { return dim3((W + C::TW - 1) / C::TW, (H + C::TH - 1) / C::TH); }

} // namespace achip
