// The first layer of ArtCNN<F> (conv3x3 1 -> F, identity) and FSRCNNX<16> (conv5x5), from the source
// image to an F-channel f32 map, each product and sum rounded in the reference's order.
//
// A lane computes four channels: F/4 neighbouring lanes make a pixel, so that a wave's store is 1 KB
// of the map without gaps.  Its weights (36 or 100) stay in registers while the wave goes down its
// strip, with the window's K rows in registers as well; a row's K new samples are loaded one row
// ahead.  Bound by the map's way to HBM and the vector ALU, about equally (ArtCNN<32>: 128 bytes and
// 608 rounded operations per pixel).
// Before, a pixel per thread stored F/4 quads at a stride of F floats.  1280 x 720, in a pass: ArtCNN<32>
// 50 / 38 us (118 MB written), ArtCNN<16> 25 / 17, FSRCNNX<16> 30 / 26.
#pragma once

#include "acnet_device.hpp"
#include "convf_rows.hpp"

namespace achip {

#pragma clang fp contract(off)

// Four channels of a pixel from its window, oldest row in slot S of r
template <int S>
__device__ __forceinline__ f32x4m head_sum(const float (&r)[3][3], const float* w, const float (&b)[4])
{
    // ArtCNN: one rounded product after the other (Common.hpp:116-164)
    f32x4m o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float s = 0.0f;
#pragma unroll
        for (int p = 0; p < 9; p++) s = __fadd_rn(s, __fmul_rn(r[(S + p / 3) % 3][p % 3], w[i * 9 + p]));
        o[i] = __fadd_rn(s, b[i]);
    }
    return o;
}

template <int S>
__device__ __forceinline__ f32x4m head_sum(const float (&r)[5][5], const float* w, const float (&b)[4])
{
    // FSRCNNX: the reference's FMA order (AVX.hpp:93-124): eight lanes accumulate taps l, l + 8, l + 16
    // with fused multiply-adds, their tree sum (AVX.hpp:24-30), then tap 24's rounded product, then
    // the bias
    f32x4m o;
    auto tap = [&](int t) { return r[(S + t / 5) % 5][t % 5]; };
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float* k = w + i * 25;
        float s[8];
#pragma unroll
        for (int l = 0; l < 8; l++) s[l] = __fmul_rn(tap(l), k[l]);
#pragma unroll
        for (int l = 0; l < 8; l++) s[l] = fmaf(tap(8 + l), k[8 + l], s[l]);
#pragma unroll
        for (int l = 0; l < 8; l++) s[l] = fmaf(tap(16 + l), k[16 + l], s[l]);
        const float a0 = __fadd_rn(s[0], s[4]), a1 = __fadd_rn(s[1], s[5]), a2 = __fadd_rn(s[2], s[6]), a3 = __fadd_rn(s[3], s[7]);
        float sum = __fadd_rn(__fadd_rn(a0, a2), __fadd_rn(a1, a3));
        sum = __fadd_rn(sum, __fmul_rn(tap(24), k[24]));
        o[i] = __fadd_rn(sum, b[i]);
    }
    return o;
}

struct HeadArgs {
    const void* src;
    long ss;
    float4* map;
    long fp;
    int W, H, rows;
    const float* k;   // [channel][tap]
    const float* b;
};

template <int F>
constexpr int head_cols() { return 64 / (F / 4); }

template <typename TIN, int F, int K>
__global__ __launch_bounds__(256) void conv_head(const HeadArgs c)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int strips = (c.W + head_cols<F>() - 1) / head_cols<F>(), id = xcd_tile(strip_block(), gridDim.x * gridDim.y) * 4 + wave;
    const int ty = id / strips, x = (id - ty * strips) * head_cols<F>() + lane / (F / 4), q = lane % (F / 4);
    const int y0 = ty * c.rows, y1 = min(y0 + c.rows, c.H);
    if (y0 >= c.H) return;
    int col[K];
#pragma unroll
    for (int d = 0; d < K; d++) col[d] = clampi(x + d - K / 2, 0, c.W - 1);
    TIN ahead[K];
    auto fetch = [&](int r) {
        const TIN* row = row_ptr<TIN>(c.src, c.ss, clampi(r, 0, c.H - 1));
#pragma unroll
        for (int d = 0; d < K; d++) ahead[d] = row[col[d]];
    };
    float r[K][K];   // row y - K/2 + i of the strip's first window in slot i
    auto take = [&](int slot) {
#pragma unroll
        for (int d = 0; d < K; d++) r[slot][d] = to_float<TIN>(ahead[d]);
    };
    fetch(y0 - K / 2);
    float w[4 * K * K], b[4];
#pragma unroll
    for (int i = 0; i < 4 * K * K; i++) w[i] = c.k[q * 4 * K * K + i];
#pragma unroll
    for (int i = 0; i < 4; i++) b[i] = c.b[4 * q + i];
#pragma unroll
    for (int i = 0; i < K - 1; i++) {
        take(i);
        fetch(y0 - K / 2 + i + 1);
    }
    float4* const out = c.map + (F / 4) * static_cast<long>(x) + q;
    // K rows per turn, so that the slots are constants; S: the slot of the window's first row
    auto step = [&](int y, auto slot) {
        constexpr int S = decltype(slot)::value;
        take((S + K - 1) % K);
        fetch(y + K / 2 + 1);
        const f32x4m o = head_sum<S>(r, w, b);
        if (x < c.W) *reinterpret_cast<f32x4m*>(reinterpret_cast<char*>(out) + static_cast<long>(y) * c.fp) = o;
    };
    for (int y = y0; y < y1; y += K) {
        step(y, std::integral_constant<int, 0>{});
        if (y + 1 < y1) step(y + 1, std::integral_constant<int, 1>{});
        if (y + 2 < y1) step(y + 2, std::integral_constant<int, 2>{});
        if constexpr (K == 5) {
            if (y + 3 < y1) step(y + 3, std::integral_constant<int, 3>{});
            if (y + 4 < y1) step(y + 4, std::integral_constant<int, 4>{});
        }
    }
}

// Rows per strip, a strip per wave: the height that puts 1 .. `most` of them on every SIMD by what
// their rows and the K to start take, a row of k waves k + 1 times one's operations (1280 x 720,
// ArtCNN<32>: 120 rows 43.3 us, 60 26.8, 20 21.0, 6 21.7; FSRCNNX<16>: 60 rows 33.5, 20 21.9, 10 24.6).
inline int head_heights(long strips, int H, int cus, int most, int K)
{
    long best = -1;
    int rows = H;
    for (int k = 1; k <= most; k++) {
        const long segs = 4L * k * cus / strips;
        if (segs < 1) continue;
        const int r = static_cast<int>((H + segs - 1) / segs);
        const long cost = (k + 1L) * (r + K);
        if (best < 0 || cost < best) {
            best = cost;
            rows = r;
        }
    }
    return best < 0 ? 64 : rows;   // more strips than fit: any height that is long against K
}

template <typename TIN, int F, int K>
inline hipError_t launch_head(HeadArgs c, int cus, hipStream_t stream)
{
    const int strips = (c.W + head_cols<F>() - 1) / head_cols<F>();
    c.rows = head_heights(strips, c.H, cus, K == 3 ? 6 : 3, K);
    const int n = strips * ((c.H + c.rows - 1) / c.rows);
    hipLaunchKernelGGL((conv_head<TIN, F, K>), strip_row((n + 3) / 4, 256), dim3(256), 0, stream, c);
    return hipGetLastError();
}

} // namespace achip
