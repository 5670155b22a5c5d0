// The FP32 conv3x3 layers of 16 and 32 channels (ArtCNN<F>, FSRCNNX<16>), one launch per layer over
// F-channel f32 maps in HBM (channel quads interleaved per pixel: pixel x at float4 index
// F/4 * x + q, rows of `fp` bytes).
//
// convf_rows, F -> F: every wave is a strip of its own, 32 columns by `rows` rows, with all of the
// layer's weights in registers (through LDS once, at the start) and no barrier after that.  M is the
// output channels of v_mfma_f32_32x32x2_f32 (F = 32) or 16x16x4 (F = 16, two blocks of 16 columns),
// N pixels of one row, and the lane groups read their input channels straight from the map.  An
// input row is loaded once and goes into three output rows (tap row 0 of the next, 1 of its own, 2
// of the one before), and a tap column's registers are loaded with the next row as soon as its MFMAs
// are issued.  A lane's sums hold 4 consecutive channels of a pixel, which with 16 channels is
// exactly the B operand a conv1x1 MFMA needs (K step i of lane group g = channel 4 g + i), so the
// fused conv1x1 costs four MFMAs and no data movement.
//
// convf_tail, F -> 4 and the pixel shuffle: v_mfma_f32_4x4x1_16b_f32 (conv8_rows.hpp), whose M is
// the four sub-pixels, on 64 pixels of a row per wave from a row of its own in LDS.
//
// Both add an output's products in the same order: tap row, tap column, q = 0 .. F/4 - 1, then
// channels q, F/4 + q, 2 F/4 + q, 3 F/4 + q.
//
// Bound by the matrix pipe and, with 16 channels, nearly as much by HBM (F 4 bytes in and out per
// pixel).  1280 x 720 maps, us: F = 32 155-165 as 16 x 16 tiles in LDS (the pipe 62-68% busy),
// 126 in strips of 29 rows (90%; without the loads 118), 146 with two waves of 16 columns on every
// SIMD instead of one of 32; F = 16 54 / 42 (15 rows, two waves per SIMD, 50; twice the look-ahead
// 44).  The last layer of ArtCNN<32> 88 / 31 (a 16x16x4 MFMA has 12 of its 16 rows idle there), of
// FSRCNNX<16> 34 / 16.  Passes: ArtCNN<32> 961 / 717, ArtCNN<16> 312 / 224, FSRCNNX<16> 285 / 203.
#pragma once

#include <utility>

#include "acnet_mfma32_item.hpp"   // mma32
#include "conv8_rows.hpp"          // mma4, quad
#include "conv_layers.hpp"

namespace achip {

#pragma clang fp contract(off)

struct RowsF {
    const float4* fin;
    float4* fout;
    long fp;
    int W, H, rows;
    LayerArgs la;
};

// The MFMA of a layer: PX pixels x F output channels, STEPS per tap.  Lane group g's input channels
// of a pixel are NQ quads from byte in(v), its output channels NQ quads at byte out(k); step s
// multiplies component c(s) of quad v(s) with operand s of the tap.
template <int F>
struct LayerMfma;

template <>
struct LayerMfma<16> {   // v_mfma_f32_16x16x4_f32: step q, lane group g: channel 4 g + q
    static constexpr int PX = 16, NB = 2, STEPS = 4, NQ = 1;
    typedef f32x4m Acc;
    static constexpr int in(int) { return 0; }
    static constexpr int kIn = 16, kOut = 16;   // bytes from a lane group to the next
    static constexpr int out(int) { return 0; }
    static constexpr int v(int) { return 0; }
    static constexpr int c(int s) { return s; }
    static __device__ __forceinline__ Acc mma(float a, float b, Acc x) { return mma32(a, b, x); }
};

template <>
struct LayerMfma<32> {   // v_mfma_f32_32x32x2_f32: step 2 q + p, lane half h: channel 8 (2 p + h) + q
    static constexpr int PX = 32, NB = 1, STEPS = 16, NQ = 4;
    typedef float Acc __attribute__((ext_vector_type(16)));
    static constexpr int in(int v) { return 64 * (v >> 1) + 16 * (v & 1); }
    static constexpr int kIn = 32, kOut = 16;
    static constexpr int out(int k) { return 32 * k; }
    static constexpr int v(int s) { return 2 * (s & 1) + (s >> 3); }
    static constexpr int c(int s) { return (s >> 1) & 3; }
    static __device__ __forceinline__ Acc mma(float a, float b, Acc x) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, x, 0, 0, 0); }
};

typedef unsigned QuadBits __attribute__((vector_size(16)));
constexpr int kStripF = 32;   // columns of a strip: NB blocks of PX

template <int F, int MODE, int WAVES>
__global__ __launch_bounds__(256, WAVES) void convf_rows(const RowsF c)
{
    typedef LayerMfma<F> M;
    typedef typename M::Acc Acc;
    constexpr int NB = M::NB, PX = M::PX, NQ = M::NQ, STEPS = M::STEPS, NW = 9 * STEPS / 4 * 64;
    constexpr bool PRELU = MODE == kPrelu || MODE == kPreluConv1x1, FEAT = MODE == kAddFeat || MODE == kPreluConv1x1;
    static_assert(MODE != kPreluConv1x1 || F == 16, "the fused conv1x1");
    __shared__ f32x4m lds[NW];
    const LayerArgs& la = c.la;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane / PX, j = lane % PX;
    const int strips = (c.W + kStripF - 1) / kStripF, id = xcd_tile(blockIdx.x, gridDim.x) * 4 + wave;
    const int ty = id / strips, x0 = (id - ty * strips) * kStripF;
    const int y0 = ty * c.rows, y1 = min(y0 + c.rows, c.H);

    // this lane's channels of patch columns 0-2, one input row, from the strip's first input column on
    const int xb = max(x0 - 1, 0);
    int off[3][NB];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int n = 0; n < NB; n++) off[d][n] = (clampi(x0 + PX * n + j + d - 1, 0, c.W - 1) - xb) * (4 * F) + g * M::kIn;
    f32x4m b[3][NB][NQ];
    auto fetch = [&](int d, int r) {
        const char* row = reinterpret_cast<const char*>(c.fin) + static_cast<long>(clampi(r, 0, c.H - 1)) * c.fp + static_cast<long>(xb) * (4 * F);
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int v = 0; v < NQ; v++) b[d][n][v] = *reinterpret_cast<const f32x4m*>(row + off[d][n] + M::in(v));
    };
#pragma unroll
    for (int d = 0; d < 3; d++) fetch(d, y0 - 1);
    // the weights: once per workgroup from memory
    const f32x4m* const wa = reinterpret_cast<const f32x4m*>(la.wa);
#pragma unroll
    for (int k = 0; k < (NW + 255) / 256; k++)
        if (NW % 256 == 0 || threadIdx.x + 256 * k < NW) lds[threadIdx.x + 256 * k] = wa[threadIdx.x + 256 * k];
    // element 4 k + i of a lane's sums: channel 4 (F/4 quad at byte out(k) + g * kOut) + i
    Acc bias;
    float al[PRELU ? 4 : 1], al1[MODE == kPreluConv1x1 ? 4 : 1], w1[4];
    f32x4m bias1;
#pragma unroll
    for (int i = 0; i < 4 * NQ; i++) bias[i] = la.bias[(M::out(i / 4) + g * M::kOut) / 4 + i % 4];
    if constexpr (PRELU)
#pragma unroll
        for (int i = 0; i < 4; i++) al[i] = la.alpha[4 * g + i];
    if constexpr (MODE == kPreluConv1x1)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            bias1[i] = la.b1[4 * g + i];
            al1[i] = la.alpha1[4 * g + i];
            w1[i] = la.w1[i * 64 + lane];   // K step i of lane group g is channel 4 g + i
        }
    __syncthreads();
    if (y0 >= c.H) return;
    float a[9][STEPS];
#pragma unroll
    for (int p = 0; p < 9; p++)
#pragma unroll
        for (int v = 0; v < STEPS / 4; v++) {
            const f32x4m f = lds[(p * (STEPS / 4) + v) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; i++) a[p][4 * v + i] = f[i];
        }

    // the strip's part of a row of the output or the skip map as a buffer: the stores of lanes right
    // of the image fall outside it and are dropped, with no branch to end the loads' overlap
    const int px = j * (4 * F) + g * M::kOut, row_bytes = min(c.W - x0, kStripF) * (4 * F);
    auto row_of = [&](const float4* map, int y) {
        return __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<char*>(const_cast<float4*>(map)) + static_cast<long>(y) * c.fp + static_cast<long>(x0) * (4 * F), 0, row_bytes,
            0x00020000);
    };
    f32x4m feat[NB][NQ];
    auto ahead = [&](int y) {
        if constexpr (FEAT) {
            const auto row = row_of(la.feat, y);
#pragma unroll
            for (int n = 0; n < NB; n++)
#pragma unroll
                for (int k = 0; k < NQ; k++)
                    feat[n][k] = __builtin_bit_cast(f32x4m, __builtin_amdgcn_raw_buffer_load_b128(row, px + n * PX * 4 * F + M::out(k), 0, 0));
        }
    };
    auto finish = [&](int y, Acc (&done)[NB]) {   // output row y from its sums
        const auto row = row_of(c.fout, y);
#pragma unroll
        for (int n = 0; n < NB; n++) {
            if constexpr (MODE == kPreluConv1x1) {
                f32x4m d = bias1;
#pragma unroll
                for (int i = 0; i < 4; i++) d = mma32(w1[i], prelu(done[n][i], al[i]), d);
                done[n] = d;
            }
#pragma unroll
            for (int k = 0; k < NQ; k++) {
                f32x4m v;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    v[i] = done[n][4 * k + i];
                    if constexpr (MODE == kRelu) v[i] = fmaxf(v[i], 0.f);
                    else if constexpr (MODE == kPrelu) v[i] = prelu(v[i], al[i]);
                    else v[i] = add_skip(v[i], feat[n][k][i]);   // * 1 + feat (then PReLU)
                    if constexpr (MODE == kPreluConv1x1) v[i] = prelu(v[i], al1[i]);
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(QuadBits, v), row, px + n * PX * 4 * F + M::out(k), 0, 0);
            }
        }
    };

    // Input row r into the sums of rows r + 1, r, r - 1, which take its tap rows 0, 1, 2 (bits 0-2 of
    // `taps`); row r - 2, whose sums are `done`, is finished meanwhile (bit 3).
    auto input_row = [&](int r, auto taps, Acc (&s0)[NB], Acc (&s1)[NB], Acc (&s2)[NB], Acc (&done)[NB]) {
        constexpr bool T0 = decltype(taps)::value & 1, T1 = decltype(taps)::value & 2, T2 = decltype(taps)::value & 4,
                       FIN = decltype(taps)::value & 8;
#pragma unroll
        for (int d = 0; d < 3; d++) {
#pragma unroll
            for (int s = 0; s < STEPS; s++)
#pragma unroll
                for (int n = 0; n < NB; n++) {
                    const float bv = b[d][n][M::v(s)][M::c(s)];
                    if constexpr (T0) s0[n] = M::mma(a[d][s], bv, d == 0 && s == 0 ? bias : s0[n]);
                    if constexpr (T1) s1[n] = M::mma(a[3 + d][s], bv, s1[n]);
                    if constexpr (T2) s2[n] = M::mma(a[6 + d][s], bv, s2[n]);
                }
            // here and no later: the next row's registers are this one's
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (T0 || T1) fetch(d, r + 1);
            if (d == 0) {
                if constexpr (FIN) finish(r - 2, done);
                if constexpr (T2) ahead(r - 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    Acc A[NB], B[NB], C[NB], D[NB];
    using std::integral_constant;
    constexpr integral_constant<int, 15> all{};
    // the sums take turns: a row's s0, s1, s2, done are the next one's s1, s2, done, s0
    input_row(y0 - 1, integral_constant<int, 1>{}, A, B, C, D);
    if (y1 - y0 == 1) {
        input_row(y0, integral_constant<int, 2>{}, D, A, B, C);
        input_row(y1, integral_constant<int, 4>{}, C, D, A, B);
        finish(y0, A);
        return;
    }
    input_row(y0, integral_constant<int, 3>{}, D, A, B, C);
    if (y1 - y0 == 2) {
        input_row(y0 + 1, integral_constant<int, 6>{}, C, D, A, B);
        input_row(y1, integral_constant<int, 12>{}, B, C, D, A);
        finish(y1 - 1, D);
        return;
    }
    input_row(y0 + 1, integral_constant<int, 7>{}, C, D, A, B);
    int r = y0 + 2;
    for (; r + 4 < y1; r += 4) {
        input_row(r, all, B, C, D, A);
        input_row(r + 1, all, A, B, C, D);
        input_row(r + 2, all, D, A, B, C);
        input_row(r + 3, all, C, D, A, B);
    }
    auto turn = [&]() {   // rename a row on
#pragma unroll
        for (int n = 0; n < NB; n++) {
            const Acc t = A[n];
            A[n] = D[n];
            D[n] = C[n];
            C[n] = B[n];
            B[n] = t;
        }
    };
    for (; r < y1 - 1; r++) {
        input_row(r, all, B, C, D, A);
        turn();
    }
    input_row(y1 - 1, integral_constant<int, 14>{}, B, C, D, A);
    input_row(y1, integral_constant<int, 12>{}, A, B, C, D);
    finish(y1 - 1, C);
}

// ---- F -> 4, pixel shuffle 2x ----

constexpr int kTailCols = 64;
template <int F>
constexpr int tail_operands() { return 9 * F; }   // ((tap column * F/4 + q) * 4 + g) * 3 + tap row: channel g F/4 + q

// One tap column of an input row into the sums whose tap rows TAPS names (bits 0-2)
template <int F, int D, int TAPS, int... I>
__device__ __forceinline__ void tail_column(const float* w, const f32x4m (&q)[F / 4], f32x4m& s0, f32x4m& s1, f32x4m& s2,
                                            std::integer_sequence<int, I...>)
{
    auto step = [&](auto i) {   // i = q * 4 + g
        constexpr int I0 = decltype(i)::value, SLOT = (D * F + I0) * 3, C = I0 % 4 * (F / 4) + I0 / 4;
        const float b = q[C / 4][C % 4];
        if constexpr (TAPS & 1) s0 = mma4<SLOT>(w, b, s0);
        if constexpr (TAPS & 2) s1 = mma4<SLOT + 1>(w, b, s1);
        if constexpr (TAPS & 4) s2 = mma4<SLOT + 2>(w, b, s2);
    };
    (step(std::integral_constant<int, I>{}), ...);
}

// `at`: this lane's first patch pixel in plane 0
template <int F, int PITCH, int TAPS, int D = 0>
__device__ __forceinline__ void tail_row(const float* w, const char* at, f32x4m& s0, f32x4m& s1, f32x4m& s2)
{
    f32x4m q[F / 4];
#pragma unroll
    for (int i = 0; i < F / 4; i++) q[i] = *reinterpret_cast<const f32x4m*>(at + i * PITCH + D * 16);
    tail_column<F, D, TAPS>(w, q, s0, s1, s2, std::make_integer_sequence<int, F>{});
    if constexpr (D < 2) tail_row<F, PITCH, TAPS, D + 1>(w, at, s0, s1, s2);
}

template <int F, typename TOUT>
__global__ __launch_bounds__(256, F == 32 ? 2 : 4) void convf_tail(const RowsF c)
{
    constexpr int KQ = F / 4, NQ = F / 4, CW = kTailCols + 2, N = CW * NQ, K = (N + 63) / 64, PITCH = CW * 16 + 16;
    __shared__ float4 lds[4][NQ * PITCH / 16];
    const LayerArgs& la = c.la;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int strips = (c.W + kTailCols - 1) / kTailCols, id = xcd_tile(blockIdx.x, gridDim.x) * 4 + wave;
    const int ty = id / strips, x0 = (id - ty * strips) * kTailCols, y0 = ty * c.rows, y1 = min(y0 + c.rows, c.H);
    if (y0 >= c.H) return;
    char* const buf = reinterpret_cast<char*>(lds[wave]);

    const int xb = max(x0 - 1, 0);   // the first input column
    int at[K], off[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int e = min(lane + 64 * k, N - 1);
        off[k] = (clampi(x0 - 1 + e / NQ, 0, c.W - 1) - xb) * (4 * F) + e % NQ * 16;
        at[k] = e % NQ * PITCH + e / NQ * 16;
    }
    f32x4m v[K];
    auto fetch = [&](int r) {
        const char* row = reinterpret_cast<const char*>(c.fin) + static_cast<long>(clampi(r, 0, c.H - 1)) * c.fp + static_cast<long>(xb) * (4 * F);
#pragma unroll
        for (int k = 0; k < K; k++) v[k] = *reinterpret_cast<const f32x4m*>(row + off[k]);
    };
    fetch(y0 - 1);
    float w[tail_operands<F>() / 16];
#pragma unroll
    for (int i = 0; i < tail_operands<F>() / 16; i++) w[i] = la.wa[i * 64 + lane];
    const f32x4m bias = { la.bias[0], la.bias[1], la.bias[2], la.bias[3] };
    f32x4m s0 = bias, s1 = bias, s2 = bias;
    const int x = x0 + lane;
    auto input_row = [&](int r, auto taps) {
        constexpr int TAPS = decltype(taps)::value;
        // only this wave reads what it stores, and a wave's LDS operations stay in order
#pragma unroll
        for (int k = 0; k < K; k++) *reinterpret_cast<f32x4m*>(buf + at[k]) = v[k];
        if constexpr (TAPS & 3) fetch(r + 1);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        s0 = bias;
        tail_row<F, PITCH, TAPS>(w, buf + lane * 16, s0, s1, s2);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if constexpr (TAPS & 4) {
            if (x < c.W) {
                const int y = r - 1;
                store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y) + 2 * x, s2[0], s2[1]);
                store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y + 1) + 2 * x, s2[2], s2[3]);
            }
        }
        s2 = s1;
        s1 = s0;
    };
    using std::integral_constant;
    input_row(y0 - 1, integral_constant<int, 1>{});
    if (y1 - y0 == 1) {
        input_row(y0, integral_constant<int, 2>{});
    } else {
        input_row(y0, integral_constant<int, 3>{});
        for (int r = y0 + 1; r < y1 - 1; r++) input_row(r, integral_constant<int, 7>{});
        input_row(y1 - 1, integral_constant<int, 6>{});
    }
    input_row(y1, integral_constant<int, 4>{});
}

// ---- launch ----

// Rows per strip, a strip per wave, at most `most` waves per SIMD: the heights that put 1, 2, .. of
// them on every SIMD, or two and four rounds of the most, by rows per SIMD plus `lead` rows to start.
inline int convf_heights(long strips, int H, int cus, int most, int lead)
{
    long best = -1;
    int rows = 64;   // more strips than four rounds take
    for (int k = 1; k <= most + 2; k++) {
        const int at = k < most ? k : most, rounds = k <= most ? 1 : k == most + 1 ? 2 : 4;
        const long slots = 4L * at * cus, segs = slots * rounds / strips;
        if (segs < 1) continue;
        const int r = static_cast<int>((H + segs - 1) / segs);
        const long waves = strips * ((H + r - 1) / r);
        const long cost = (waves + slots - 1) / slots * (static_cast<long>(at) * r + lead);
        if (best < 0 || cost <= best) {
            best = cost;
            rows = r;
        }
    }
    return rows;
}

template <int F, int MODE>
inline hipError_t launch_convf(RowsF c, int cus, hipStream_t stream)
{
    constexpr int WAVES = F == 32 ? 1 : 2;
    const int strips = (c.W + kStripF - 1) / kStripF;
    c.rows = convf_heights(strips, c.H, cus, WAVES, 1);
    const int n = strips * ((c.H + c.rows - 1) / c.rows);
    hipLaunchKernelGGL((convf_rows<F, MODE, WAVES>), dim3((n + 3) / 4), dim3(256), 0, stream, c);
    return hipGetLastError();
}

template <int F, typename TOUT>
inline hipError_t launch_convf_tail(RowsF c, int cus, hipStream_t stream)
{
    const int strips = (c.W + kTailCols - 1) / kTailCols;
    c.rows = convf_heights(strips, c.H, cus, F == 32 ? 2 : 4, 2);
    const int n = strips * ((c.H + c.rows - 1) / c.rows);
    hipLaunchKernelGGL((convf_tail<F, TOUT>), dim3((n + 3) / 4), dim3(256), 0, stream, c);
    return hipGetLastError();
}

} // namespace achip
