// FSRCNNX<F> 2x pass, F = 8 or 16 (core/src/processor/cpu/CPUProcessor.cpp:1629-1659 and the
// F = 16 twin at :1687-1717), layer by layer, FP32 throughout:
//   head   conv5x5 1 -> F, identity                  -> feat         fsrcnnx_head (F = 8), conv_head (16)
//   body   B - 1 x conv3x3 F -> F + PReLU                            kPrelu
//          conv3x3 F -> F + PReLU, conv1x1 F -> F, * 1 + feat, PReLU kPreluConv1x1
//   tail   conv3x3 F -> 4, identity, pixel shuffle 2x -> dst         kShuffle
// (Backend.hpp:225-305; Common.hpp:116-164, 199-341.)  F = 8 runs in conv8_rows, F = 16 in
// convf_rows and convf_tail; the conv1x1 is in the last block's epilogue, fed from the conv3x3's
// own D registers.
// F-channel f32 maps live in HBM between layers, as for ACNet<8> and ArtCNN.
#include "acnet_device.hpp"
#include "acnet_kernels.hpp"
#include "conv_head.hpp"
#include "convf_rows.hpp"

namespace achip {

#pragma clang fp contract(off)

// ---- head of F = 8: conv5x5 1 -> 8, identity; one pixel per thread, 64 x 4 per workgroup ----
// A pixel is two float4 here, and the two stores of a wave fill their lines between them, so a pixel
// per thread keeps up with conv_head and needs no weights in vector registers: the 1001 x 777 u16
// pass takes 83.7 us with it and 85.6 with conv_head (F = 16, 1280 x 720: 203 and 197).
// Taps clamp to the image (Common.hpp:199-225).  The sum follows the reference's FMA order
// (AVX.hpp:93-124): eight lanes accumulate taps l, l + 8, l + 16 with fused multiply-adds,
// their tree sum (AVX.hpp:24-30), then tap 24's rounded product, then the bias.
template <typename TIN, int F>
__global__ __launch_bounds__(256) void fsrcnnx_head(const void* __restrict__ src, long ss, int W, int H,
                                                    float4* __restrict__ feat, long fp, const float* __restrict__ k,
                                                    const float* __restrict__ b)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= W || y >= H) return;
    float r[25];
#pragma unroll
    for (int dy = 0; dy < 5; dy++) {
        const TIN* row = row_ptr<TIN>(src, ss, clampi(y + dy - 2, 0, H - 1));
#pragma unroll
        for (int dx = 0; dx < 5; dx++) r[dy * 5 + dx] = to_float<TIN>(row[clampi(x + dx - 2, 0, W - 1)]);
    }
    float4* px = reinterpret_cast<float4*>(reinterpret_cast<char*>(feat) + static_cast<long>(y) * fp) + (F / 4) * x;
#pragma unroll
    for (int q = 0; q < F / 4; q++) {
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float* kn = k + (4 * q + i) * 25;
            float s[8];
#pragma unroll
            for (int l = 0; l < 8; l++) s[l] = __fmul_rn(r[l], kn[l]);
#pragma unroll
            for (int l = 0; l < 8; l++) s[l] = fmaf(r[8 + l], kn[8 + l], s[l]);
#pragma unroll
            for (int l = 0; l < 8; l++) s[l] = fmaf(r[16 + l], kn[16 + l], s[l]);
            const float a0 = __fadd_rn(s[0], s[4]), a1 = __fadd_rn(s[1], s[5]), a2 = __fadd_rn(s[2], s[6]),
                        a3 = __fadd_rn(s[3], s[7]);
            float sum = __fadd_rn(__fadd_rn(a0, a2), __fadd_rn(a1, a3));
            sum = __fadd_rn(sum, __fmul_rn(r[24], kn[24]));
            o[i] = __fadd_rn(sum, b[4 * q + i]);
        }
        px[q] = make_float4(o[0], o[1], o[2], o[3]);
    }
}

// ---- launch ----

long fsrcnnx_feature_pitch(int f, int w) { return (static_cast<long>(w) * f * 4 + 255) / 256 * 256; }

template <int F, typename TIN, typename TOUT>
static hipError_t fsrcnnx_pass_t(int blocks, const void* src, long ss, int W, int H, void* dst, long ds,
                                 const float* kernels, const float* biases, const float* alphas, const float* wa,
                                 const float* w1, char* ws, int cus, hipStream_t stream)
{
    const long fp = fsrcnnx_feature_pitch(F, W);
    float4* feat = reinterpret_cast<float4*>(ws);
    float4* m0 = reinterpret_cast<float4*>(ws + fp * H);
    float4* m1 = reinterpret_cast<float4*>(ws + 2 * fp * H);
    // every launch's error is its own (the helpers read hipGetLastError): the pass ends at the first
    hipError_t e = hipSuccess;
    if constexpr (F == 8) {
        hipLaunchKernelGGL((fsrcnnx_head<TIN, F>), dim3((W + 63) / 64, (H + 3) / 4), dim3(256), 0, stream, src, ss, W, H, feat,
                           fp, kernels, biases);
        e = hipGetLastError();
    } else {
        e = launch_head<TIN, F, 5>({ src, ss, feat, fp, W, H, 0, kernels, biases }, cus, stream);
    }
    const long wl = static_cast<long>(conv_operand_floats(F));
    auto body_args = [&](int l) {
        LayerArgs la{};
        la.wa = wa + (l - 1) * wl;
        la.bias = biases + F * l;
        la.alpha = alphas + F * (l - 1);
        if (l == blocks) {   // layer `blocks` fused with the conv1x1 (layer blocks + 1) and the skip
            la.w1 = w1;
            la.b1 = biases + F * (blocks + 1);
            la.alpha1 = alphas + F * blocks;
            la.feat = feat;
        }
        return la;
    };
    const float4* in = feat;
    float4* out = m0;
    auto advance = [&]() {
        in = out;
        out = out == m0 ? m1 : m0;
    };
    if constexpr (F == 8) {   // two layers per launch, the last one alone where the count is odd
        for (int l = 1; l <= blocks && e == hipSuccess; l += 2) {
            if (l == blocks) {
                e = launch_rows8<kRowsMap, 1, kRelu, kPreluConv1x1, float, float>(rows8_args(in, out, fp, W, H, { body_args(l) }), cus, stream);
            } else {
                const Rows8 c = rows8_args(in, out, fp, W, H, { body_args(l), body_args(l + 1) });
                e = l + 1 < blocks ? launch_rows8<kRowsMap, 2, kPrelu, kPrelu, float, float>(c, cus, stream)
                                   : launch_rows8<kRowsMap, 2, kPrelu, kPreluConv1x1, float, float>(c, cus, stream);
            }
            advance();
        }
    } else {
        for (int l = 1; l <= blocks && e == hipSuccess; l++) {
            const RowsF c{ in, out, fp, W, H, 0, body_args(l) };
            e = l < blocks ? launch_convf<F, kPrelu>(c, cus, stream) : launch_convf<F, kPreluConv1x1>(c, cus, stream);
            advance();
        }
    }
    if (e != hipSuccess) return e;
    LayerArgs lt{};
    lt.wa = wa + blocks * wl;
    lt.bias = biases + F * (blocks + 2);
    lt.dst = dst;
    lt.ds = ds;
    if constexpr (F == 8)
        return launch_rows8<kRowsMap, 1, kRelu, kShuffle, float, TOUT>(rows8_args(in, nullptr, fp, W, H, { lt }), cus, stream);
    else
        return launch_convf_tail<F, TOUT>({ in, nullptr, fp, W, H, 0, lt }, cus, stream);
}

template <int F>
static hipError_t fsrcnnx_types(int blocks, int stype, int dtype, const void* src, long ss, int W, int H, void* dst,
                                long ds, const float* kernels, const float* biases, const float* alphas,
                                const float* wa, const float* w1, char* ws, int cus, hipStream_t stream)
{
#define CALL(TI, TO) fsrcnnx_pass_t<F, TI, TO>(blocks, src, ss, W, H, dst, ds, kernels, biases, alphas, wa, w1, ws, cus, stream)
    switch (stype) {
    case U8: switch (dtype) {
        case U8: return CALL(uint8_t, uint8_t); case U16: return CALL(uint8_t, uint16_t);
        case F16: return CALL(uint8_t, __half); case F32: return CALL(uint8_t, float);
        default: return hipErrorInvalidValue; }
    case U16: switch (dtype) {
        case U8: return CALL(uint16_t, uint8_t); case U16: return CALL(uint16_t, uint16_t);
        case F16: return CALL(uint16_t, __half); case F32: return CALL(uint16_t, float);
        default: return hipErrorInvalidValue; }
    case F16: switch (dtype) {
        case U8: return CALL(__half, uint8_t); case U16: return CALL(__half, uint16_t);
        case F16: return CALL(__half, __half); case F32: return CALL(__half, float);
        default: return hipErrorInvalidValue; }
    case F32: switch (dtype) {
        case U8: return CALL(float, uint8_t); case U16: return CALL(float, uint16_t);
        case F16: return CALL(float, __half); case F32: return CALL(float, float);
        default: return hipErrorInvalidValue; }
    default: return hipErrorInvalidValue;
    }
#undef CALL
}

hipError_t launch_fsrcnnx(int f, int blocks, int stype, int dtype, const void* src, long ss, int W, int H, void* dst,
                          long ds, const float* kernels, const float* biases, const float* alphas, const float* wa,
                          const float* w1, void* workspace, int cus, hipStream_t stream)
{
    char* ws = static_cast<char*>(workspace);
    if (f == 8)
        return fsrcnnx_types<8>(blocks, stype, dtype, src, ss, W, H, dst, ds, kernels, biases, alphas, wa, w1, ws, cus, stream);
    if (f == 16)
        return fsrcnnx_types<16>(blocks, stype, dtype, src, ss, W, H, dst, ds, kernels, biases, alphas, wa, w1, ws, cus, stream);
    return hipErrorInvalidValue;
}

// ---- host-side operand packing (layouts read by conv8_rows.hpp and convf_rows.hpp) ----

void pack_conv8_operands(const float* k, int cout, float* out)
{
    // operand ((t * 8 + c) * 3 + ky) * halves + h: output channels 4 h .. 4 h + 3 of tap (ky, t),
    // input channel c; 16 operands per register, four lanes each
    const int halves = cout / 4;
    for (int i = 0; i < kRows8Floats; i++) out[i] = 0.0f;
    for (int t = 0; t < 3; t++)
        for (int c = 0; c < 8; c++)
            for (int ky = 0; ky < 3; ky++)
                for (int n = 0; n < cout; n++) {
                    const int s = ((t * 8 + c) * 3 + ky) * halves + n / 4;
                    out[s / 16 * 64 + s % 16 * 4 + n % 4] = k[n * 72 + (ky * 3 + t) * 8 + c];
                }
}

void pack_legacy_l0(const float* k, float* out)
{
    // operand (t * 3 + ky) * 2 + h, as above
    for (int i = 0; i < 2 * 64; i++) out[i] = 0.0f;
    for (int t = 0; t < 3; t++)
        for (int ky = 0; ky < 3; ky++)
            for (int n = 0; n < 8; n++) {
                const int s = (t * 3 + ky) * 2 + n / 4;
                out[s / 16 * 64 + s % 16 * 4 + n % 4] = k[n * 9 + ky * 3 + t];
            }
}

void pack_conv8_1x1(const float* k1, float* out)
{
    // operand i: output channels 4 (i % 2) .., input channel 4 (i / 2 % 2) + i / 4
    for (int i = 0; i < 16; i++)
        for (int r = 0; r < 4; r++) out[i * 4 + r] = k1[(4 * (i % 2) + r) * 8 + 4 * (i / 2 % 2) + i / 4];
}

void pack_convf_operands(const float* k, int f, int cout, float* out)
{
    const int kq = f / 4;
    if (cout == 4) {   // the tail: operand ((t * kq + q) * 4 + g) * 3 + ky, 16 per register
        for (int t = 0; t < 3; t++)
            for (int q = 0; q < kq; q++)
                for (int g = 0; g < 4; g++)
                    for (int ky = 0; ky < 3; ky++)
                        for (int n = 0; n < 4; n++) {
                            const int s = ((t * kq + q) * 4 + g) * 3 + ky;
                            out[s / 16 * 64 + s % 16 * 4 + n] = k[static_cast<size_t>(n) * 9 * f + (ky * 3 + t) * f + g * kq + q];
                        }
        return;
    }
    // output channel lane % f, step s of lane group g = lane / f: channel 4 g + s (16 channels),
    // 8 (2 (s % 2) + g) + s / 2 (32); [tap][s / 4][lane][s % 4]
    const int steps = f == 16 ? 4 : 16;
    for (int p = 0; p < 9; p++)
        for (int s = 0; s < steps; s++)
            for (int lane = 0; lane < 64; lane++) {
                const int o = lane % f, g = lane / f, c = f == 16 ? 4 * g + s : 8 * (2 * (s % 2) + g) + s / 2;
                out[((static_cast<size_t>(p) * (steps / 4) + s / 4) * 64 + lane) * 4 + s % 4] = k[static_cast<size_t>(o) * 9 * f + p * f + c];
            }
}

void pack_convf_1x1(const float* k1, int f, float* out)
{
    // K step 4 h + r of lane group g: input channel 16 h + 4 g + r; output channel 16 h2 + lane % 16
    const int mt = f / 16;
    for (int h = 0; h < mt; h++)
        for (int r = 0; r < 4; r++)
            for (int lane = 0; lane < 64; lane++)
                for (int h2 = 0; h2 < mt; h2++)
                    out[((static_cast<size_t>(4 * h + r)) * 64 + lane) * mt + h2] =
                        k1[(16 * h2 + lane % 16) * f + 16 * h + 4 * (lane / 16) + r];
}

} // namespace achip
