// ArtCNN<F> 2x pass, F = 16 or 32 (core/src/processor/cpu/CPUProcessor.cpp:1519-1546 and the
// F = 32 twin), layer by layer, FP32 throughout:
//   head   conv3x3 1 -> F, identity                   -> feat        conv_head
//   body   B x conv3x3 F -> F + ReLU                                  convf_rows<kRelu>
//          conv3x3 F -> F, identity, + feat                           convf_rows<kAddFeat>
//   tail   conv3x3 F -> 4, identity, pixel shuffle 2x -> dst          convf_tail
// (Backend.hpp:135-215; Common.hpp:116-164, 290-341.)  F-channel f32 maps live in HBM between
// layers (convf_rows.hpp).
#include "acnet_device.hpp"
#include "acnet_kernels.hpp"
#include "conv_head.hpp"
#include "convf_rows.hpp"

namespace achip {

#pragma clang fp contract(off)

// ---- launch ----

long artcnn_feature_pitch(int f, int w) { return (static_cast<long>(w) * f * 4 + 255) / 256 * 256; }

template <int F, typename TIN, typename TOUT>
static hipError_t artcnn_pass_t(int blocks, const void* src, long ss, int W, int H, void* dst, long ds,
                                const float* kernels, const float* biases, const float* wa, char* ws, int cus, hipStream_t stream)
{
    const long fp = artcnn_feature_pitch(F, W);
    float4* feat = reinterpret_cast<float4*>(ws);
    float4* m0 = reinterpret_cast<float4*>(ws + fp * H);
    float4* m1 = reinterpret_cast<float4*>(ws + 2 * fp * H);
    // every launch's error is its own (the helpers read hipGetLastError): the pass ends at the first
    hipError_t e = launch_head<TIN, F, 3>({ src, ss, feat, fp, W, H, 0, kernels, biases }, cus, stream);
    const long wl = static_cast<long>(conv_operand_floats(F));   // A-operand floats per layer
    const float4* in = feat;
    float4* out = m0;
    for (int l = 1; l <= blocks && e == hipSuccess; l++) {   // body: F -> F + ReLU
        LayerArgs la{};
        la.wa = wa + (l - 1) * wl;
        la.bias = biases + F * l;
        e = launch_convf<F, kRelu>({ in, out, fp, W, H, 0, la }, cus, stream);
        in = out;
        out = out == m0 ? m1 : m0;
    }
    if (e != hipSuccess) return e;
    LayerArgs la{};
    la.wa = wa + blocks * wl;
    la.bias = biases + F * (blocks + 1);
    la.feat = feat;
    e = launch_convf<F, kAddFeat>({ in, out, fp, W, H, 0, la }, cus, stream);
    if (e != hipSuccess) return e;
    LayerArgs lt{};
    lt.wa = wa + (blocks + 1) * wl;
    lt.bias = biases + F * (blocks + 2);
    lt.dst = dst;
    lt.ds = ds;
    return launch_convf_tail<F, TOUT>({ out, nullptr, fp, W, H, 0, lt }, cus, stream);
}

template <int F>
static hipError_t artcnn_types(int blocks, int stype, int dtype, const void* src, long ss, int W, int H, void* dst, long ds,
                               const float* kernels, const float* biases, const float* wa, char* ws, int cus, hipStream_t stream)
{
#define CALL(TI, TO) artcnn_pass_t<F, TI, TO>(blocks, src, ss, W, H, dst, ds, kernels, biases, wa, ws, cus, stream)
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

hipError_t launch_artcnn(int f, int blocks, int stype, int dtype, const void* src, long ss, int W, int H, void* dst,
                         long ds, const float* kernels, const float* biases, const float* wa, void* workspace,
                         int cus, hipStream_t stream)
{
    char* ws = static_cast<char*>(workspace);
    if (f == 16) return artcnn_types<16>(blocks, stype, dtype, src, ss, W, H, dst, ds, kernels, biases, wa, ws, cus, stream);
    if (f == 32) return artcnn_types<32>(blocks, stype, dtype, src, ss, W, H, dst, ds, kernels, biases, wa, ws, cus, stream);
    return hipErrorInvalidValue;
}

} // namespace achip
