// The FP32 passes of the 8-channel networks, a few layers per launch (conv8_rows.hpp):
//   ACNet<8> (core/src/processor/cpu/CPUProcessor.cpp:1417-1436)
//     L0     conv3x3 1 -> 8 + PReLU            (Backend.hpp:58-75)        from the source rows in the first launch
//     L1..LB conv3x3 8 -> 8 + PReLU            (Backend.hpp:95-98)
//     final  conv3x3 8 -> 4, pixel shuffle 2x, + the source pixel  (Backend.hpp:116-133, Common.hpp:290-341)
//   ACNetLegacy, the layer-split form of the fused FP32 pass, with its bits
//     L0 conv3x3 1 -> 8 + ReLU, L1..L8 conv3x3 8 -> 8 + ReLU, deconv 2x2 8 -> 1 (Backend.hpp:17-56)
// Features between launches are 8-channel f32 maps in HBM (32 bytes per pixel, rows padded to 256
// bytes).  Borders replicate the edge pixel at every layer, as the reference's clamped taps
// (Common.hpp:120-160) do.
#include <algorithm>
#include <cmath>
#include <utility>

#include "acnet_device.hpp"
#include "acnet_kernels.hpp"
#include "conv8_rows.hpp"

namespace achip {

#pragma clang fp contract(off)

long acnet8_feature_pitch(int w) { return (static_cast<long>(w) * 32 + 255) / 256 * 256; }

// The layers of a pass, split into launches: `head` of them with layer 0, then `pair` (0 or 1) of
// two layers and the rest `per` at a time, at least one launch after the head.
//
// Two layers per launch keep 62 of the 64 columns computed (the head 60) and fill a CU with four
// strips; four layers keep 58 (56), take half the launches and passes over HBM, and start four
// layers' pipelines instead of twice two.  So four where the pairs' strips would be short, up to 12
// rows with four strips on every CU (us, pairs / fours; ACNetLegacy, then ACNet<8> of 18 blocks):
//   128 x 96   23.2 / 20.1   54.7 / 48.6      960 x 540    85.1 / 81.1   204 / 188
//   480 x 270  40.1 / 34.8   96.9 / 85.3     1280 x 720   118.0 / 125    282 / 302
//   720 x 480  66.0 / 61.0   157  / 148      1920 x 1080  213   / 233    548 / 545
// The head takes what is left over, three layers rather than one (5 layers at 1080p: 3 + 2 151 us,
// 1 + 4 167, 1 + 2 + 2 161); launches of three layers in between are slower than either (2 + 3 162).
struct Split8 {
    int head, pair, per;
};

static Split8 split8(int total, int W, int H, int cus)
{
    const long strips = (W + (rows8_out<kRowsMap, 2>()) - 1) / (rows8_out<kRowsMap, 2>());
    const bool fours = strips * H <= 12L * (rows8_per_cu<kRowsMap, 2>()) * cus;
    if (total <= 3) return { 1, 0, total - 1 };
    // three layers in the head are 512 threads: not for images of more columns than most_strips takes
    // (487 Mpix; the other launches take any width)
    const bool wide = (W + rows8_out<kRowsAcnet8, 3>() - 1) / (rows8_out<kRowsAcnet8, 3>()) > most_strips(rows8_threads<kRowsAcnet8, 3>());
    if (!fours || total == 4) return { total % 2 ? (wide ? 1 : 3) : 2, 0, 2 };
    switch (total % 4) {
    case 0: return { 4, 0, 4 };
    case 1: return { 3, 1, 4 };
    default: return { total % 4, 0, 4 };
    }
}

template <int MID>
static hipError_t map_launch(int n, const Rows8& c, int cus, hipStream_t stream)
{
    return n == 2 ? launch_rows8<kRowsMap, 2, MID, MID, float, float>(c, cus, stream)
                  : launch_rows8<kRowsMap, 4, MID, MID, float, float>(c, cus, stream);
}

template <int MID, int MODE, typename TIN, typename TOUT>
static hipError_t last_launch(int n, const Rows8& c, int cus, hipStream_t stream)
{
    if constexpr (MODE == kShuffleSrc)   // ACNet<8> of one block
        if (n == 1) return launch_rows8<kRowsMap, 1, MID, MODE, TIN, TOUT>(c, cus, stream);
    return n == 2 ? launch_rows8<kRowsMap, 2, MID, MODE, TIN, TOUT>(c, cus, stream)
                  : launch_rows8<kRowsMap, 4, MID, MODE, TIN, TOUT>(c, cus, stream);
}

template <int HEAD, int MODE, typename TIN>
static hipError_t head_launch(int n, const Rows8& c, int cus, hipStream_t stream)
{
    if constexpr (HEAD == kRowsAcnet8) {   // odd heads: layer counts other than ACNetLegacy's 8
        if (n == 1) return launch_rows8<HEAD, 1, MODE, MODE, TIN, float>(c, cus, stream);
        if (n == 3) return launch_rows8<HEAD, 3, MODE, MODE, TIN, float>(c, cus, stream);
    }
    return n == 2 ? launch_rows8<HEAD, 2, MODE, MODE, TIN, float>(c, cus, stream)
                  : launch_rows8<HEAD, 4, MODE, MODE, TIN, float>(c, cus, stream);
}

// Layers 1 .. total (layer(l): their arguments), split as split8 says; the last one ends in MODE.
template <int HEAD, int MID, int MODE, typename TIN, typename TOUT, class Layer>
static hipError_t rows8_pass(const Rows8& args, int total, Layer layer, float4* f0, float4* f1, int cus, hipStream_t stream)
{
    const Split8 sp = split8(total, args.W, args.H, cus);
    Rows8 c = args;
    float4 *in = f0, *out = f1;
    c.fout = in;
    for (int i = 0; i < sp.head; i++) c.la[i] = layer(1 + i);
    hipError_t e = head_launch<HEAD, MID, TIN>(sp.head, c, cus, stream);
    for (int l = sp.head + 1, n = sp.pair ? 2 : sp.per; l <= total && e == hipSuccess; l += n, n = sp.per) {
        c.fin = in;
        c.fout = out;
        for (int i = 0; i < n; i++) c.la[i] = layer(l + i);
        e = l + n > total ? last_launch<MID, MODE, TIN, TOUT>(n, c, cus, stream) : map_launch<MID>(n, c, cus, stream);
        std::swap(in, out);
    }
    return e;
}

template <typename TIN, typename TOUT>
static hipError_t acnet8_pass_t(int blocks, const void* src, long ss, int W, int H, void* dst, long ds,
                                const float* wts, const float* wa, float4* f0, float4* f1, long fp, int cus, hipStream_t stream)
{
    Rows8 c = rows8_args(nullptr, nullptr, fp, W, H, {});
    c.src = src;
    c.ss = ss;
    c.w0 = wts;
    return rows8_pass<kRowsAcnet8, kPrelu, kShuffleSrc, TIN, TOUT>(c, blocks + 1, [&](int l) {
        LayerArgs la{};
        la.wa = wa + static_cast<long>(l - 1) * kRows8Floats;
        if (l <= blocks) {
            la.bias = wts + kA8OffLayer + (l - 1) * 16;   // 8 biases, then 8 slopes
            la.alpha = la.bias + 8;
        } else {
            la.bias = wts + kA8OffFinalB;
            la.src = src;
            la.ss = ss;
            la.dst = dst;
            la.ds = ds;
        }
        return la;
    }, f0, f1, cus, stream);
}

// ACNetLegacy's layer l
static LayerArgs legacy_layer(int l, const float* wts, const float* wa4, void* dst, long ds)
{
    LayerArgs la{};
    la.wa = wa4 + kRows8L0Floats + static_cast<long>(l - 1) * kRows8Floats;
    la.bias = wts + offB(l);
    if (l == 8) {
        la.k2 = wts + kOffK2;
        la.dst = dst;
        la.ds = ds;
    }
    return la;
}

template <typename TIN, typename TOUT>
static hipError_t legacy_split_t(const void* src, long ss, int W, int H, void* dst, long ds, const float* wts,
                                 const float* wa4, float4* f0, float4* f1, long fp, int cus, hipStream_t stream)
{
    Rows8 c = rows8_args(nullptr, nullptr, fp, W, H, {});
    c.src = src;
    c.ss = ss;
    c.w0 = wa4;
    c.b0 = wts + kOffB0;
    return rows8_pass<kRowsLegacy, kRelu, kReluDeconv, TIN, TOUT>(c, 8,
        [&](int l) { return legacy_layer(l, wts, wa4, dst, ds); }, f0, f1, cus, stream);
}

// ---- the layer-split form over a batch of images: every launch takes the strips of all of them,
// each image with its own two maps, all launches cut into the first one's columns: layer 0 with
// layers 1-2 and then two layers per launch, or layer 0 with layers 1-4 and then 5-8.
// 64 images of sides 128-2048 (30.7 Mpix): 3.04 ms, 4.06 before; three of 96 kpix in all 42 us, 58 ----

// What a launch of n strips of `rows` rows takes: a strip has two steps per layer after the first and
// about three to start, a step takes a fixed part and one for every layer and strip on the CU, and
// strips beyond one round of the CUs come in where others end, a third of a round late at the end.
// One round alone takes a fifth more: its strips are not spread evenly over the CUs, and a short
// image's strips hold their places for a whole strip's steps.
// Over 28 batches (u8) within 1.4% of the best of 12 heights and both numbers of layers on average, 8%
// at worst; without the fifth 3.6% and 33%: 48 of 300 x 200 in strips of 64 rows 430 us, 40 rows 322
// (62 x 16 tiles before: 453), 24 of 5.2 Mpix 4 / 256 790, 2 / 48 643 (before: 760).
static double batch_cost(double n, int rows, int layers, int per_cu, int cus)
{
    const double at = std::min<double>(per_cu, std::ceil(n / cus)), rounds = n / (at * cus);
    return (rows / 2 + 2 * (layers - 1) + 3) * (4.0 + at * layers) * (rounds <= 1.0 ? 1.2 : rounds + 0.3);
}

BatchSplit legacy_batch_split(const SplitDesc* desc, int n, int cus)
{
    BatchSplit best{ rows8_out<kRowsLegacy, 2>(), 32, 2 };
    double least = -1.0;
    for (int layers : { 2, 4 }) {
        const int cols = layers == 2 ? rows8_out<kRowsLegacy, 2>() : rows8_out<kRowsLegacy, 4>();
        const int per_cu = layers == 2 ? rows8_per_cu<kRowsMap, 2>() : rows8_per_cu<kRowsMap, 4>();
        for (int r : { 4, 6, 8, 10, 12, 16, 20, 24, 28, 32, 40, 48, 64, 80, 96, 128, 192, 256 }) {
            double strips = 0.0;
            for (int i = 0; i < n; i++)
                strips += static_cast<double>((desc[i].w + cols - 1) / cols) * ((desc[i].h + r - 1) / r);
            const double cost = 8 / layers * batch_cost(strips, r, layers, per_cu, cus);
            if (least < 0.0 || cost < least) {
                least = cost;
                best = { cols, r, layers };
            }
        }
    }
    return best;
}

template <int HEAD, int NL, int MODE, typename TIN, typename TOUT>
static void batch_launch(const SplitDesc* desc, int n, int total, const BatchSplit& sp, int first, const float* wts, const float* wa4,
                         hipStream_t stream)
{
    Rows8 c{};
    c.w0 = wa4;
    c.b0 = wts + kOffB0;
    c.rows = sp.rows;
    for (int i = 0; i < NL; i++) c.la[i] = legacy_layer(first + i, wts, wa4, nullptr, 0);
    // the first launch writes map 0 (it reads no map), then 0 -> 1 -> 0 -> the outputs
    constexpr int threads = rows8_threads<HEAD, NL>();
    hipLaunchKernelGGL((conv8_rows_batch<HEAD, NL, kRelu, MODE, TIN, TOUT>), strip_row(total, threads), dim3(threads), 0, stream, desc, n, total, sp.cols, ((first - 1) / NL & 1) == 0, c);
}

template <typename TIN, typename TOUT>
static hipError_t legacy_split_batch_t(const SplitDesc* desc, int n, int total, const BatchSplit& sp, const float* wts, const float* wa4,
                                       hipStream_t stream)
{
    if (sp.layers == 4) {
        batch_launch<kRowsLegacy, 4, kRelu, TIN, float>(desc, n, total, sp, 1, wts, wa4, stream);
        batch_launch<kRowsMap, 4, kReluDeconv, float, TOUT>(desc, n, total, sp, 5, wts, wa4, stream);
    } else {
        batch_launch<kRowsLegacy, 2, kRelu, TIN, float>(desc, n, total, sp, 1, wts, wa4, stream);
        batch_launch<kRowsMap, 2, kRelu, float, float>(desc, n, total, sp, 3, wts, wa4, stream);
        batch_launch<kRowsMap, 2, kRelu, float, float>(desc, n, total, sp, 5, wts, wa4, stream);
        batch_launch<kRowsMap, 2, kReluDeconv, float, TOUT>(desc, n, total, sp, 7, wts, wa4, stream);
    }
    return hipGetLastError();
}

#define ACHIP_TYPES(CALL)                                                                   \
    switch (stype) {                                                                        \
    case U8: switch (dtype) {                                                               \
        case U8: return CALL(uint8_t, uint8_t); case U16: return CALL(uint8_t, uint16_t);   \
        case F16: return CALL(uint8_t, __half); case F32: return CALL(uint8_t, float);      \
        default: return hipErrorInvalidValue; }                                             \
    case U16: switch (dtype) {                                                              \
        case U8: return CALL(uint16_t, uint8_t); case U16: return CALL(uint16_t, uint16_t); \
        case F16: return CALL(uint16_t, __half); case F32: return CALL(uint16_t, float);    \
        default: return hipErrorInvalidValue; }                                             \
    case F16: switch (dtype) {                                                              \
        case U8: return CALL(__half, uint8_t); case U16: return CALL(__half, uint16_t);     \
        case F16: return CALL(__half, __half); case F32: return CALL(__half, float);        \
        default: return hipErrorInvalidValue; }                                             \
    case F32: switch (dtype) {                                                              \
        case U8: return CALL(float, uint8_t); case U16: return CALL(float, uint16_t);       \
        case F16: return CALL(float, __half); case F32: return CALL(float, float);          \
        default: return hipErrorInvalidValue; }                                             \
    default: return hipErrorInvalidValue;                                                   \
    }

hipError_t launch_legacy_split(int stype, int dtype, const void* src, long ss, int W, int H, void* dst, long ds,
                               const float* wts, const float* wa4, void* workspace, int cus, hipStream_t stream)
{
    const long fp = acnet8_feature_pitch(W);
    float4* f0 = static_cast<float4*>(workspace);
    float4* f1 = reinterpret_cast<float4*>(static_cast<char*>(workspace) + fp * H);
#define CALL(TI, TO) legacy_split_t<TI, TO>(src, ss, W, H, dst, ds, wts, wa4, f0, f1, fp, cus, stream)
    ACHIP_TYPES(CALL)
#undef CALL
}

hipError_t launch_legacy_split_batch(int stype, int dtype, const SplitDesc* desc, int n, int total, const BatchSplit& sp,
                                     const float* wts, const float* wa4, hipStream_t stream)
{
    if (n <= 0 || total <= 0) return hipSuccess;
#define CALL(TI, TO) legacy_split_batch_t<TI, TO>(desc, n, total, sp, wts, wa4, stream)
    ACHIP_TYPES(CALL)
#undef CALL
}

hipError_t launch_acnet8(int blocks, int stype, int dtype, const void* src, long ss, int W, int H, void* dst, long ds,
                         const float* wts, const float* wa, void* workspace, int cus, hipStream_t stream)
{
    const long fp = acnet8_feature_pitch(W);
    float4* f0 = static_cast<float4*>(workspace);
    float4* f1 = reinterpret_cast<float4*>(static_cast<char*>(workspace) + fp * H);
#define CALL(TI, TO) acnet8_pass_t<TI, TO>(blocks, src, ss, W, H, dst, ds, wts, wa, f0, f1, fp, cus, stream)
    ACHIP_TYPES(CALL)
#undef CALL
}
#undef ACHIP_TYPES

} // namespace achip
