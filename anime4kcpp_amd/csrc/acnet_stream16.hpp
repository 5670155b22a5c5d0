// ACNetLegacy 2x pass with the 8 -> 8 layers as an FP16 or BF16 implicit GEMM on gfx950 MFMA
// (v_mfma_f32_16x16x32_{f16,bf16}, FP32 accumulation), streamed: one wave per layer, see
// stream16.hpp.  Layer 0 (1 -> 8) is an FP32 MFMA (v_mfma_f32_16x16x4_f32) on the f32 source
// rows; bias, ReLU and the deconv are FP32.
//
// The GEMM of one item (16 pixels x 2 rows):
//   D[16 x 16] = A[16 x 96] * B[96 x 16]
//   rows i of D/A : i = 8*ro + n, output channel n of output row y + ro (ro = 0, 1);
//   columns j     : the item's 16 pixels;
//   K = 96        : a 4 x 3 input patch (rows y-1..y+2, columns x-1..x+1) x 8 channels.
// Both output rows are linear in the same 4 x 3 patch, so all 16 MFMA rows are useful;
// 72 of each row's 96 weights are nonzero.  K is split over three MFMAs, one per patch
// column t; inside one MFMA lane group g = lane/16 holds patch row g, so each lane's B
// operand is the 8 channels of one pixel: a single 16-byte LDS read.  The last layer uses
// contiguous 16-pixel items so that the deconv's stores are contiguous.
//
// D lands as lane l holding rows 4*(l/16)..+3 of column l%16: 4 channels of one pixel.
// The bias is the accumulator's initial value; the sum is rounded to 16 bits (RNE) and
// ReLU'd on the packed bits (max with +0 as signed 16-bit integers, exact for both
// formats); after layer 8 the FP32 sums feed the deconv.
//
// Bound by the matrix pipes at the clock the card holds under them: at two workgroups per CU
// a step issues 576-672 cycles of MFMAs per SIMD and workgroup (FP32 layer 0 included) and
// takes about 900.  1920 x 1080 u8 in FP16: 45.5 us against 56.7 for the tile form it
// replaced (64 x 32 tiles, all layers of a tile one after the other between barriers, matrix
// pipes 31% busy); 3840 x 2160 149 against 199, 256 x 256 12.4 against 21.3.
#pragma once

#include <algorithm>

#include "stream16.hpp"

namespace achip {

#pragma clang fp contract(off)

// Waves of a workgroup: the last layer (two: two of its four 16-pixel segments each), layer 0
// (two: three and two of the unit's five items), layers 1, 3, 5, 7 and 2, 4, 6, the loader.
// In this order wave w runs on SIMD w % 4 beside waves w + 4 and w + 8, and the four SIMDs
// get 576, 576, 672 and 528 MFMA cycles per step.
constexpr int kSLWaves = 12, kSLThreads = 64 * kSLWaves;
constexpr int kSLLayers = 8;                                 // after layer 0
constexpr int kSLMargin = kSLLayers, kSLOut = kSCols - 2 * kSLMargin;   // 64 output columns
// the rings of layers 0..7 with a pixel before and after, then the source rows: 63.5 KB, two
// workgroups per CU for every source type
constexpr unsigned kSLLds = kSLLayers * kSRingBytes + 32 + kSImgBytes;

// Items O0 .. O0 + N - 1 of layer 0: 3 FP32 MFMAs each on the loader's f32 rows.
template <typename T16, int O0, int N, bool EDGE>
__device__ __forceinline__ void legacy_first(int W, int xs, const StripRows& sr, int nsteps, const float* __restrict__ wts,
                                             const float* __restrict__ wa0, const char* img, char* ring, int lane)
{
    const int j = lane & 15, g = lane >> 4, half = g & 1, ro = g >> 1;
    const float a0 = wa0[lane], a1 = wa0[64 + lane], a2 = wa0[128 + lane];
    const float* bl = wts + kOffB0 + 4 * half;
    const f32x4 bias = { bl[0], bl[1], bl[2], bl[3] };
    const int first = sr.first(0), end = sr.end(0);
    ImgRow ir(2 * first + g);
    RingRow out(2 * first + ro);
    const int lane_rd = (kSPh * j + O0) * 4;   // img column c is plane column c - 1
    int s = 0;
    for (const int sb = sr.step(0, first); s < sb; s++) step_barrier();
    for (int p = first; p < end; p++, s++) {
        const float* r = reinterpret_cast<const float*>(img + ir.off + lane_rd);
        float q[N + 2];
#pragma unroll
        for (int d = 0; d < N + 2; d++) q[d] = r[d];
        f32x4 acc[N];
#pragma unroll
        for (int o = 0; o < N; o++) acc[o] = mma_f32(a0, q[o], bias);
#pragma unroll
        for (int o = 0; o < N; o++) acc[o] = mma_f32(a1, q[o + 1], acc[o]);
#pragma unroll
        for (int o = 0; o < N; o++) acc[o] = mma_f32(a2, q[o + 2], acc[o]);
        uint2 res[N];
#pragma unroll
        for (int o = 0; o < N; o++)
            res[o] = make_uint2(relu_pack<T16>(acc[o][0], acc[o][1]), relu_pack<T16>(acc[o][2], acc[o][3]));
        write_unit<EDGE, O0, N>(reinterpret_cast<uint2*>(ring + out.off) + (kSPh * j + O0) * 2 + half, res,
                                xs + kSPh * j + O0, j, W);
        ir.next_pair();
        out.next_pair();
        step_barrier();
    }
    for (; s < nsteps; s++) step_barrier();
}

// this lane's A operands and bias of layer l, and the ReLU + rounding of its sums
template <typename T16>
struct LegacyOp {
    typename Mma<T16>::v8 a[3];
    f32x4 bias;
    __device__ __forceinline__ LegacyOp(int l, const float* __restrict__ wts, const uint4* __restrict__ wa, int lane)
    {
#pragma unroll
        for (int t = 0; t < 3; t++) a[t] = __builtin_bit_cast(typename Mma<T16>::v8, wa[((l - 1) * 3 + t) * 64 + lane]);
        const float* bl = wts + offB(l) + 4 * ((lane >> 4) & 1);
        bias = (f32x4){ bl[0], bl[1], bl[2], bl[3] };
    }
    __device__ __forceinline__ uint2 finish(const f32x4& v) const
    {
        return make_uint2(relu_pack<T16>(v[0], v[1]), relu_pack<T16>(v[2], v[3]));
    }
};

// layer 8 and the deconv, 16-pixel segments S0, S0 + 1 of the strip's 64 output columns
template <typename T16, typename TOUT, int S0>
__device__ __forceinline__ void legacy_last(int W, int xs, const StripRows& sr, const float* __restrict__ wts,
                                            const uint4* __restrict__ wa, const char* in, void* __restrict__ dst, long ds,
                                            int lane)
{
    using M = Mma<T16>;
    using v8 = typename M::v8;
    constexpr int l = kSLLayers;
    const int j = lane & 15, g = lane >> 4, half = g & 1, ro = g >> 1;
    const LegacyOp<T16> op(l, wts, wa, lane);
    const float* k2 = wts + kOffK2 + 16 * half;
    float kd[4][4];
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int q = 0; q < 4; q++) kd[c][q] = k2[c * 4 + q];
    const int first = sr.first(l), end = sr.end(l);
    const int x0 = xs + kSLMargin + 16 * S0 + j, lane_rd = (kSLMargin + 16 * S0 + j - 1) * 16;
    // this lane's output pair of segment i: columns 2 (x0 + 16 i), + 1 of output row 2 y + half.
    // 2 x is even, so every pair is aligned for one store if the image is.
    TOUT* o = row_ptr<TOUT>(dst, ds, 2 * (sr.y0 + 2 * first + ro) + half) + 2 * x0;
    const bool paired = ((reinterpret_cast<uintptr_t>(dst) | static_cast<uintptr_t>(ds)) & (2 * sizeof(TOUT) - 1)) == 0;
    RingRow ir(2 * first + g);
    int s = 0;
    for (const int sb = sr.step(l, first); s < sb; s++) step_barrier();
    for (int p = first; p < end; p++) {
        unsigned rd = ir.off;
        if (sr.clamped(l, p)) rd = sr.clamped_off(l, p, g);
        const uint4* r = reinterpret_cast<const uint4*>(in + static_cast<int>(rd) + lane_rd);
        v8 q[2][3];
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 3; t++) q[i][t] = __builtin_bit_cast(v8, r[16 * i + t]);
        f32x4 acc[2];
#pragma unroll
        for (int i = 0; i < 2; i++) acc[i] = M::mma(op.a[0], q[i][0], op.bias);
#pragma unroll
        for (int i = 0; i < 2; i++) acc[i] = M::mma(op.a[1], q[i][1], acc[i]);
#pragma unroll
        for (int i = 0; i < 2; i++) acc[i] = M::mma(op.a[2], q[i][2], acc[i]);
        const bool row_in = sr.y0 + 2 * p + ro < sr.y1;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            float v[4], sum[4];
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = relu1(acc[i][c]);
#pragma unroll
            for (int k = 0; k < 4; k++)
                sum[k] = fmaf(v[3], kd[3][k], fmaf(v[2], kd[2][k], fmaf(v[1], kd[1][k], v[0] * kd[0][k])));
            // half = 0 lanes keep sub-pixels 0 and 1 (output row 2 y), half = 1 lanes 2 and 3
            const float s0 = add_halves(sum[0], sum[2]), s1 = add_halves(sum[1], sum[3]);
            if (row_in && x0 + 16 * i < W) store_pair_as(o + 32 * i, s0, s1, paired);
        }
        o = reinterpret_cast<TOUT*>(reinterpret_cast<char*>(o) + 4 * ds);
        ir.next_pair();
        step_barrier();
    }
}

// Output rows [y0, y1) of the strip whose output columns start at x0; lds: kSLLds bytes.  Ends
// with every wave past the last step's barrier.
template <typename T16, typename TIN, typename TOUT>
__device__ __forceinline__ void legacy_strip(const void* __restrict__ src, long ss, int W, int H, void* __restrict__ dst,
                                             long ds, const float* __restrict__ wts, const uint4* __restrict__ wa,
                                             const float* __restrict__ wa0, int x0, int y0, int y1, char* lds)
{
    // through an empty asm statement: nothing derived from the thread index is kept in
    // registers across a persistent kernel's strips
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const StripRows sr(y0, y1, H, kSLLayers, 1);
    const int nsteps = sr.steps(), xs = x0 - kSLMargin;
    const bool edge = xs < 0 || xs + kSCols > W;
    char* const ring0 = lds + 16;
    char* const img = lds + kSLLayers * kSRingBytes + 32;
    // The three waves of a SIMD at three priorities: one's MFMAs run beside another's packing
    // and LDS accesses instead of all three at once (1080p FP16 48.7 -> 45.5 us).
    if (wave >= 8) __builtin_amdgcn_s_setprio(2);
    else if (wave >= 4) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
    if (wave == 0) {
        legacy_last<T16, TOUT, 0>(W, xs, sr, wts, wa, ring0 + (kSLLayers - 1) * kSRingBytes, dst, ds, lane);
    } else if (wave == 1) {
        legacy_last<T16, TOUT, 2>(W, xs, sr, wts, wa, ring0 + (kSLLayers - 1) * kSRingBytes, dst, ds, lane);
    } else if (wave == 2) {
        if (edge) legacy_first<T16, 3, 2, true>(W, xs, sr, nsteps, wts, wa0, img, ring0, lane);
        else legacy_first<T16, 3, 2, false>(W, xs, sr, nsteps, wts, wa0, img, ring0, lane);
    } else if (wave == 3) {
        if (edge) legacy_first<T16, 0, 3, true>(W, xs, sr, nsteps, wts, wa0, img, ring0, lane);
        else legacy_first<T16, 0, 3, false>(W, xs, sr, nsteps, wts, wa0, img, ring0, lane);
    } else if (wave == kSLWaves - 1) {
        image_loader<TIN>(src, ss, W, H, xs, sr, nsteps, img, lane);
    } else {
        const int l = wave < 8 ? 2 * (wave - 4) + 1 : 2 * (wave - 8) + 2;
        const LegacyOp<T16> op(l, wts, wa, lane);
        const char* in = ring0 + (l - 1) * kSRingBytes;
        char* out = ring0 + l * kSRingBytes;
        if (edge) strip_layer<Mma<T16>, LegacyOp<T16>, true>(op, l, W, xs, sr, nsteps, in, out, lane);
        else strip_layer<Mma<T16>, LegacyOp<T16>, false>(op, l, W, xs, sr, nsteps, in, out, lane);
    }
}

// 12 waves, two workgroups per CU: 6 waves per SIMD, at most 80 VGPRs
template <typename T16, typename TIN, typename TOUT>
__global__ __launch_bounds__(kSLThreads, 6) void acnet_stream16(const void* __restrict__ src, long ss, int W, int H,
                                                                void* __restrict__ dst, long ds,
                                                                const float* __restrict__ wts, const uint4* __restrict__ wa,
                                                                const float* __restrict__ wa0, int rows, int tx0)
{
    __shared__ uint4 lds[kSLLds / 16];
    const int t = xcd_tile(strip_block(), gridDim.x * gridDim.y);
    const int ty = t / gridDim.x, tx = tx0 + t - ty * gridDim.x;
    legacy_strip<T16, TIN, TOUT>(src, ss, W, H, dst, ds, wts, wa, wa0, tx * kSLOut, ty * rows, min((ty + 1) * rows, H),
                                 reinterpret_cast<char*>(lds));
}

// Persistent batched form: resident workgroups (at most one per strip) take strips of `rows` rows, the
// first one by their own number and the rest from a queue.  Drawing the first ones too let the workgroups
// that started first take a second strip before the last ones had drawn any, which then found the queue
// empty (150 strips of 20 rows: 39.5 us against 23.8 now; three u8 images of 700 x 500 in FP16: 72 against 48).
template <typename T16, typename TIN, typename TOUT>
__global__ __launch_bounds__(kSLThreads, 6) void acnet_stream16_batch(const BatchDesc* __restrict__ desc, int n, int total,
                                                                      int* __restrict__ counter,
                                                                      const float* __restrict__ wts,
                                                                      const uint4* __restrict__ wa,
                                                                      const float* __restrict__ wa0, int rows)
{
    __shared__ uint4 lds[kSLLds / 16];
    __shared__ int s_tile;
    int t = blockIdx.x;
    while (t < total) {
        // The next strip is drawn as this one starts and read once it is done, so the atomic's
        // round trip overlaps the strip.  Each workgroup draws exactly one index past its last.
        int next = 0;
        if (threadIdx.x == 0) next = gridDim.x + atomicAdd(counter, 1);
        const BatchDesc d = find_tile(desc, n, t);
        const int local = t - d.first_tile;
        const int ly = local / d.tiles_x;
        const int tx = local - ly * d.tiles_x;
        const int y0 = (d.ty0 + ly) * rows;
        legacy_strip<T16, TIN, TOUT>(d.src, d.sstride, d.w, d.h, d.dst, d.dstride, wts, wa, wa0, tx * kSLOut, y0,
                                     min(y0 + rows, d.h), reinterpret_cast<char*>(lds));
        __syncthreads();                    // s_tile has been read by every wave
        if (threadIdx.x == 0) s_tile = next;
        __syncthreads();
        t = __builtin_amdgcn_readfirstlane(s_tile);
    }
}

// ---- launch ----

template <typename T16, typename TIN, typename TOUT>
static hipError_t launch_one(int cfg, const void* src, long ss, int W, int H, void* dst, long ds, const float* wts,
                             const uint4* wa, const float* wa0, int cus, hipStream_t stream)
{
    const int strips = (W + kSLOut - 1) / kSLOut;
    const int rows = cfg ? kStreamConfigs[cfg].th : strip_rows(strips, H, kSLLayers, cus, 2);
    hipError_t e = hipSuccess;
    for (int tx0 = 0; tx0 < strips && e == hipSuccess; tx0 += most_strips(kSLThreads)) {   // one launch but for very wide images
        hipLaunchKernelGGL((acnet_stream16<T16, TIN, TOUT>), dim3(std::min(strips - tx0, most_strips(kSLThreads)), (H + rows - 1) / rows),
                           dim3(kSLThreads), 0, stream, src, ss, W, H, dst, ds, wts, wa, wa0, rows, tx0);
        e = hipGetLastError();
    }
    return e;
}

template <typename T16, typename TIN, typename TOUT>
static hipError_t launch_batch_one(const BatchDesc* desc, int n, int total, int rows, int* counter, const float* wts,
                                   const uint4* wa, const float* wa0, int max_wg, hipStream_t stream)
{
    auto kern = acnet_stream16_batch<T16, TIN, TOUT>;
    const int grid = persistent_grid(reinterpret_cast<const void*>(kern), kSLThreads, total, max_wg);
    if (grid <= 0) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kSLThreads), 0, stream, desc, n, total, counter, wts, wa, wa0, rows);
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

template <typename T16>
hipError_t launch_stream16_types(int cfg, int stype, int dtype, const void* src, long ss, int W, int H, void* dst, long ds,
                               const float* wts, const uint4* wa, const float* wa0, int cus, hipStream_t stream)
{
#define CALL(TI, TO) launch_one<T16, TI, TO>(cfg, src, ss, W, H, dst, ds, wts, wa, wa0, cus, stream)
    ACHIP_TYPES(CALL)
#undef CALL
}

template <typename T16>
hipError_t launch_stream16_batch_types(int stype, int dtype, const BatchDesc* desc, int n, int total, int rows, int* counter,
                                     const float* wts, const uint4* wa, const float* wa0, int max_wg, hipStream_t stream)
{
#define CALL(TI, TO) launch_batch_one<T16, TI, TO>(desc, n, total, rows, counter, wts, wa, wa0, max_wg, stream)
    ACHIP_TYPES(CALL)
#undef CALL
}
#undef ACHIP_TYPES

} // namespace achip
