// The streamed form of the 16-bit MFMA passes: one wave per layer, rows flowing through all
// layers in one launch.
//
// A workgroup owns a strip: 80 columns of the image (the output columns plus a margin of one
// pixel per layer on each side) over a range of rows.  Every 8 -> 8 layer is a wave of its
// own that keeps its A operands and bias in registers for the whole strip; the waves advance
// in steps of one row pair over rings in LDS (stream.hpp).
//
// A step's work item is the tile kernels' unit (80 columns x 2 rows: item o of 5 holds the
// columns o + 5 j, so lane j's 7 pixel reads feed 15 MFMAs), and each output's arithmetic is
// theirs, so the bits are.
//
// Columns: all layers compute all 80; layer l's outputs are good in [l, 80 - l) and the
// strip's last layer is good over the output columns.  The columns outside read the
// neighbouring row's end (the pitch is exactly 80 pixels): an MFMA column depends on its own
// operand column only, so what they hold never reaches a good column.  Rows: layer l covers
// its rows [y0 - (L - l), y1 + (L - l)), an even number of them unless the image ends there,
// so every patch row it reads, those with zero weights included, is a computed one (a stale
// NaN times zero would be a NaN).  Image borders: rows are clamped when read; the columns next
// to the image's first and last are written along with them, which is the replicate padding
// of every layer (Common.hpp:120-143).
#pragma once

#include "mfma16.hpp"
#include "stream.hpp"

namespace achip {

constexpr int kSPh = 5;   // items of a unit
static_assert(kSCols == 16 * kSPh, "a unit is a whole row pair of a strip");

// Source rows as f32 in a ring of three pairs: image columns xs - 1 .. xs + 80 and rows
// base(0) - 1 .., converted once (layer 0's items read each pixel up to 12 times).
constexpr int kSImgCols = kSCols + 2;
constexpr unsigned kSImgRowBytes = (kSImgCols + 2) * 4;
constexpr unsigned kSImgBytes = kSRows * kSImgRowBytes;

struct ImgRow {
    unsigned off;
    __device__ __forceinline__ explicit ImgRow(int row) : off(static_cast<unsigned>(row) % kSRows * kSImgRowBytes) {}
    __device__ __forceinline__ void next_pair()
    {
        off += 2 * kSImgRowBytes;
        off = min(off, off - kSImgBytes);
    }
};

template <typename TIN>
__device__ __forceinline__ void image_loader(const void* __restrict__ src, long ss, int W, int H, int xs, const StripRows& sr,
                                             int nsteps, char* img, int lane)
{
    ImgRow out(2 * sr.first(0));
    strip_loader<TIN, kSImgCols, 6>(
        src, ss, W, H, xs - 1, sr.base(0) - 1, sr.first(0), sr.end(0) + 1, nsteps, lane,
        [&](int r, int c, TIN v) { reinterpret_cast<float*>(img + out.off + r * kSImgRowBytes)[c] = to_float<TIN>(v); },
        [&]() { out.next_pair(); });
}

// Write items O0 .. O0 + N - 1 of a unit (res[o]: 4 channels of column O0 + o + 5 j, image
// column x + o, row ro of the pair) at `w` (this lane's first).  In a strip that reaches past
// the image, columns outside it are not written and its first and last columns are copied one
// outward.
template <bool EDGE, int O0, int N>
__device__ __forceinline__ void write_unit(uint2* w, const uint2 (&res)[N], int x, int j, int W)
{
#pragma unroll
    for (int o = 0; o < N; o++) {
        if constexpr (!EDGE) {
            w[2 * o] = res[o];
        } else {
            const int gx = x + o, c = O0 + o + kSPh * j;
            if (gx >= 0 && gx < W) {
                w[2 * o] = res[o];
                if (gx == 0 && c > 0) w[2 * o - 2] = res[o];
                if (gx == W - 1 && c < kSCols - 1) w[2 * o + 2] = res[o];
            }
        }
    }
}

// A wave's middle layer l: ring `in` -> ring `out`, one unit per step.  op: the layer's A
// operands, bias and activation (Op::v8 a[3], f32x4 bias, uint2 finish(f32x4)).  Every MFMA
// and store of an interior strip's step is unconditional: 15 MFMAs, 10 LDS accesses and, with
// ReLU, 29 VALU instructions.
template <class M, class Op, bool EDGE>
__device__ __forceinline__ void strip_layer(const Op& op, int l, int W, int xs, const StripRows& sr, int nsteps,
                                            const char* in, char* out, int lane)
{
    using v8 = typename M::v8;
    const int j = lane & 15, g = lane >> 4, half = g & 1, ro = g >> 1;
    const int first = sr.first(l), end = sr.end(l);
    const int lane_rd = (kSPh * j - 1) * 16, lane_wr = kSPh * j * 16 + half * 8;
    RingRow ir(2 * first + g), orow(2 * first + ro);
    int s = 0;
    for (const int sb = sr.step(l, first); s < sb; s++) step_barrier();
    for (int p = first; p < end; p++, s++) {
        unsigned rd = ir.off;
        if (sr.clamped(l, p)) rd = sr.clamped_off(l, p, g);
        const uint4* r = reinterpret_cast<const uint4*>(in + static_cast<int>(rd) + lane_rd);
        v8 q[kSPh + 2];
#pragma unroll
        for (int d = 0; d < kSPh + 2; d++) q[d] = __builtin_bit_cast(v8, r[d]);
        f32x4 acc[kSPh];
#pragma unroll
        for (int o = 0; o < kSPh; o++) acc[o] = M::mma(op.a[0], q[o], op.bias);
#pragma unroll
        for (int o = 0; o < kSPh; o++) acc[o] = M::mma(op.a[1], q[o + 1], acc[o]);
#pragma unroll
        for (int o = 0; o < kSPh; o++) acc[o] = M::mma(op.a[2], q[o + 2], acc[o]);
        uint2 res[kSPh];
#pragma unroll
        for (int o = 0; o < kSPh; o++) res[o] = op.finish(acc[o]);
        write_unit<EDGE, 0, kSPh>(reinterpret_cast<uint2*>(out + orow.off + lane_wr), res, xs + kSPh * j, j, W);
        ir.next_pair();
        orow.next_pair();
        step_barrier();
    }
    for (; s < nsteps; s++) step_barrier();
}

// The two halves (lanes 16 apart) of a pixel: half = 0 lanes hold channels 0-3, half = 1 lanes
// 4-7.  other_half: a for half = 0 lanes, the partner's b for half = 1 lanes.  add_halves: the sum
// of both halves' a for half = 0 lanes, of both halves' b for half = 1 lanes.
__device__ __forceinline__ float other_half(float a, float b)
{
    return __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false)[0]);
}
__device__ __forceinline__ float add_halves(float a, float b)
{
    const auto e = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(e[0]) + __uint_as_float(e[1]);
}

// max(v, 0) of an accumulator as fmaxf gives it (0 for a NaN), in one instruction: fmaxf of a
// value the compiler cannot prove quiet costs two.
__device__ __forceinline__ float relu1(float v) { return __builtin_amdgcn_fmed3f(v, 0.f, __builtin_inff()); }

} // namespace achip
