// ACNet<8> 2x pass (core/src/processor/cpu/CPUProcessor.cpp:1417-1436) with the conv3x3 layers
// as an FP16 or BF16 implicit GEMM on gfx950 MFMA (v_mfma_f32_16x16x32_{f16,bf16}), FP32
// accumulation, streamed: one wave per block, see stream16.hpp.
//   L0     conv3x3 1 -> 8 + PReLU in FP32 (the FP32 path's arithmetic), rounded to 16 bits
//   L1..LB conv3x3 8 -> 8, bias and PReLU in FP32, rounded to 16 bits
//   final  conv3x3 8 -> 4, pixel shuffle 2x, + the source pixel, all in FP32 from the FP32
//          accumulators, then fromFloat to the output type
// Nets of up to 8 blocks are one launch.  Deeper ones are cut into launches of at most 9 blocks
// with an 8-channel 16-bit map in HBM (16 bytes per pixel) between them: a launch's last layer
// writes the map, the next one's loader streams it in as layer 0.  A strip of n layers after
// layer 0 has 80 - 2 n output columns.
//
// Bound by the vector units: PReLU and packing are 14 instructions an item (80 a unit against its
// 15 MFMAs), L0's separately rounded products and sums 187 a wave; the busiest SIMD issues about
// 350 per step and workgroup.  1920 x 1080 u8 in FP16, 4 / 8 / 18 blocks: 52 / 74 / 144 us against
// 72 / 117 / 224 for the form it replaced (two blocks per launch, 16-bit maps in HBM between
// them, 43-52% of wave cycles waiting); 256 x 256: 12 / 18 / 37 against 23 / 36 / 69.
#pragma once

#include <algorithm>

#include "conv_layers.hpp"
#include "stream16.hpp"

namespace achip {

#pragma clang fp contract(off)

// At most 12 waves, three per SIMD: a workgroup's waves are dealt to the SIMDs from the first one
// on, so 14 (4, 4, 3, 3) left no room for a second workgroup.
constexpr int kS8MaxWaves = 12;
// Layers after layer 0, the last one included: with L0 (three waves; the last layer's wave is
// also the loader) 9, behind a map (one loader wave) 10, so at most 10 rings, two workgroups
// per CU.
constexpr int kS8L0Waves = 3, kS8MaxImg = 9, kS8MaxMap = 10;

// The last layer's wave takes whole segments of 16 pixels: five where a strip has more than 64 output
// columns, else four.  Lane j's patch in segment i starts at pixel n - 1 + j + 16 i, so with five the
// lanes past the strip's columns read up to pixel n + 80 of a row of 80 (and store nothing).
constexpr int s8_segments(int n) { return kSCols - 2 * n > 64 ? 5 : 4; }
constexpr int s8_last_pixel(int n) { return n - 1 + 15 + 16 * (s8_segments(n) - 1) + 2; }
// LDS of a launch of n layers: a pixel, the rings, then a pixel and the source rows (image head), or
// the pixels that the last segment reads past the last ring's last row.
constexpr unsigned s8_lds_bytes(bool img, int n)
{
    return 16 + n * kSRingBytes +
           (img ? 16 + kSImgBytes : 16u * static_cast<unsigned>(s8_last_pixel(n) >= kSCols ? s8_last_pixel(n) + 1 - kSCols : 1));
}
static_assert(16 * (s8_last_pixel(7) + 1 - kSCols) <= 16 + static_cast<int>(kSImgBytes), "with an image head that is the source rows");

enum S8Role : unsigned char { kS8L0 = 1, kS8Last = 4, kS8Layer = 8 };   // kS8L0 + part, kS8Layer + layer

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

struct Chunk8 {
    const void* src;        // source image (L0; the final layer adds it)
    void* dst;              // output image (final layer)
    const float* wts;       // ACNet<8> blob
    const uint4* wa;        // A operands of every layer, 3 x 64 each
    const uint4* fin;       // 16-bit map in (no image head)
    uint4* fout;            // 16-bit map out (no final layer)
    long ss, ds, fp;
    int W, H, rows;
    int tx0;                // first strip of the launch
    int l0;                 // block of this launch's layer 1
    int n;                  // layers after layer 0
    unsigned long long roles[2];   // S8Role of every wave, a byte each
};

// PReLU as prelu() rounds it, for a value about to be rounded to 16 bits, in three instructions:
// one of the two terms is zero, so fma(a, min(v, 0), max(v, 0)) rounds once, and a NaN gives 0 in
// both.  The upper bound of the median is the largest finite value, which rounds to infinity in
// either 16-bit type (with infinity itself the compiler makes it a max of a quieted v: two
// instructions).  min reads v only after the median has (the extra operand), so the compiler's
// wait for an MFMA's result covers it.
__device__ __forceinline__ float prelu3(float v, float a)
{
    const float m = __builtin_amdgcn_fmed3f(v, 0.f, 3.402823466e+38f);
    float t;
    asm("v_min_f32 %0, 0, %1" : "=v"(t) : "v"(v), "v"(m));
    return fmaf(a, t, m);
}

// A block's A operands, bias and slopes (this lane's 4 channels)
template <typename T16>
struct Block8 {
    typename Mma<T16>::v8 a[3];
    f32x4 bias;
    float alpha[4];
    __device__ __forceinline__ Block8(int block, const float* __restrict__ wts, const uint4* __restrict__ wa, int lane)
    {
#pragma unroll
        for (int t = 0; t < 3; t++) a[t] = __builtin_bit_cast(typename Mma<T16>::v8, wa[((block - 1) * 3 + t) * 64 + lane]);
        const float* bl = wts + kA8OffLayer + (block - 1) * 16 + 4 * ((lane >> 4) & 1);   // 8 biases, then 8 slopes
        bias = (f32x4){ bl[0], bl[1], bl[2], bl[3] };
#pragma unroll
        for (int r = 0; r < 4; r++) alpha[r] = bl[8 + r];
    }
    __device__ __forceinline__ uint2 finish(const f32x4& v) const
    {
        return make_uint2(pack16<T16>(prelu3(v[0], alpha[0]), prelu3(v[1], alpha[1])),
                          pack16<T16>(prelu3(v[2], alpha[2]), prelu3(v[3], alpha[3])));
    }
};

// L0, one pixel of the row pair per lane (pixels 64 part .. of 160), each product and sum rounded
// in the reference's order (Backend.hpp:58-75).  The weights are uniform: 72 scalar registers,
// an operand of each product.
template <typename T16, bool EDGE>
struct S8First {
    float w[9][8], bias[8], alpha[8];
    int c, gx, W;
    bool mine;
    ImgRow r0, r1, r2;
    RingRow out;
    // from pair p on (p >= -3)
    __device__ __forceinline__ S8First(int part, int W_, int xs, int p, const float* __restrict__ wts, int lane)
        : W(W_), r0(0), r1(0), r2(0), out(0)
    {
        const int t = min(64 * part + lane, 2 * kSCols - 1), ro = t >= kSCols ? 1 : 0;
        mine = 64 * part + lane < 2 * kSCols;
        c = t - ro * kSCols;
        gx = xs + c;
#pragma unroll
        for (int n = 0; n < 8; n++) {
#pragma unroll
            for (int k = 0; k < 9; k++)
                w[k][n] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(wts[kA8OffW0 + k * 8 + n])));
            bias[n] = wts[kA8OffB0 + n];
            alpha[n] = wts[kA8OffAlpha0 + n];
            asm volatile("" : "+v"(bias[n]), "+v"(alpha[n]));   // in vector registers: the scalar ones are full
        }
        const int row = 2 * p + ro + kSRows;
        r0 = ImgRow(row);
        r1 = ImgRow(row + 1);
        r2 = ImgRow(row + 2);
        out = RingRow(row);
    }
    __device__ __forceinline__ void step(const char* img, char* ring)
    {
        float q[9];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            q[d] = reinterpret_cast<const float*>(img + r0.off)[c + d];
            q[3 + d] = reinterpret_cast<const float*>(img + r1.off)[c + d];
            q[6 + d] = reinterpret_cast<const float*>(img + r2.off)[c + d];
        }
        float o[8];
#pragma unroll
        for (int n = 0; n < 8; n++) {
            float v = __fmul_rn(q[0], w[0][n]);
#pragma unroll
            for (int k = 1; k < 9; k++) v = __fadd_rn(v, __fmul_rn(q[k], w[k][n]));
            v = __fadd_rn(v, bias[n]);
            o[n] = fmaf(alpha[n], fminf(v, 0.0f), fmaxf(v, 0.0f));   // prelu(), see prelu3
        }
        const uint4 px = make_uint4(pack16<T16>(o[0], o[1]), pack16<T16>(o[2], o[3]), pack16<T16>(o[4], o[5]), pack16<T16>(o[6], o[7]));
        uint4* at = reinterpret_cast<uint4*>(ring + out.off) + c;
        if constexpr (!EDGE) {
            if (mine) *at = px;
        } else if (mine && gx >= 0 && gx < W) {
            *at = px;
            if (gx == 0 && c > 0) at[-1] = px;
            if (gx == W - 1 && c < kSCols - 1) at[1] = px;
        }
        r0.next_pair();
        r1.next_pair();
        r2.next_pair();
        out.next_pair();
    }
};

template <typename T16, bool EDGE>
__device__ __forceinline__ void s8_first(int part, int W, int xs, const StripRows& sr, int nsteps, const float* __restrict__ wts,
                                         const char* img, char* ring, int lane)
{
    const int first = sr.first(0), end = sr.end(0);
    S8First<T16, EDGE> f(part, W, xs, first, wts, lane);
    int s = 0;
    for (const int sb = sr.step(0, first); s < sb; s++) step_barrier();
    for (int p = first; p < end; p++, s++) {
        f.step(img, ring);
        step_barrier();
    }
    for (; s < nsteps; s++) step_barrier();
}

// The launch's last layer, N segments of 16 contiguous pixels: the next launch's map, or the
// final layer with the pixel shuffle and the source pixel.  step() takes its pairs in turn.
template <typename T16, typename TIN, typename TOUT, bool FINAL, int N, int G>
struct S8Last {
    using M = Mma<T16>;
    using v8 = typename M::v8;
    const Chunk8& c;
    const StripRows& sr;
    const char* in;
    Block8<T16> op;
    RingRow ir;
    int l, p, y, x0, nx, half, g, lane_rd;
    // final layer: the output pairs (columns 2 x, 2 x + 1 of row 2 y + half), and the source
    // pixels they add, loaded at the end of the step before (the loader read them long ago: L2)
    TOUT* o = nullptr;
    bool paired = false;
    TIN cur[N] = {};

    __device__ __forceinline__ void fetch(TIN (&t)[N], int yy) const
    {
        const TIN* r = row_ptr<TIN>(c.src, c.ss, min(yy, c.H - 1));
#pragma unroll
        for (int i = 0; i < N; i++) t[i] = r[clampi(x0 + 16 * i, 0, c.W - 1)];
    }
    __device__ __forceinline__ S8Last(const Chunk8& c_, int xs, const StripRows& sr_, const char* in_, int lane)
        : c(c_), sr(sr_), in(in_), op(FINAL ? 1 : c_.l0 + c_.n - 1, c_.wts, c_.wa, lane), ir(0)
    {
        l = c.n;
        p = sr.first(l);
        const int j = lane & 15, ro = lane >> 5;
        g = lane >> 4;
        half = g & 1;
        if constexpr (FINAL) {   // four output channels, all in the half = 0 lanes
#pragma unroll
            for (int t = 0; t < 3; t++) op.a[t] = __builtin_bit_cast(v8, c.wa[((c.l0 + l - 2) * 3 + t) * 64 + lane]);
            const float* b = c.wts + kA8OffFinalB;
            op.bias = half ? (f32x4){ 0.f, 0.f, 0.f, 0.f } : (f32x4){ b[0], b[1], b[2], b[3] };
        }
        x0 = xs + l + j;
        lane_rd = (l + j - 1) * 16;
        nx = min(kSCols - 2 * l - j, c.W - x0);   // segment i is inside if 16 i < nx
        y = sr.y0 + 2 * p + ro;
        if constexpr (FINAL) {
            o = row_ptr<TOUT>(c.dst, c.ds, 2 * y + half) + 2 * x0;
            paired = ((reinterpret_cast<uintptr_t>(c.dst) | static_cast<uintptr_t>(c.ds)) & (2 * sizeof(TOUT) - 1)) == 0;
            fetch(cur, y);
        }
        ir = RingRow(2 * p + g);
    }
    __device__ __forceinline__ void step()
    {
        unsigned rd = ir.off;
        if (sr.clamped(l, p)) rd = sr.clamped_off(l, p, g);
        const uint4* r = reinterpret_cast<const uint4*>(in + static_cast<int>(rd) + lane_rd);
        const bool row_in = y < sr.y1;
#pragma unroll
        for (int i0 = 0; i0 < N; i0 += G) {   // G segments at a time: registers
            v8 q[G][3];
            f32x4 acc[G];
#pragma unroll
            for (int i = 0; i < G && i0 + i < N; i++)
#pragma unroll
                for (int t = 0; t < 3; t++) q[i][t] = __builtin_bit_cast(v8, r[16 * (i0 + i) + t]);
#pragma unroll
            for (int i = 0; i < G && i0 + i < N; i++) acc[i] = M::mma(op.a[0], q[i][0], op.bias);
#pragma unroll
            for (int i = 0; i < G && i0 + i < N; i++) acc[i] = M::mma(op.a[1], q[i][1], acc[i]);
#pragma unroll
            for (int i = 0; i < G && i0 + i < N; i++) acc[i] = M::mma(op.a[2], q[i][2], acc[i]);
#pragma unroll
            for (int i = 0; i < G && i0 + i < N; i++) {
                const int k = i0 + i;
                if constexpr (FINAL) {
                    // half = 0 lanes hold the four sub-pixels n = 0..3 (output (2x + n % 2, 2y + n / 2));
                    // half = 1 lanes take row 2y + 1 from them
                    const float res = to_float<TIN>(cur[k]);
                    const float a = add_skip(other_half(acc[i][0], acc[i][2]), res);
                    const float b = add_skip(other_half(acc[i][1], acc[i][3]), res);
                    if (row_in && 16 * k < nx) store_pair_as(o + 32 * k, a, b, paired);
                } else if (row_in && 16 * k < nx) {
                    uint2* px = reinterpret_cast<uint2*>(reinterpret_cast<char*>(c.fout) + static_cast<long>(y) * c.fp) + 2 * (x0 + 16 * k) + half;
                    *px = op.finish(acc[i]);
                }
            }
        }
        y += 2;
        p++;
        if constexpr (FINAL) {
            o = reinterpret_cast<TOUT*>(reinterpret_cast<char*>(o) + 4 * c.ds);
            fetch(cur, y);
        }
        ir.next_pair();
    }
};

// The last layer's wave; with an image head it is also the loader, which then runs to the
// strip's end (past its last row it stores rows that no layer reads; the ring takes them).
template <typename T16, typename TIN, typename TOUT, bool IMG, bool FINAL, int N>
__device__ __forceinline__ void s8_last(const Chunk8& c, int xs, const StripRows& sr, int nsteps, char* img, char* ring0, int lane)
{
    S8Last<T16, TIN, TOUT, FINAL, N, IMG ? 1 : 2> last(c, xs, sr, ring0 + (c.n - 1) * kSRingBytes, lane);
    const int first = sr.first(0), sb = sr.step(c.n, last.p);
    int s = 0;
    if constexpr (IMG) {
        ImgRow out(2 * first);
        strip_loader<TIN, kSImgCols, 3>(
            c.src, c.ss, c.W, c.H, xs - 1, sr.base(0) - 1, first, first + nsteps, nsteps, lane,
            [&](int r, int col, TIN v) { reinterpret_cast<float*>(img + out.off + r * kSImgRowBytes)[col] = to_float<TIN>(v); },
            [&]() {
                out.next_pair();
                if (s++ >= sb) last.step();
            });
    } else {
        for (; s < sb; s++) step_barrier();
        for (; s < nsteps; s++) {
            last.step();
            step_barrier();
        }
    }
}

// IMG: layer 0 is L0 on the source image, else the map in; FINAL: the last layer is the net's
// final one, else it writes the map out.  Six waves per SIMD with two workgroups per CU: 80 VGPRs.
template <typename T16, typename TIN, typename TOUT, bool IMG, bool FINAL>
__global__ __launch_bounds__(64 * kS8MaxWaves, 6) void acnet8_stream16(const Chunk8 c)
{
    extern __shared__ uint4 s8_lds[];
    char* const ring0 = reinterpret_cast<char*>(s8_lds) + 16;   // s8_lds_bytes
    char* const img = reinterpret_cast<char*>(s8_lds) + c.n * kSRingBytes + 32;
    const int t = xcd_tile(strip_block(), gridDim.x * gridDim.y);
    const int ty = t / gridDim.x, tx = c.tx0 + t - ty * gridDim.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const StripRows sr(ty * c.rows, min((ty + 1) * c.rows, c.H), c.H, c.n, IMG ? 1 : 0);
    const int nsteps = sr.steps(), xs = tx * (kSCols - 2 * c.n) - c.n;
    const bool edge = xs < 0 || xs + kSCols > c.W;
    // The waves of a SIMD at different priorities, as the ACNetLegacy kernel's, where there is no
    // L0 (18 blocks at 1080p 146 -> 144 us); with its vector work every wave waits for the same
    // units and the priorities cost (8 blocks at 4K 257 against 235 us).
    if (!IMG && wave >= 8) __builtin_amdgcn_s_setprio(2);
    else if (!IMG && wave >= 4) __builtin_amdgcn_s_setprio(1);
    const int role = static_cast<int>((wave < 8 ? c.roles[0] : c.roles[1]) >> (8 * (wave & 7))) & 255;
    if (role >= kS8Layer) {
        const int l = role - kS8Layer;
        const Block8<T16> op(c.l0 + l - 1, c.wts, c.wa, lane);
        const char* in = ring0 + (l - 1) * kSRingBytes;
        char* out = ring0 + l * kSRingBytes;
        if (edge) strip_layer<Mma<T16>, Block8<T16>, true>(op, l, c.W, xs, sr, nsteps, in, out, lane);
        else strip_layer<Mma<T16>, Block8<T16>, false>(op, l, c.W, xs, sr, nsteps, in, out, lane);
    } else if (role == kS8Last) {
        if (s8_segments(c.n) == 5) s8_last<T16, TIN, TOUT, IMG, FINAL, 5>(c, xs, sr, nsteps, img, ring0, lane);
        else s8_last<T16, TIN, TOUT, IMG, FINAL, 4>(c, xs, sr, nsteps, img, ring0, lane);
    } else {
        if constexpr (IMG) {
            if (edge) s8_first<T16, true>(role - kS8L0, c.W, xs, sr, nsteps, c.wts, img, ring0, lane);
            else s8_first<T16, false>(role - kS8L0, c.W, xs, sr, nsteps, c.wts, img, ring0, lane);
        } else {
            RingRow out(2 * sr.first(0));
            strip_loader<u32x4, kSCols, 4>(
                c.fin, c.fp, c.W, c.H, xs, sr.base(0), sr.first(0), sr.end(0), nsteps, lane,
                [&](int r, int col, u32x4 v) { reinterpret_cast<u32x4*>(ring0 + out.off + r * kSRowBytes)[col] = v; },
                [&]() { out.next_pair(); });
        }
    }
}

// ---- launch ----

// Deal the launch's waves to the SIMDs (wave w runs on SIMD w % 4) so that their vector work
// per step (in instructions, counted in the compiled steps) is even: heaviest first, each to
// the least loaded SIMD with a wave left.  Returns the number of waves.
inline int s8_roles(bool img, bool fin, int n, unsigned long long (&roles)[2])
{
    struct W { unsigned char role; int cost; } w[kS8MaxWaves];
    int k = 0;
    if (img)
        for (int i = 0; i < kS8L0Waves; i++) w[k++] = { static_cast<unsigned char>(kS8L0 + i), 185 };
    else
        w[k++] = { kS8L0, 15 };   // the map's loader
    for (int l = 1; l < n; l++) w[k++] = { static_cast<unsigned char>(kS8Layer + l), 80 };
    w[k++] = { kS8Last, (img ? 20 : 5) + (kSCols - 2 * n + 15) / 16 * (fin ? 25 : 20) };
    for (int i = 1; i < k; i++)   // few entries: insertion sort, heaviest first
        for (int m = i; m > 0 && w[m].cost > w[m - 1].cost; m--) {
            const W t = w[m];
            w[m] = w[m - 1];
            w[m - 1] = t;
        }
    int load[4] = { 0, 0, 0, 0 }, have[4] = { 0, 0, 0, 0 };
    roles[0] = roles[1] = 0;
    for (int i = 0; i < k; i++) {
        int best = -1;
        for (int q = 0; q < 4; q++)
            if (have[q] < (k + 3 - q) / 4 && (best < 0 || load[q] < load[best])) best = q;
        const int wave = 4 * have[best] + best;
        roles[wave >> 3] |= static_cast<unsigned long long>(w[i].role) << (8 * (wave & 7));
        have[best]++;
        load[best] += w[i].cost;
    }
    return k;
}

template <typename T16, typename TIN, typename TOUT, bool IMG, bool FINAL>
hipError_t s8_launch(Chunk8 c, int cus, hipStream_t stream)
{
    const int waves = s8_roles(IMG, FINAL, c.n, c.roles);
    if (waves > kS8MaxWaves) return hipErrorInvalidValue;
    const int out_cols = kSCols - 2 * c.n, strips = (c.W + out_cols - 1) / out_cols, most = most_strips(64 * waves);
    const unsigned lds = s8_lds_bytes(IMG, c.n);
    // workgroups per CU: 160 KB of LDS and six waves per SIMD
    const int per_cu = std::min(static_cast<int>(160 * 1024 / lds), 6 / ((waves + 3) / 4));
    c.rows = strip_rows(strips, c.H, c.n, cus, per_cu);
    hipError_t e = hipSuccess;
    for (c.tx0 = 0; c.tx0 < strips && e == hipSuccess; c.tx0 += most) {   // one launch but for very wide images
        hipLaunchKernelGGL((acnet8_stream16<T16, TIN, TOUT, IMG, FINAL>), dim3(std::min(strips - c.tx0, most), (c.H + c.rows - 1) / c.rows),
                           dim3(64 * waves), lds, stream, c);
        e = hipGetLastError();
    }
    return e;
}

template <typename T16, typename TIN, typename TOUT>
hipError_t s8_pass(int blocks, const void* src, long ss, int W, int H, void* dst, long ds, const float* wts,
                   const uint4* wa, void* workspace, int cus, hipStream_t stream)
{
    Chunk8 c{};
    c.src = src;
    c.dst = dst;
    c.ss = ss;
    c.ds = ds;
    c.wts = wts;
    c.wa = wa;
    c.W = W;
    c.H = H;
    c.fp = acnet8_map16_pitch(W);
    // one launch with the final layer as its last, or blocks in launches of equal depth
    const int launches = blocks + 1 <= kS8MaxImg ? 1 : std::max(2, (blocks + kS8MaxImg - 1) / kS8MaxImg);
    static_assert(kS8MaxMap == kS8MaxImg + 1, "a last launch holds as many blocks as a first one, and the final layer");
    char* map = static_cast<char*>(workspace);
    int done = 0;
    for (int k = 0; k < launches; k++) {
        const int take = (blocks - done + launches - k - 1) / (launches - k);
        const bool first = k == 0, last = k == launches - 1;
        c.l0 = done + 1;
        c.n = take + (last ? 1 : 0);
        c.fin = reinterpret_cast<const uint4*>(map + ((k + 1) & 1) * c.fp * H);
        c.fout = reinterpret_cast<uint4*>(map + (k & 1) * c.fp * H);
        const hipError_t e = first ? (last ? s8_launch<T16, TIN, TOUT, true, true>(c, cus, stream)
                                           : s8_launch<T16, TIN, float, true, false>(c, cus, stream))
                                   : (last ? s8_launch<T16, TIN, TOUT, false, true>(c, cus, stream)
                                           : s8_launch<T16, float, float, false, false>(c, cus, stream));
        if (e != hipSuccess) return e;
        done += take;
    }
    return hipSuccess;
}

template <typename T16>
hipError_t launch_acnet8_16_types(int blocks, int stype, int dtype, const void* src, long ss, int W, int H, void* dst,
                                  long ds, const float* wts, const uint4* wa, void* workspace, int cus, hipStream_t stream)
{
#define CALL(TI, TO) s8_pass<T16, TI, TO>(blocks, src, ss, W, H, dst, ds, wts, wa, workspace, cus, stream)
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

} // namespace achip
