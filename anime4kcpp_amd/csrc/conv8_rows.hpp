// The FP32 8-channel conv3x3 layers (ACNetLegacy's layer-split form, ACNet<8>, FSRCNNX<8>) on
// v_mfma_f32_4x4x1_16b_f32, several layers per launch, streamed: row pairs of a strip move through
// the layers over rings of three pairs in LDS (stream.hpp), two waves per layer, one per row of
// the pair.
//
// The MFMA: 16 blocks of 4 x 4 with K = 1.  Lane l's column is pixel l of the row (64 columns of a
// strip), its D registers are four output channels of that pixel, B is one input channel of the
// tap's pixel as it comes from LDS, and A (four output channels' weights of one tap and input
// channel) is broadcast to all blocks from one of them, so a register holds 16 such operands and
// a layer's 144 take 9.  Every MFMA is 256 useful multiply-adds; the 16x16x4 form of the fused
// kernel spends a quarter of its own on zero weights (two output rows from a patch of four).
// Both instructions are chains of FMAs (16x16x4: over k = 0..3 in turn), and each output's FMAs
// run in the fused kernel's order -- two accumulators, even input channels from the bias and odd
// ones from zero, patch column, channel, patch row, then their sum -- so the bits are its.
//
// Bound by the matrix pipe: a row of a layer is 144 MFMAs of 8.1 cycles, and with four strips (16
// waves of a layer pair) on every CU the pipe is busy 83% of a step, the rest being the steps'
// barriers and the last strips' tails.  A strip's first steps fill the pipeline (two per layer), so
// heights follow the number of strips (rows8_rows).  Two map layers at 1920 x 1080: 69.1 us with
// 62 x 16 tiles and 16x16x4 MFMAs, 50.2 streamed in strips of 34 rows (28 rows 51.5, 46 52.9, 68
// 56.3, 136 69.3).  Whole passes, before / now: ACNetLegacy 288 / 213 us at 1080p, 50 / 28 at
// 256 x 256; ACNet<8> of 18 blocks 716 / 548 and 116 / 67; FSRCNNX<8> 215 / 164 and 38 / 25.
#pragma once

#include <initializer_list>
#include <type_traits>
#include <utility>

#include "acnet_mfma32_item.hpp"   // f32x4m
#include "conv_layers.hpp"
#include "stream.hpp"

namespace achip {

#pragma clang fp contract(off)

// What the first layer of a launch reads: a map, or layer 0 from the source image (two more waves)
// with ACNetLegacy's FMAs or ACNet<8>'s separately rounded products and sums.
enum RowsHead : int { kRowsMap = 0, kRowsLegacy = 1, kRowsAcnet8 = 2 };

constexpr int kR8Cols = 64;                       // columns of every layer
constexpr int kR8In = kR8Cols + 2;                // columns of the first one's input; pitch of every ring
constexpr unsigned kR8Row = kR8In * 16;           // bytes of a ring row in one plane (channels 0-3 or 4-7)
constexpr unsigned kR8Plane = kSRows * kR8Row, kR8Ring = 2 * kR8Plane;
constexpr unsigned kR8ImgRow = (kR8In + 2) * 4, kR8ImgBytes = kSRows * kR8ImgRow;

// Output columns of a strip of NL layers after its input or layer 0.
template <int HEAD, int NL>
constexpr int rows8_out() { return kR8Cols - 2 * (HEAD == kRowsMap ? NL - 1 : NL); }
template <int HEAD, int NL>
constexpr unsigned rows8_lds() { return NL * kR8Ring + (HEAD == kRowsMap ? 0 : kR8ImgBytes); }
template <int HEAD, int NL>
constexpr int rows8_threads() { return 128 * (NL + (HEAD == kRowsMap ? 0 : 1)); }

struct RowsIo {
    const float4* fin;      // map in (kRowsMap)
    float4* fout;           // map out
    long fp;                // their pitch
    const void* src;        // source image (the other heads)
    long ss;
    const float* w0;        // layer 0: ACNetLegacy A operands (18 x 4, two registers) or the ACNet<8> blob
    const float* b0;        // ACNetLegacy: its biases
    int W, H, rows;         // rows per strip, even
};

struct Rows8 : RowsIo {
    LayerArgs la[4];        // the layers; la[NL - 1] is the last
};

// acc += w[channel quad `h`][operand s] * b, s counted per output quad: [t][c][ky], the A operand
// of slot s * HALVES + h
template <int SLOT>
__device__ __forceinline__ f32x4m mma4(const float* w, float b, f32x4m c)
{
    return __builtin_amdgcn_mfma_f32_4x4x1f32(w[SLOT / 16], b, c, 4, SLOT % 16, 0);
}

__device__ __forceinline__ float quad(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// The MFMAs of patch column T: q[ky][0] channels 0-3, q[ky][1] channels 4-7 of the three patch rows.
// acc[h][parity]: output channels 4 h ..; consecutive MFMAs go to 2 * HALVES different chains.
template <int T, int HALVES, int... I>
__device__ __forceinline__ void column4(const float* w, const float4 (&q)[3][2], f32x4m (&acc)[HALVES][2], std::integer_sequence<int, I...>)
{
    // I = ((pair of channels * 3 + ky) * 2 + parity) * HALVES + h
    ((acc[I % HALVES][I / HALVES % 2] =
          mma4<((T * 8 + I / (6 * HALVES) * 2 + I / HALVES % 2) * 3 + I / (2 * HALVES) % 3) * HALVES + I % HALVES>(
              w, quad(q[I / (2 * HALVES) % 3][I / (12 * HALVES)], I / (6 * HALVES) % 2 * 2 + I / HALVES % 2),
              acc[I % HALVES][I / HALVES % 2])),
     ...);
}

// One row of 64 pixels of a conv3x3 8 -> 4 HALVES: rows r0..r2 (plane a of this lane's first
// patch pixel).
template <int HALVES>
__device__ __forceinline__ void conv_row(const char* r0, const char* r1, const char* r2, const float* w,
                                         const f32x4m (&bias)[HALVES], f32x4m (&out)[HALVES])
{
    float4 q[3][3][2];   // [t][ky][plane]
#pragma unroll
    for (int t = 0; t < 3; t++) {
        const char* r[3] = { r0, r1, r2 };
#pragma unroll
        for (int ky = 0; ky < 3; ky++) {
            q[t][ky][0] = *reinterpret_cast<const float4*>(r[ky] + 16 * t);
            q[t][ky][1] = *reinterpret_cast<const float4*>(r[ky] + kR8Plane + 16 * t);
        }
    }
    f32x4m acc[HALVES][2];
#pragma unroll
    for (int h = 0; h < HALVES; h++) {
        acc[h][0] = bias[h];
        acc[h][1] = (f32x4m){ 0.f, 0.f, 0.f, 0.f };
    }
    column4<0, HALVES>(w, q[0], acc, std::make_integer_sequence<int, 24 * HALVES>{});
    column4<1, HALVES>(w, q[1], acc, std::make_integer_sequence<int, 24 * HALVES>{});
    column4<2, HALVES>(w, q[2], acc, std::make_integer_sequence<int, 24 * HALVES>{});
#pragma unroll
    for (int h = 0; h < HALVES; h++) out[h] = acc[h][0] + acc[h][1];
}

// PReLU as prelu() rounds it: one of the two terms is zero, so the FMA rounds once
__device__ __forceinline__ float prelu_fma(float v, float a) { return fmaf(a, fminf(v, 0.0f), fmaxf(v, 0.0f)); }

// ---- a layer's epilogue: one pixel per lane, its 8 (or 4) sums in v ----
template <int MODE, typename TIN, typename TOUT>
struct RowEpi {
    static constexpr bool SHUFFLE = MODE == kShuffle || MODE == kShuffleSrc;
    static constexpr int HALVES = SHUFFLE ? 1 : 2;
    static constexpr int OPS = (72 * HALVES + 15) / 16;
    float w[OPS], w1 = 0.f;
    f32x4m bias[HALVES], bias1[2];
    const LayerArgs& la;
    __device__ __forceinline__ RowEpi(const LayerArgs& la_, int lane) : la(la_)
    {
#pragma unroll
        for (int s = 0; s < OPS; s++) w[s] = la.wa[s * 64 + lane];
#pragma unroll
        for (int h = 0; h < HALVES; h++) bias[h] = (f32x4m){ la.bias[4 * h], la.bias[4 * h + 1], la.bias[4 * h + 2], la.bias[4 * h + 3] };
        if constexpr (MODE == kPreluConv1x1) {
            w1 = la.w1[lane];
#pragma unroll
            for (int h = 0; h < 2; h++) bias1[h] = (f32x4m){ la.b1[4 * h], la.b1[4 * h + 1], la.b1[4 * h + 2], la.b1[4 * h + 3] };
        }
    }
    // what the epilogue reads from global memory, loaded before the layer's MFMAs
    struct Ahead {
        float4 f[2];
        TIN s;
    };
    __device__ __forceinline__ void ahead(Ahead& a, int x, int y, int W, int H, long fp) const
    {
        const int cx = clampi(x, 0, W - 1), cy = clampi(y, 0, H - 1);
        if constexpr (MODE == kPreluConv1x1) {
            const float4* f = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(la.feat) + static_cast<long>(cy) * fp) + 2 * cx;
            a.f[0] = f[0];
            a.f[1] = f[1];
        }
        if constexpr (MODE == kShuffleSrc) a.s = row_ptr<TIN>(la.src, la.ss, cy)[cx];
    }
    // the layer's 8 outputs (modes that end in a map or the next layer's ring)
    __device__ __forceinline__ void activate(f32x4m (&v)[HALVES], const Ahead& a) const
    {
#pragma unroll
        for (int h = 0; h < HALVES; h++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (MODE == kRelu || MODE == kReluDeconv) v[h][i] = fmaxf(v[h][i], 0.f);
                else if constexpr (MODE == kPrelu || MODE == kPreluConv1x1) v[h][i] = prelu_fma(v[h][i], la.alpha[4 * h + i]);
            }
        if constexpr (MODE == kPreluConv1x1) {
            f32x4m d[2] = { bias1[0], bias1[1] };
            one_by_one(v, d, std::make_integer_sequence<int, 16>{});
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int i = 0; i < 4; i++) v[h][i] = prelu_fma(add_skip(d[h][i], quad(a.f[h], i)), la.alpha1[4 * h + i]);
        }
    }
    // conv1x1: input channels 0, 4, 1, 5, 2, 6, 3, 7 in turn (the 16x16x4 form's order), both output quads
    template <int... I>
    __device__ __forceinline__ void one_by_one(const f32x4m (&v)[HALVES], f32x4m (&d)[2], std::integer_sequence<int, I...>) const
    {
        ((d[I % 2] = mma4<I>(&w1, v[I / 2 % 2][I / 4], d[I % 2])), ...);
    }
    __device__ __forceinline__ void store(const f32x4m (&v)[HALVES], const Ahead& a, int x, int y, long fp, float4* fout) const
    {
        if constexpr (SHUFFLE) {   // sub-pixels n: output (2x + n % 2, 2y + n / 2)
            f32x4m o = v[0];
            if constexpr (MODE == kShuffleSrc) {
                const float res = to_float<TIN>(a.s);
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] = add_skip(o[i], res);
            }
            store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y) + 2 * x, o[0], o[1]);
            store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y + 1) + 2 * x, o[2], o[3]);
        } else if constexpr (MODE == kReluDeconv) {
            // channels 0-3 and 4-7 as two chains, then their sum (the fused kernel's lanes)
            float o[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float s[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const float* k = la.k2 + 16 * h + q;
                    s[h] = fmaf(v[h][3], k[12], fmaf(v[h][2], k[8], fmaf(v[h][1], k[4], v[h][0] * k[0])));
                }
                o[q] = s[0] + s[1];
            }
            store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y) + 2 * x, o[0], o[1]);
            store_pair<TOUT>(row_ptr<TOUT>(la.dst, la.ds, 2 * y + 1) + 2 * x, o[2], o[3]);
        } else {
            float4* px = reinterpret_cast<float4*>(reinterpret_cast<char*>(fout) + static_cast<long>(y) * fp) + 2 * x;
            px[0] = make_float4(v[0][0], v[0][1], v[0][2], v[0][3]);
            px[1] = make_float4(v[1][0], v[1][1], v[1][2], v[1][3]);
        }
    }
};

// One pixel of a layer's output into the next layer's ring: plane a at `at`, image column gx,
// strip column `col`.  Columns outside the image take the nearest one inside, written along
// with it.
__device__ __forceinline__ void ring_put(char* at, const f32x4m& lo, const f32x4m& hi, bool edge, int gx, int col, int W)
{
    auto put = [&](char* p) {
        *reinterpret_cast<f32x4m*>(p) = lo;
        *reinterpret_cast<f32x4m*>(p + kR8Plane) = hi;
    };
    if (!edge) {
        put(at);
    } else if (gx >= 0 && gx < W) {
        put(at);
        if (gx == 0 && col > 0) put(at - 16);
        if (gx == W - 1) put(at + 16);   // the pitch has two columns more
    }
}

// The rows of a strip: ring l holds layer l's rows from base(l) on (layer 0: the map or L0),
// row v at v % 6.
struct RowsOf {
    int y0, nl, H;
    __device__ __forceinline__ int base(int l) const { return y0 - (nl - l); }
    // ring offset of image row `row` of layer l, the nearest row inside the image
    __device__ __forceinline__ unsigned off(int l, int row) const
    {
        return static_cast<unsigned>(clampi(row, 0, H - 1) - base(l)) % kSRows * kR8Row;
    }
};

// ---- the loaders: one pair of input rows per step, their loads a step ahead in registers ----

// a map's rows, 2 x 66 pixels x 2 channel quads over NT threads
template <int NT>
struct RowsMapFeed {
    static constexpr int N = 4 * kR8In, K = (N + NT - 1) / NT;
    f32x4m v[K];
    int o[K], at[K];
    const char* fin;
    long fp;
    int H, row, tid;
    unsigned off = 0;
    __device__ __forceinline__ RowsMapFeed(const RowsIo& c, int xs, int row0, int tid_)
        : fin(reinterpret_cast<const char*>(c.fin) + 32L * clampi(xs, 0, c.W - 1)), fp(c.fp), H(c.H), row(row0), tid(tid_)
    {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int e = min(tid + k * NT, N - 1), f = e % (2 * kR8In);
            o[k] = 32 * (clampi(xs + (f >> 1), 0, c.W - 1) - clampi(xs, 0, c.W - 1)) + 16 * (f & 1);
            at[k] = e / (2 * kR8In) * kR8Row + (f & 1) * kR8Plane + (f >> 1) * 16;
        }
    }
    __device__ __forceinline__ void fetch()
    {
        const char* p0 = fin + static_cast<long>(clampi(row, 0, H - 1)) * fp;
        const char* p1 = fin + static_cast<long>(clampi(row + 1, 0, H - 1)) * fp;
#pragma unroll
        for (int k = 0; k < K; k++)
            if (k == 0 || tid + k * NT < N) v[k] = *reinterpret_cast<const f32x4m*>((tid + k * NT < 2 * kR8In ? p0 : p1) + o[k]);
        row += 2;
    }
    __device__ __forceinline__ void store(char* ring)
    {
#pragma unroll
        for (int k = 0; k < K; k++)
            if ((k == 0 && NT <= N) || tid + k * NT < N) *reinterpret_cast<f32x4m*>(ring + off + at[k]) = v[k];
        off = off + 2 * kR8Row == kR8Plane ? 0 : off + 2 * kR8Row;
    }
};

// source rows as f32, 2 x 66 pixels
template <typename TIN>
struct RowsImageFeed {
    TIN v;
    const void* src;
    long ss;
    int H, row, col, at;
    bool low, mine;
    unsigned off = 0;
    __device__ __forceinline__ RowsImageFeed(const RowsIo& c, int xs, int row0, int tid) : src(c.src), ss(c.ss), H(c.H), row(row0)
    {
        low = tid < kR8In;
        mine = tid < 2 * kR8In;
        const int f = min(low ? tid : tid - kR8In, kR8In - 1);
        col = clampi(xs + f, 0, c.W - 1);
        at = (low ? 0 : kR8ImgRow) + f * 4;
    }
    __device__ __forceinline__ void fetch()
    {
        const TIN* p0 = row_ptr<TIN>(src, ss, clampi(row, 0, H - 1));
        const TIN* p1 = row_ptr<TIN>(src, ss, clampi(row + 1, 0, H - 1));
        v = (low ? p0 : p1)[col];
        row += 2;
    }
    __device__ __forceinline__ void store(char* img)
    {
        if (mine) *reinterpret_cast<float*>(img + off + at) = to_float<TIN>(v);
        off = off + 2 * kR8ImgRow == kR8ImgBytes ? 0 : off + 2 * kR8ImgRow;
    }
};

// ---- layer 0 from the source rows: row `ro` of the pair, one pixel per lane ----

// ACNetLegacy: conv3x3 1 -> 8 + ReLU, the FMAs in the fused kernel's order (patch column, then row)
struct L0Legacy {
    float w[2];
    f32x4m bias[2];
    __device__ __forceinline__ L0Legacy(const RowsIo& c, int lane)
    {
        w[0] = c.w0[lane];
        w[1] = c.w0[64 + lane];
#pragma unroll
        for (int h = 0; h < 2; h++) bias[h] = (f32x4m){ c.b0[4 * h], c.b0[4 * h + 1], c.b0[4 * h + 2], c.b0[4 * h + 3] };
    }
    template <int... I>
    __device__ __forceinline__ void chain(const float (&q)[9], f32x4m (&v)[2], std::integer_sequence<int, I...>) const
    {
        ((v[I % 2] = mma4<I>(w, q[I / 2 % 3 * 3 + I / 6], v[I % 2])), ...);   // I = (t * 3 + ky) * 2 + h
    }
    __device__ __forceinline__ void row(const float (&q)[9], f32x4m (&v)[2]) const
    {
        v[0] = bias[0];
        v[1] = bias[1];
        chain(q, v, std::make_integer_sequence<int, 18>{});
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int i = 0; i < 4; i++) v[h][i] = fmaxf(v[h][i], 0.f);
    }
};

// ACNet<8>: conv3x3 1 -> 8 + PReLU, each product and sum rounded in the reference's order
// (Backend.hpp:58-75)
struct L0Acnet8 {
    float w[9][8];
    const float* wts;
    __device__ __forceinline__ L0Acnet8(const RowsIo& c, int) : wts(c.w0)
    {
#pragma unroll
        for (int k = 0; k < 9; k++)
#pragma unroll
            for (int n = 0; n < 8; n++)
                w[k][n] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(wts[kA8OffW0 + k * 8 + n])));
    }
    __device__ __forceinline__ void row(const float (&q)[9], f32x4m (&v)[2]) const
    {
#pragma unroll
        for (int n = 0; n < 8; n++) {
            float s = __fmul_rn(q[0], w[0][n]);
#pragma unroll
            for (int k = 1; k < 9; k++) s = __fadd_rn(s, __fmul_rn(q[k], w[k][n]));
            v[n >> 2][n & 3] = prelu_fma(__fadd_rn(s, wts[kA8OffB0 + n]), wts[kA8OffAlpha0 + n]);
        }
    }
};

// ---- a strip ----

// Output rows [y0, y1) and columns [x0, x0 + out_cols) of a strip (out_cols at most rows8_out) of
// layers mid[0 .. NL - 2] and `end`.  Step s: the loader stores input pair s + 2, the first consumer
// of the input runs pair s, every layer after it two pairs later.
template <int HEAD, int NL, int MID, int MODE, typename TIN, typename TOUT>
__device__ __forceinline__ void rows8_strip(const RowsIo& c, const LayerArgs* mid, const LayerArgs& end, int x0, int out_cols,
                                            int y0, int y1, int turn, char* lds)
{
    constexpr int NT = rows8_threads<HEAD, NL>(), L0 = HEAD == kRowsMap ? 0 : 1;
    const int tid = threadIdx.x, lane = tid & 63;
    // waves 2 (l - 1), + 1: layer l (turned around from one workgroup to the next, as the first
    // layers start earlier and have more rows), then layer 0's two
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave < 2 * NL) wave = wave + 2 * turn >= 2 * NL ? wave + 2 * turn - 2 * NL : wave + 2 * turn;
    const int l = wave < 2 * NL ? (wave >> 1) + 1 : 0, ro = wave & 1;
    const RowsOf rw{ y0, NL, c.H };
    const int n = c.rows >> 1, nsteps = n + 2 * (NL - 1 + L0);
    const int xs = x0 - NL;                                    // image column of ring 0's column 0
    const bool edge = xs < 0 || xs + kR8In > c.W;
    char* const img = lds + NL * kR8Ring;

    using Feed = std::conditional_t<HEAD == kRowsMap, RowsMapFeed<NT>, RowsImageFeed<TIN>>;
    Feed feed(c, HEAD == kRowsMap ? xs : xs - 1, HEAD == kRowsMap ? rw.base(0) : rw.base(0) - 1, tid);
    char* const into = HEAD == kRowsMap ? lds : img;
    feed.fetch();
    auto run = [&](int first, int pairs, auto&& row) {   // `row(pair)` in steps first .. first + pairs - 1
        feed.store(into);
        feed.fetch();
        feed.store(into);
        feed.fetch();
        step_barrier();
        for (int s = 0; s < nsteps; s++) {
            feed.store(into);
            feed.fetch();
            if (s >= first && s < first + pairs) row(s - first);
            step_barrier();
        }
    };
    auto layer = [&](const auto& epi, auto last) {
        constexpr bool LAST = decltype(last)::value;
        using E = std::remove_cv_t<std::remove_reference_t<decltype(epi)>>;
        const char* in = lds + (l - 1) * kR8Ring + lane * 16;
        char* out = lds + l * kR8Ring + lane * 16;
        const int gx = xs + l + lane, gx1 = min(x0 + out_cols, c.W);   // image column of this lane's output
        run(2 * (l - 1 + L0), n + NL - l, [&](int p) {
            const int y = rw.base(l) + 2 * p + ro;
            if (y - 1 >= c.H) return;   // below the image (the last strip)
            typename E::Ahead a;
            epi.ahead(a, gx, y, c.W, c.H, c.fp);
            unsigned o[3];
#pragma unroll
            for (int k = 0; k < 3; k++)
                o[k] = HEAD == kRowsMap && l == 1 ? static_cast<unsigned>(2 * p + ro + k) % kSRows * kR8Row : rw.off(l - 1, y - 1 + k);
            f32x4m v[E::HALVES];
            conv_row<E::HALVES>(in + o[0], in + o[1], in + o[2], epi.w, epi.bias, v);
            epi.activate(v, a);
            if constexpr (LAST) {
                if (gx < gx1 && y < y1) epi.store(v, a, gx, y, c.fp, c.fout);
            } else {
                ring_put(out + static_cast<unsigned>(2 * p + ro) % kSRows * kR8Row, v[0], v[1], edge, gx, lane, c.W);
            }
        });
    };
    if (l == NL) {
        const RowEpi<MODE, TIN, TOUT> epi(end, lane);
        layer(epi, std::true_type{});
    } else if (l > 0) {
        if constexpr (NL > 1) {
            const RowEpi<MID, TIN, TOUT> epi(mid[l - 1], lane);
            layer(epi, std::false_type{});
        }
    } else if constexpr (HEAD != kRowsMap) {
        const std::conditional_t<HEAD == kRowsLegacy, L0Legacy, L0Acnet8> l0(c, lane);
        run(0, n + NL, [&](int p) {
            float q[9];
#pragma unroll
            for (int ky = 0; ky < 3; ky++) {
                const float* r = reinterpret_cast<const float*>(img + static_cast<unsigned>(2 * p + ro + ky) % kSRows * kR8ImgRow) + lane;
#pragma unroll
                for (int t = 0; t < 3; t++) q[3 * ky + t] = r[t];
            }
            f32x4m v[2];
            l0.row(q, v);
            ring_put(lds + static_cast<unsigned>(2 * p + ro) % kSRows * kR8Row + lane * 16, v[0], v[1], edge, xs + lane, lane, c.W);
        });
    }
}

// Workgroups of a launch per CU, at most (160 KB of LDS, four of the layers' waves per SIMD), and
// the waves per SIMD that makes, of which the registers are to allow six
template <int HEAD, int NL>
constexpr int rows8_per_cu()
{
    const int by_lds = static_cast<int>(160 * 1024 / rows8_lds<HEAD, NL>()), by_waves = 8 / NL;
    return by_lds < by_waves ? by_lds : by_waves;
}
template <int HEAD, int NL>
constexpr int rows8_waves()
{
    const int n = (rows8_per_cu<HEAD, NL>() * rows8_threads<HEAD, NL>() / 64 + 3) / 4;
    return n < 6 ? n : 6;
}

template <int HEAD, int NL, int MID, int MODE, typename TIN, typename TOUT>
__global__ __launch_bounds__((rows8_threads<HEAD, NL>()), (rows8_waves<HEAD, NL>())) void conv8_rows(const Rows8 c)
{
    __shared__ float4 lds[rows8_lds<HEAD, NL>() / 16];
    constexpr int out = rows8_out<HEAD, NL>();
    const int t = xcd_tile(strip_block(), gridDim.x * gridDim.y);
    const int ty = t / gridDim.x, tx = t - ty * gridDim.x;
    rows8_strip<HEAD, NL, MID, MODE, TIN, TOUT>(c, c.la, c.la[NL - 1], tx * out, out, ty * c.rows,
                                                min((ty + 1) * c.rows, c.H), (tx + ty) % NL, reinterpret_cast<char*>(lds));
}

// The strips of every image of a batch, numbered image by image: `out` columns x c.rows rows.
// from_m1: the launch reads map 1 and writes map 0 (else the other way).
template <int HEAD, int NL, int MID, int MODE, typename TIN, typename TOUT>
__global__ __launch_bounds__((rows8_threads<HEAD, NL>()), (rows8_waves<HEAD, NL>())) void conv8_rows_batch(const SplitDesc* __restrict__ desc, int n, int total,
                                                                                  int out, int from_m1, const Rows8 c0)
{
    __shared__ float4 lds[rows8_lds<HEAD, NL>() / 16];
    const int t = xcd_tile(strip_block(), total);
    const SplitDesc d = find_tile(desc, n, t);
    const int local = t - d.first_tile, ty = local / d.tiles_x, tx = local - ty * d.tiles_x;
    RowsIo c = c0;
    LayerArgs end = c0.la[NL - 1];
    c.fin = from_m1 ? d.m1 : d.m0;
    c.fout = from_m1 ? d.m0 : d.m1;
    c.fp = d.fp;
    c.src = d.src;
    c.ss = d.sstride;
    c.W = d.w;
    c.H = d.h;
    end.dst = d.dst;
    end.ds = d.dstride;
    rows8_strip<HEAD, NL, MID, MODE, TIN, TOUT>(c, c0.la, end, tx * out, out, ty * c.rows, min((ty + 1) * c.rows, c.H), (tx + ty) % NL,
                                                reinterpret_cast<char*>(lds));
}

// ---- launch ----

inline Rows8 rows8_args(const float4* in, float4* out, long fp, int W, int H, std::initializer_list<LayerArgs> layers)
{
    Rows8 c{};
    c.fin = in;
    c.fout = out;
    c.fp = fp;
    c.W = W;
    c.H = H;
    int i = 0;
    for (const LayerArgs& la : layers) c.la[i++] = la;
    return c;
}

// Rows per strip.  A strip of r rows takes r / 2 + 2 (layers - 1) steps and one or two more to
// start; with w waves per SIMD at work a step takes about 1150 (1 + w) cycles (two layers at
// 1080p: one strip per CU 2280, two 3510, three 4640, four 5660), so the heights that put 1, 2, ..
// strips on every CU are compared by that, and several rounds of the last.  One step to start for one
// or two layers, by small images: FSRCNNX<8> 640 x 360 43.8 us with two (16 rows, one strip per CU), 40.0
// with one (8 rows, two; 64 x 16 tiles before: 42.7), 327 x 641 44.4 / 39.7 (41.8); ACNetLegacy and
// ACNet<8> within 2% either way.
inline int rows8_rows(long strips, int H, int layers, int lead, int cus, int per_cu)
{
    const int start = layers <= 2 ? 1 : 2;
    long best = -1;
    int rows = (H + 1) / 2 * 2;
    for (int k = 1; k <= per_cu + 2; k++) {
        const int at = k < per_cu ? k : per_cu, rounds = k <= per_cu ? 1 : k == per_cu + 1 ? 2 : 4;
        const long segs = static_cast<long>(at) * rounds * cus / strips;
        if (segs < 1) continue;
        const int r = static_cast<int>(((H + segs - 1) / segs + 1) / 2 * 2);
        const long n = strips * ((H + r - 1) / r);
        const long cost = (r / 2 + 2 * (layers - 1 + lead) + start) * (2L + at * layers) * ((n + static_cast<long>(at) * cus - 1) / (static_cast<long>(at) * cus));
        if (best < 0 || cost < best) {
            best = cost;
            rows = r;
        }
    }
    return rows;
}

template <int HEAD, int NL, int MID, int MODE, typename TIN, typename TOUT>
inline hipError_t launch_rows8(Rows8 c, int cus, hipStream_t stream)
{
    const int out = rows8_out<HEAD, NL>(), strips = (c.W + out - 1) / out;
    c.rows = rows8_rows(strips, c.H, NL, HEAD == kRowsMap ? 0 : 1, cus, rows8_per_cu<HEAD, NL>());
    constexpr int threads = rows8_threads<HEAD, NL>();
    hipLaunchKernelGGL((conv8_rows<HEAD, NL, MID, MODE, TIN, TOUT>), dim3(strips, (c.H + c.rows - 1) / c.rows), dim3(threads), 0,
                       stream, c);
    return hipGetLastError();
}

} // namespace achip
