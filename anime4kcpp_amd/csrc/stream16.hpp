// The streamed form of the 16-bit MFMA passes: one wave per layer, rows flowing through all
// layers in one launch.
//
// A workgroup owns a strip: 80 columns of the image (the output columns plus a margin of one
// pixel per layer on each side) over a range of rows.  Every 8 -> 8 layer is a wave of its
// own that keeps its A operands and bias in registers for the whole strip.  The waves advance
// in steps of one row pair; a layer's pairs start one row below those of the layer before it,
// so pair p needs exactly that layer's pairs p and p + 1 (patch rows 2p .. 2p + 3 of its
// strip), and layer l computes pair s - 2 l in step s.  Between layers only a ring of three
// pairs exists, in LDS: a layer reads pairs p, p + 1 while the layer before it writes pair
// p + 2, so the reads and writes of a step never meet and one barrier per step is enough.
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

#include "acnet_device.hpp"
#include "acnet_kernels.hpp"
#include "mfma16.hpp"

namespace achip {

constexpr int kSPh = 5;                         // items of a unit
constexpr int kSCols = 16 * kSPh;               // columns of a strip's planes
constexpr int kSRows = 6;                       // rows of a ring
constexpr unsigned kSRowBytes = kSCols * 16;    // 8 x 16-bit channels per pixel
constexpr unsigned kSRingBytes = kSRows * kSRowBytes;
constexpr int kSLag = 2;                        // steps between consecutive layers

// End of a step: this wave's LDS accesses are done, then the workgroup's barrier.  Global
// loads and stores stay in flight across it (each wave waits for its own loads where it uses
// them, and no wave reads what another stored to global memory).
__device__ __forceinline__ void step_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Byte offset of a row of a ring (row: counted from the layer's first row, >= 0), advanced by
// one row pair per step without a division.
struct RingRow {
    unsigned off;
    __device__ __forceinline__ explicit RingRow(int row) : off(static_cast<unsigned>(row) % kSRows * kSRowBytes) {}
    __device__ __forceinline__ void next_pair()
    {
        off += 2 * kSRowBytes;
        off = min(off, off - kSRingBytes);   // unsigned: below the ring's end the difference wraps
    }
};

// The rows and steps of the layers 0 .. last of a strip with output rows [y0, y1) (y1 - y0
// even, or y1 the image's end).  Layer l's pair p is rows base(l) + 2p, + 1; pairs that lie
// outside the image are left out.
// lead: 1 where a loader fills layer 0's source rows (it counts as layer -1), 0 where the loader
// fills layer 0's ring itself.
struct StripRows {
    int y0, y1, H, last, s0;
    __device__ __forceinline__ StripRows(int y0_, int y1_, int H_, int last_, int lead) : y0(y0_), y1(y1_), H(H_), last(last_), s0(0)
    {
        s0 = first(0) - kSLag * lead;
    }
    __device__ __forceinline__ int base(int l) const { return y0 - (last - l); }
    __device__ __forceinline__ int first(int l) const { return max(-base(l), 0) >> 1; }
    __device__ __forceinline__ int end(int l) const { return (min(y1 + (last - l), H) - base(l) + 1) >> 1; }
    __device__ __forceinline__ int step(int l, int p) const { return p + kSLag * l - s0; }
    __device__ __forceinline__ int steps() const { return step(last, end(last)); }
    // Whether pair p's patch reaches outside the image, and for those pairs the offset of patch
    // row g in the ring of layer l - 1: the nearest row inside.
    __device__ __forceinline__ bool clamped(int l, int p) const { const int r = base(l) + 2 * p; return r < 1 || r + 2 >= H; }
    __device__ __forceinline__ unsigned clamped_off(int l, int p, int g) const
    {
        return RingRow(clampi(base(l) + 2 * p - 1 + g, 0, H - 1) - base(l - 1)).off;
    }
};

// ---- loaders ----
// One wave: pairs first .. end - 1 of rows row0 + 2p, + 1 (clamped to the image) of the columns
// xs .. xs + COLS - 1 (clamped) into a ring, put(row of the pair, column, element) storing one
// element and next() moving on by a pair.  The rows of the next AHEAD pairs are in flight in
// registers: a step is shorter than a load's latency.
template <typename T, int COLS, int AHEAD, class Put, class Next>
__device__ __forceinline__ void strip_loader(const void* __restrict__ src, long ss, int W, int H, int xs, int row0, int first,
                                             int end, int nsteps, int lane, Put put, Next next)
{
    static_assert(COLS > 64 && COLS <= 96, "three elements per lane and pair");
    // lane: column lane of both rows, and column 64 + lane % 32 of row lane / 32
    const int ct = 64 + (lane & 31);
    const int c0 = clampi(xs + lane, 0, W - 1), c2 = clampi(xs + ct, 0, W - 1);
    const bool low = lane < 32, tail = ct < COLS;
    int row = row0 + 2 * first;
    T v[AHEAD][3];
    auto fetch = [&](T (&t)[3]) {
        const T* r0 = row_ptr<T>(src, ss, clampi(row, 0, H - 1));
        const T* r1 = row_ptr<T>(src, ss, clampi(row + 1, 0, H - 1));
        t[0] = r0[c0];
        t[1] = r1[c0];
        t[2] = (low ? r0 : r1)[c2];
        row += 2;
    };
    auto store = [&](const T (&t)[3]) {
        put(0, lane, t[0]);
        put(1, lane, t[1]);
        if (tail) put(low ? 0 : 1, ct, t[2]);
        next();
    };
#pragma unroll
    for (int u = 0; u < AHEAD; u++) fetch(v[u]);
    int s = 0;
    for (int left = end - first; left >= AHEAD; left -= AHEAD) {
#pragma unroll
        for (int u = 0; u < AHEAD; u++) {
            store(v[u]);
            fetch(v[u]);
            step_barrier();
        }
        s += AHEAD;
    }
    const int rest = (end - first) % AHEAD;
#pragma unroll
    for (int u = 0; u < AHEAD - 1; u++) {
        if (u < rest) {
            store(v[u]);
            step_barrier();
        }
    }
    for (s += rest; s < nsteps; s++) step_barrier();
}

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

// ---- the heights of strips (host) ----
// Steps of a strip of `rows` output rows and `layers` layers after layer 0: its row pairs and
// the lag of the layers and the loader.
inline int strip_steps(int rows, int layers) { return (rows + 1) / 2 + kSLag * (layers + 1); }

// Rows per strip of an image of `strips` strips x H rows on a device of `cus` compute units that
// hold per_cu workgroups each.  Measured on 1080p and 4K u8 in FP16 (8 layers, two per CU): a
// step takes about 0.72 us with one workgroup per CU and 0.97 us with two, so the candidates are
// the heights that fill one workgroup per CU or 1, 2, 4 rounds of all, and the cheapest by
// that count is taken.  1080p: 64 rows 46 us (32: 56, 136: 62); 4K: 270 rows 150 (128: 149, 64:
// 163); 256 x 256: 4 rows 12.4 (2: 14.5, 16: 17).
inline int strip_rows(long strips, int H, int layers, int cus, int per_cu)
{
    long best = -1;
    int rows = (H + 1) / 2 * 2;
    const int rounds[] = { 0, 1, 2, 4 };
    const long all = static_cast<long>(per_cu) * cus;
    for (int k : rounds) {
        const long segs = (k ? k * all : cus) / strips;
        if (segs < 1) continue;
        const int r = static_cast<int>(((H + segs - 1) / segs + 1) / 2 * 2);
        const long n = strips * ((H + r - 1) / r);
        const long cost = strip_steps(r, layers) * (n <= cus ? 3L : (2L + per_cu) * ((n + all - 1) / all));
        if (best < 0 || cost < best) {
            best = cost;
            rows = r;
        }
    }
    return rows;
}

// Rows per strip of a tile queue over n images (sizes w, h of a[i]) with out_cols output
// columns per strip: the height whose steps, over the two workgroups of every CU, plus half a
// strip's for the uneven end, are fewest.
template <class A>
inline int batch_strip_rows(const A* a, int n, int out_cols, int layers, int cus)
{
    double best = -1.0;
    int rows = 64;
    for (int r : { 16, 32, 48, 64, 96, 128, 192, 256, 512 }) {
        double steps = 0.0;
        for (int i = 0; i < n; i++)
            steps += static_cast<double>((a[i].w + out_cols - 1) / out_cols) *
                     (a[i].h / 2 + static_cast<double>((a[i].h + r - 1) / r) * strip_steps(0, layers));
        const double cost = steps / (2.0 * cus) + 0.5 * strip_steps(r, layers);
        if (best < 0.0 || cost < best) {
            best = cost;
            rows = r;
        }
    }
    return rows;
}

} // namespace achip
