// What the streamed kernels share: a workgroup takes a strip of the image (some columns over a
// range of rows), and row pairs move through its layers, one pair per step, over rings of three
// pairs in LDS.  A layer's pairs start one row below those of the layer before it, so pair p
// needs exactly that layer's pairs p and p + 1 (patch rows 2p .. 2p + 3 of its strip), and layer
// l computes pair s - 2 l in step s.  In a step a layer reads pairs p, p + 1 while the layer
// before it writes pair p + 2, so reads and writes never meet and one barrier per step is
// enough.
#pragma once

#include "acnet_device.hpp"
#include "acnet_kernels.hpp"

namespace achip {

constexpr int kSCols = 80;                      // pitch of a ring's planes, in pixels (a multiple of 256 bytes)
constexpr int kSRows = 6;                       // rows of a ring
constexpr unsigned kSRowBytes = kSCols * 16;    // 16 bytes per pixel: 8 x 16-bit channels or 4 x f32
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

// ---- the heights of strips (host) ----
// Steps of a strip of `rows` output rows and `layers` layers after layer 0: its row pairs and
// the lag of the layers and the loader.
inline int strip_steps(int rows, int layers) { return (rows + 1) / 2 + kSLag * (layers + 1); }

// What strips of `rows` rows of an image of `strips` strips x H rows take on a device of `cus` compute
// units that hold per_cu workgroups each.  Measured (u8 in FP16, 4 to 18 blocks and ACNetLegacy,
// 256 x 256 to 4K): a strip of r rows with a compute unit of its own takes time with r + 3 (layers + 1)
// (the steps that fill and drain it, two per layer, run fewer layers than the rest), two to a compute
// unit 4/3 of that.
inline long strip_cost(long strips, int H, int layers, int cus, int per_cu, int rows)
{
    const long n = strips * ((H + rows - 1) / rows), all = static_cast<long>(per_cu) * cus;
    return (rows + 3L * (layers + 1)) * (n <= cus ? 3L : (2L + per_cu) * ((n + all - 1) / all));
}

// Rows per strip: the heights that fill one workgroup per CU or 1, 2, 4 rounds of all, the cheapest by
// that count.  ACNetLegacy, us: 1080p 64 rows 47 (36: 58, 80: 55); 4K 270 rows 150 (128: 149, 64: 163);
// 800 x 600 16 rows 21.8 (32 rows, one per CU: 23.7; 64 x 32 tiles before: 22); 256 x 256 4 rows 12.7
// (8: 13.8, 16: 17).
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
        const long cost = strip_cost(strips, H, layers, cus, per_cu, r);
        if (best < 0 || cost < best) {
            best = cost;
            rows = r;
        }
    }
    return rows;
}

// Rows per strip of a tile queue over n images (sizes w, h of a[i]) with out_cols output
// columns per strip.  In steps of a full device, two workgroups on every compute unit at different
// layers: strips that get a compute unit each take 0.95 a step, one round of two per compute unit 1.4
// (all of them in the same layers at a time), more strips the sum of their steps over the workgroups and
// 0.8 of a strip for the uneven end.  The least of these over 28 batches (8 of 128 x 128 up to 34 images of
// 11 Mpix, u8 in FP16) is within 1% of the best of 14 heights on average and 9% at worst.
template <class A>
inline int batch_strip_rows(const A* a, int n, int out_cols, int layers, int cus)
{
    double best = -1.0;
    int rows = 64, tallest = 1;
    for (int i = 0; i < n; i++) tallest = a[i].h > tallest ? a[i].h : tallest;
    for (int r : { 8, 12, 16, 20, 24, 32, 40, 48, 64, 80, 96, 128, 192, 256 }) {
        double strips = 0.0, steps = 0.0;
        for (int i = 0; i < n; i++) {
            const double s = (a[i].w + out_cols - 1) / out_cols, k = (a[i].h + r - 1) / r;
            strips += s * k;
            steps += s * ((a[i].h + 1) / 2 + k * strip_steps(0, layers));
        }
        const double strip = strip_steps(r < tallest ? r : tallest, layers);
        const double cost = strips <= cus ? 0.95 * strip : strips <= 2.0 * cus ? 1.4 * strip : steps / (2.0 * cus) + 0.8 * strip;
        if (best < 0.0 || cost < best) {
            best = cost;
            rows = r;
        }
    }
    return rows;
}

} // namespace achip
