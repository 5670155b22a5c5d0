// The FP16 kernels of the streamed ACNetLegacy pass (acnet_stream16.hpp), its configurations and
// its launch entry points; the BF16 kernels are compiled beside it (acnet_stream16_bf16.hip).
#include <algorithm>

#include "acnet_stream16.hpp"

namespace achip {

// 64-column strips.  Configuration 0 chooses the strips' height for the image (strip_rows) or
// the batch (batch_strip_rows); the serving loop's steps cut images at multiples of the
// height given here.  Configuration 1 takes 128 rows always.
const Fp32Config kStreamConfigs[] = {
    { kSLOut, 64, kSLThreads, 0, static_cast<int>(kSLLds) },
    { kSLOut, 128, kSLThreads, 0, static_cast<int>(kSLLds) },
};
const int kStreamConfigCount = sizeof(kStreamConfigs) / sizeof(kStreamConfigs[0]);

bool stream16_config_suits(int cfg, int w, int h, int cus)
{
    if (cfg == 0) return true;
    const long strips = (static_cast<long>(w) + kSLOut - 1) / kSLOut;
    const long rule = strip_cost(strips, h, kSLLayers, cus, 2, strip_rows(strips, h, kSLLayers, cus, 2));
    return strip_cost(strips, h, kSLLayers, cus, 2, std::min(kStreamConfigs[cfg].th, (h + 1) / 2 * 2)) * 20 <= rule * 21;
}

int stream16_batch_rows(int cfg, const BatchDesc* desc, int n, int cus)
{
    return cfg ? kStreamConfigs[cfg].th : batch_strip_rows(desc, n, kSLOut, kSLLayers, cus);
}

template hipError_t launch_stream16_types<_Float16>(int, int, int, const void*, long, int, int, void*, long, const float*,
                                                  const uint4*, const float*, int, hipStream_t);
template hipError_t launch_stream16_batch_types<_Float16>(int, int, const BatchDesc*, int, int, int, int*, const float*,
                                                        const uint4*, const float*, int, hipStream_t);
extern template hipError_t launch_stream16_types<__bf16>(int, int, int, const void*, long, int, int, void*, long,
                                                          const float*, const uint4*, const float*, int, hipStream_t);
extern template hipError_t launch_stream16_batch_types<__bf16>(int, int, const BatchDesc*, int, int, int, int*, const float*,
                                                                const uint4*, const float*, int, hipStream_t);

hipError_t launch_stream16(int bf16, int cfg, int stype, int dtype, const void* src, long ss, int W, int H, void* dst,
                           long ds, const float* wts, const void* wa, const float* wa0, int cus, hipStream_t stream)
{
    const uint4* a = static_cast<const uint4*>(wa);
    if (cfg < 0 || cfg >= kStreamConfigCount) return hipErrorInvalidValue;
    if (bf16) return launch_stream16_types<__bf16>(cfg, stype, dtype, src, ss, W, H, dst, ds, wts, a, wa0, cus, stream);
    return launch_stream16_types<_Float16>(cfg, stype, dtype, src, ss, W, H, dst, ds, wts, a, wa0, cus, stream);
}

hipError_t launch_stream16_batch(int bf16, int stype, int dtype, const BatchDesc* desc, int n, int total, int rows,
                                 int* counter, const float* wts, const void* wa, const float* wa0, int max_wg,
                                 hipStream_t stream)
{
    const uint4* a = static_cast<const uint4*>(wa);
    if (bf16) return launch_stream16_batch_types<__bf16>(stype, dtype, desc, n, total, rows, counter, wts, a, wa0, max_wg, stream);
    return launch_stream16_batch_types<_Float16>(stype, dtype, desc, n, total, rows, counter, wts, a, wa0, max_wg, stream);
}

} // namespace achip
