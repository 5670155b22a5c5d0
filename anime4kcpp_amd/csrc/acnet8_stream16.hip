// The FP16 kernels of the streamed ACNet<8> pass (acnet8_stream16.hpp) and its launch entry
// points; the BF16 kernels are compiled beside it (acnet8_stream16_bf16.hip).
#include "acnet8_stream16.hpp"

namespace achip {

long acnet8_map16_pitch(int w) { return (static_cast<long>(w) * 16 + 255) / 256 * 256; }

extern template hipError_t launch_acnet8_16_types<__bf16>(int, int, int, const void*, long, int, int, void*, long, const float*,
                                                           const uint4*, void*, int, hipStream_t);

hipError_t launch_acnet8_16(int bf16, int blocks, int stype, int dtype, const void* src, long ss, int W, int H, void* dst,
                            long ds, const float* wts, const void* wa16, void* workspace, int cus, hipStream_t stream)
{
    const uint4* wa = static_cast<const uint4*>(wa16);
    if (bf16) return launch_acnet8_16_types<__bf16>(blocks, stype, dtype, src, ss, W, H, dst, ds, wts, wa, workspace, cus, stream);
    return launch_acnet8_16_types<_Float16>(blocks, stype, dtype, src, ss, W, H, dst, ds, wts, wa, workspace, cus, stream);
}

} // namespace achip
