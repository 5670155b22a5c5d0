// The BF16 kernels of the streamed ACNet<8> pass (acnet8_stream16.hpp).
#include "acnet8_stream16.hpp"

namespace achip {

template hipError_t launch_acnet8_16_types<__bf16>(int, int, int, const void*, long, int, int, void*, long, const float*,
                                                    const uint4*, void*, int, hipStream_t);

} // namespace achip
