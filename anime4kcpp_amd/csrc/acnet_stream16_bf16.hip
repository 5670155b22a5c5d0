// The BF16 kernels of the streamed ACNetLegacy pass (acnet_stream16.hpp).
#include "acnet_stream16.hpp"

namespace achip {

template hipError_t launch_stream16_types<__bf16>(int, int, int, const void*, long, int, int, void*, long, const float*,
                                                  const uint4*, const float*, int, hipStream_t);
template hipError_t launch_stream16_batch_types<__bf16>(int, int, const BatchDesc*, int, int, int, int*, const float*,
                                                        const uint4*, const float*, int, hipStream_t);

} // namespace achip
