// mxfp8_quant.hpp -- host launch interface of the MX-FP8 quantiser
// (mxfp8_quant.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace wave {
namespace quant {

// X [outer][n][inner] (contiguous; dtype wave::kF32 / kF16 / kBF16) -> E
// e4m3 bytes of the same layout and S e8m0 bytes [outer][ceil(n/32)][inner]:
// blocks of 32 along n.
hipError_t launch_mxfp8(const void *X, void *E, void *S, size_t outer, size_t n, size_t inner,
                        int dtype, hipStream_t stream);

} // namespace quant
} // namespace wave
