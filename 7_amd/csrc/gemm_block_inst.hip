// gemm_block_inst.hip -- explicit instantiation of one (input dtype, output
// dtype) slice of the small-block GEMM (WAVE_IN / WAVE_OUT, one compile each).
#include "gemm_block.hpp"

namespace wave {
namespace gemm {
namespace block {
template hipError_t launch_block<WAVE_IN, WAVE_OUT>(const BlockParams &, int, int, bool, bool,
                                                    hipStream_t);
} // namespace block
} // namespace gemm
} // namespace wave
