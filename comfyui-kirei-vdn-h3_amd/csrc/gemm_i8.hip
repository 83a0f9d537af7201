// The GEMM kernel (gemm_kernel.h) for one operand kind; a source of its own so that the three build in parallel.
#define VDNH3_GEMM_KERNEL
#include "gemm_kernel.h"

namespace vdnh3 {
template void launch_gemm_tiles<kI8>(int mi, const GemmArgs &args, hipStream_t stream);
}
