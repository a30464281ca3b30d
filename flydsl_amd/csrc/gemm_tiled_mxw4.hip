// Instantiations of the 256x256 tile (gemm_tiled8.h) for fp8 and fp6 activations against fp4 weights, dense; batches are a launch each.
// Against the 128x256 tile of the general MX kernel, whose A goes through registers and whose steps wait for LDS behind their
// barrier: fp8 x fp4 4096x4096x8192 169 -> 92 us (2.98 PFLOP/s), 8192x4096x2048 102 -> 57; the bits are the same.
#include "gemm_tiled8.h"

hipError_t psg_launch_tiled_mxw4(const A8W8Params& p, bool fp6, hipStream_t stream) {
    if (fp6) return p.out == OUT_BF16 ? launch_tiled8<KIND_MXA6W4, STORE_C>(p, stream) : launch_tiled8<KIND_MXA6W4, STORE_C_GENERIC>(p, stream);
    return p.out == OUT_BF16 ? launch_tiled8<KIND_MXA8W4, STORE_C>(p, stream) : launch_tiled8<KIND_MXA8W4, STORE_C_GENERIC>(p, stream);
}
