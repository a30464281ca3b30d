// Instantiations of the tiled MFMA mainloop (gemm_tiled.h; 256x256 gemm_tiled8.h) for fp8 and fp6 activations against fp4 weights, dense; batches are
// a launch each.  Against the 128x256 tile of the general MX kernel, whose A goes through registers and whose steps wait for LDS behind their
// barrier, the 256x256 tile took fp8 x fp4 4096x4096x8192 from 169 to 92 us (2.98 PFLOP/s), 8192x4096x2048 from 102 to 57; the bits are the same.
#include "gemm_tiled8.h"

namespace {

template <int KIND, int STORE>
hipError_t launch_w4(const A8W8Params& p, int tile_m, int tile_n, hipStream_t stream) {
    const bool large = tile_m == 256 && tile_n == 256;
    if (large && c_in_descriptor(p, 256)) return launch_tiled8<KIND, STORE>(p, stream);
    if (large || (tile_m == 128 && tile_n == 256)) return launch_one<KIND, 8, 4, 1, STORE>(p, stream);
    if (tile_m == 64 && tile_n == 256) return launch_one<KIND, 4, 4, 1, STORE>(p, stream);
    if (tile_m == 32 && tile_n == 256) return launch_one<KIND, 2, 4, 1, STORE>(p, stream);
    if (tile_m == 64 && tile_n == 128) return launch_one<KIND, 4, 2, 1, STORE>(p, stream);
    if (tile_m == 32 && tile_n == 128) return launch_one<KIND, 2, 2, 1, STORE>(p, stream);
    return hipErrorInvalidConfiguration;
}

}  // namespace

hipError_t psg_launch_tiled_mxw4(const A8W8Params& p, bool fp6, int tile_m, int tile_n, hipStream_t stream) {
    if (fp6) return p.out == OUT_BF16 ? launch_w4<KIND_MXA6W4, STORE_C>(p, tile_m, tile_n, stream) : launch_w4<KIND_MXA6W4, STORE_C_GENERIC>(p, tile_m, tile_n, stream);
    return p.out == OUT_BF16 ? launch_w4<KIND_MXA8W4, STORE_C>(p, tile_m, tile_n, stream) : launch_w4<KIND_MXA8W4, STORE_C_GENERIC>(p, tile_m, tile_n, stream);
}
