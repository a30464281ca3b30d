// Tiles of the dense MXFP4 GEMM: 128x256 on its own mainloop (gemm_mx_pair.hip), the smaller ones on the register-staged one (gemm_tiled.h).
#include "gemm_tiled.h"

hipError_t psg_launch_mx_pair(const A8W8Params& p, int store, hipStream_t stream);

namespace {

template <int STORE>
hipError_t launch_fp4(const A8W8Params& p, int tile_m, int tile_n, hipStream_t stream) {
    constexpr int KIND = KIND_MXFP4;
    // there is one large tile, whichever is asked for
    const bool large = (tile_m == 256 && tile_n == 256) || (tile_m == 128 && (tile_n == 256 || tile_n == 512));
    if (large && c_in_descriptor(p, 128)) return psg_launch_mx_pair(p, STORE, stream);
    if (large || (tile_m == 64 && tile_n == 256)) return launch_one<KIND, 4, 4, 1, STORE>(p, stream);
    if (tile_m == 32 && tile_n == 256) return launch_one<KIND, 2, 4, 1, STORE>(p, stream);
    if (tile_m == 64 && tile_n == 128) return launch_one<KIND, 4, 2, 1, STORE>(p, stream);
    if (tile_m == 32 && tile_n == 128) return launch_one<KIND, 2, 2, 1, STORE>(p, stream);
    return hipErrorInvalidConfiguration;
}

}  // namespace

hipError_t psg_launch_tiled_mxfp4(const A8W8Params& p, int store, int tile_m, int tile_n, hipStream_t stream) {
    if (store == STORE_ACC) return launch_fp4<STORE_ACC>(p, tile_m, tile_n, stream);
    if (store == STORE_C_GENERIC) return launch_fp4<STORE_C_GENERIC>(p, tile_m, tile_n, stream);
    return launch_fp4<STORE_C>(p, tile_m, tile_n, stream);
}
