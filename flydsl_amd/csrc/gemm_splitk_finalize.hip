// Second pass of the split-K tiled path: sums the per-split accumulator slices in a fixed order (deterministic)
// and applies the same epilogue as the single-pass kernels.  One thread per four consecutive columns.
#include "psg_common.h"

namespace {

// SPLITS: slices, 0 = p.splits of them.  Everything a thread reads is asked for at once: one after the other the slices, the scales and the bias were three and more memory latencies
// of a launch that lasts four us.  us of the pair of launches before / now: fp8 96x4096x14336 (8 slices) 19.8 / 19.1, fp16 65x5120x8192 21.8 / 21.3, bf16 139x2112x7168 18.2 / 17.4, int8
// 384x1664x10240 20.6 / 20.2, with its quantiser and a bias 132x1408x8448 17.2 / 16.0; fp8 200x8192x8192 (2 slices) with both 28.9 / 28.5.
template <int IS_INT, int SPLITS>
__global__ void __launch_bounds__(256) k_splitk_finalize(A8W8Params p, const void* partial, int scaled) {
    using acc_t = typename std::conditional<IS_INT != 0, v4i, v4f>::type;
    const size_t quads = (size_t)p.M * (size_t)(p.N >> 2);
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= quads) return;
    const uint32_t row = (uint32_t)p.N >> 2;
    int m, n;
    if (quads <= 0xFFFFFFFFull) {  // (a division of 64 bits is a hundred instructions)
        m = (int)((uint32_t)q / row);
        n = (int)((uint32_t)q - (uint32_t)m * row) << 2;
    } else {
        m = (int)(q / row);
        n = (int)(q % row) << 2;
    }
    const size_t idx = (size_t)m * (size_t)p.N + (size_t)n;
    const size_t slice = (size_t)p.M * (size_t)p.N;
    const uint32_t* from = static_cast<const uint32_t*>(partial) + idx;
    acc_t part[SPLITS ? SPLITS : 1];
#pragma unroll
    for (int s = 0; s < (SPLITS ? SPLITS : 1); s++) part[s] = *reinterpret_cast<const acc_t*>(from + s * slice);
    float sa = 1.0f;
    v4f sb = {1.0f, 1.0f, 1.0f, 1.0f};
    if (scaled) {
        sa = p.sa[m];
        sb = *reinterpret_cast<const v4f*>(p.sb + n);
    }
    v2i bias = {0, 0};
    if (p.epi != EPI_NONE) bias = *reinterpret_cast<const v2i*>(p.bias + n);
    acc_t sum = part[0];
#pragma unroll
    for (int s = 1; s < SPLITS; s++) sum += part[s];
    if constexpr (SPLITS == 0)
        for (int s = 1; s < p.splits; s++) sum += *reinterpret_cast<const acc_t*>(from + s * slice);
    v4f x = {(float)sum[0], (float)sum[1], (float)sum[2], (float)sum[3]};
    if (scaled) x = (v4f){(x[0] * sa) * sb[0], (x[1] * sa) * sb[1], (x[2] * sa) * sb[2], (x[3] * sa) * sb[3]};
    const uint16_t* b = reinterpret_cast<const uint16_t*>(&bias);
    const v2i r = p.out == OUT_BF16 ? finish4_rt<OUT_BF16>(x, b, p.epi) : finish4_rt<OUT_FP16>(x, b, p.epi);
    *reinterpret_cast<v2i*>(static_cast<uint16_t*>(p.c) + idx) = r;
}

}  // namespace

// p.c / p.sa / p.sb / p.bias / p.epi / p.out describe the final output; p.splits slices of [M,N] accumulators at `partial`
hipError_t psg_launch_splitk_finalize(const A8W8Params& p, const void* partial, int is_int, int scaled, hipStream_t stream) {
    const size_t quads = (size_t)p.M * (size_t)(p.N >> 2);
    const unsigned grid = (unsigned)((quads + 255) / 256);
    auto go = [&](auto S) {
        if (is_int) hipLaunchKernelGGL((k_splitk_finalize<1, decltype(S)::value>), dim3(grid), dim3(256), 0, stream, p, partial, scaled);
        else hipLaunchKernelGGL((k_splitk_finalize<0, decltype(S)::value>), dim3(grid), dim3(256), 0, stream, p, partial, scaled);
    };
    switch (p.splits) {
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        case 4: go(std::integral_constant<int, 4>{}); break;
        case 5: go(std::integral_constant<int, 5>{}); break;
        case 6: go(std::integral_constant<int, 6>{}); break;
        case 7: go(std::integral_constant<int, 7>{}); break;
        case 8: go(std::integral_constant<int, 8>{}); break;
        default: go(std::integral_constant<int, 0>{}); break;
    }
    return hipGetLastError();
}
