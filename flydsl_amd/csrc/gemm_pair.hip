// Dense GEMM on 128x256 tiles, two workgroups per CU (mainloop: pair_loop.h), for int8, fp8, fp16 and bf16 operands.
//
// Bound: MFMA at the clock the power limit leaves; on long rows the 256x256 tile (gemm_tiled8.h), which moves two thirds of the bytes, is as fast or faster, on short
// ones, where a tile's start and end count, and for problems of few 256x256 tiles this one.  us, 256x256 tiles / 128x256 tiles with A through registers / these: fp8
// 8192x4096x4096 106.7 / 121.4 / 107.8, 8192x8192x1024 78.9 / 85.1 / 69.3, 1024x8192x2048 25.6 / 22.3 / 19.5, 1500x11264x4096 86.1 / 84.9 / 71.8, 5120x5120x8320
// 170 / 201 / 181; int8 4096x8192x2048 65.2 / 67.9 / 60.4, 4096x28672x8192 701 / 720 / 688 (the estimates of pick_plain_tile see it the other way round, 674 / 692, and take the larger tile); bf16 1500x5264x4096 84.4 / 64.6 / 57.7, 5133x5120x8320 348 / 371 / 346.
// Same bits.
#include "pair_loop.h"

namespace {

template <int KIND, int STORE>
__global__ void __launch_bounds__(256, 2) k_pair(A8W8Params p) {
    using acc_t = typename Acc<KIND>::type;
    using P = Pair<KIND>;
    constexpr int MR = P::MR, NR = P::NR, TM = P::TM, TN = P::TN;
    constexpr bool SCALED = KIND == KIND_INT8 || KIND == KIND_FP8, BIAS = STORE == STORE_C_GENERIC;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[P::LDS_BYTES];
    __shared__ float s_a[SCALED ? TM : 1], s_b[SCALED ? TN : 1];
    __shared__ __attribute__((aligned(8))) uint16_t s_bias[BIAS ? TN : 1];
    static_assert(P::fits(TM * 4 + TN * 6), "two workgroups a CU");
    const int tid = threadIdx.x;
    const int wave = wave_id();
    const int lane = tid & 63, li = lane & 15, lg = lane >> 4;
    int tm, tn;
    tile_coords((int)blockIdx.x, (p.M + TM - 1) / TM, (p.N + TN - 1) / TN, p.group_m, tm, tn);
    const int m0 = tm * TM, n0 = tn * TN;
    const uint32_t K = SCALED ? (uint32_t)p.K : (uint32_t)p.K * 2u;  // bytes of a row
    const int steps = (int)((K + TK - 1) / TK), per = STORE == STORE_ACC ? (steps + p.splits - 1) / p.splits : steps;
    uint32_t k0 = STORE == STORE_ACC ? blockIdx.y * (uint32_t)(per * TK) : 0u;
    if (k0 > K) k0 = K;
    const uint32_t kn = K - k0 < (uint32_t)(per * TK) ? K - k0 : (uint32_t)(per * TK);
    if (kn == 0) k0 = 0;
    const uint32_t b_step = p.b_rowmajor ? 128u : 2048u, b_half = p.b_rowmajor ? 64u : 1024u, b0 = k0 / TK * b_step;

    // rows >= M and weight rows >= N lie behind the descriptors' bounds and read as zero
    const __amdgpu_buffer_rsrc_t ra = make_rsrc_uniform(p.a + (uint64_t)m0 * K + k0, (uint64_t)(p.M - m0) * K - k0);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc_uniform(p.b + (uint64_t)n0 * K + b0, (uint64_t)(p.N - n0) * K - b0);
    uint32_t a_voff[4], b_voff[NR];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = (wave * 4 + j) * 8 + (lane >> 3);
        a_voff[j] = (uint32_t)row * K + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
#pragma unroll
    for (int ni = 0; ni < NR; ni++) b_voff[ni] = (uint32_t)(wave * NR + ni) * 16u * K + (p.b_rowmajor ? (uint32_t)li * K + (uint32_t)lg * 16u : (uint32_t)lane * 16u);
    if constexpr (SCALED && STORE != STORE_ACC) {
        if (tid < TM) s_a[tid] = p.sa[m0 + tid < p.M ? m0 + tid : p.M - 1];
        s_b[tid] = p.sb[n0 + tid < p.N ? n0 + tid : p.N - 1];
    }
    if constexpr (BIAS) s_bias[tid] = p.epi != EPI_NONE ? p.bias[n0 + tid < p.N ? n0 + tid : p.N - 1] : 0;

    acc_t acc[MR][NR];
    pair_loop<KIND>(acc, lds, ra, a_voff, rb, b_voff, (int)kn, wave, lane, b_step, b_half, ra, ra);

    if constexpr (STORE == STORE_ACC) {
        static_for<MR>([&](auto MI) {
            constexpr int mi = decltype(MI)::value;
            const int m = m0 + mi * 16 + li;
            if (m < p.M) {
                static_for<NR>([&](auto NI) {
                    constexpr int ni = decltype(NI)::value;
                    const int n = n0 + (wave * NR + ni) * 16 + lg * 4;
                    if (n < p.N) *reinterpret_cast<acc_t*>(static_cast<uint8_t*>(p.c) + (((size_t)blockIdx.y * (size_t)p.M + (size_t)m) * (size_t)p.N + (size_t)n) * 4) = acc[mi][ni];
                });
            }
        });
    } else {
        // C through LDS, in halves: the stores of one are under way while the other is converted
        const __amdgpu_buffer_rsrc_t rc = make_rsrc(static_cast<uint16_t*>(p.c) + (size_t)m0 * (size_t)p.N, (uint64_t)(p.M - m0) * (uint64_t)p.N * 2ull);
        v4f sb_v[NR], bias_v[NR] = {};
#pragma unroll
        for (int ni = 0; ni < NR; ni++) {
            if constexpr (SCALED) sb_v[ni] = *reinterpret_cast<const v4f*>(&s_b[(wave * NR + ni) * 16 + lg * 4]);
            if constexpr (BIAS) bias_v[ni] = load_bias4(&s_bias[(wave * NR + ni) * 16 + lg * 4], p.out, p.epi);
        }
        static_for<2>([&](auto HALF) {
            constexpr int half = decltype(HALF)::value;
            epi_dispatch<STORE, false>(p.out, p.epi, [&](auto finish4) __attribute__((always_inline)) {
                static_for<MR / 2>([&](auto MI) {
                    constexpr int mi = half * (MR / 2) + decltype(MI)::value;
                    float sa = 0.f;
                    if constexpr (SCALED) sa = s_a[mi * 16 + li];
                    static_for<NR>([&](auto NI) {
                        constexpr int ni = decltype(NI)::value;
                        const acc_t r = acc[mi][ni];
                        v4f x;
                        if constexpr (!SCALED) {
                            x = (v4f){(float)r[0], (float)r[1], (float)r[2], (float)r[3]};
                        } else {
                            const v4f sb = sb_v[ni];
                            x = (v4f){((float)r[0] * sa) * sb[0], ((float)r[1] * sa) * sb[1], ((float)r[2] * sa) * sb[2], ((float)r[3] * sa) * sb[3]};
                        }
                        *reinterpret_cast<v2i*>(pair_c_at(lds, mi, wave * NR + ni, li, lg)) = finish4(x, bias_v[ni]);
                    });
                });
            });
            __syncthreads();
            pair_store_rows(lds, half, rc, n0, p.N, tid);
        });
    }
}

template <int KIND>
void go(const A8W8Params& p, int store, dim3 grid, hipStream_t stream) {
    if (store == STORE_ACC) hipLaunchKernelGGL((k_pair<KIND, STORE_ACC>), grid, dim3(256), 0, stream, p);
    else if (store == STORE_C) hipLaunchKernelGGL((k_pair<KIND, STORE_C>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((k_pair<KIND, STORE_C_GENERIC>), grid, dim3(256), 0, stream, p);
}

}  // namespace

// store: STORE_ACC (p.splits slices), STORE_C or STORE_C_GENERIC
hipError_t psg_launch_pair(const A8W8Params& p, int kind, int store, hipStream_t stream) {
    A8W8Params q = p;
    q.splits = store == STORE_ACC && p.splits > 1 ? p.splits : 1;
    const dim3 grid((unsigned)(((p.M + 127) / 128) * ((p.N + 255) / 256)), (unsigned)q.splits);
    switch (kind) {
        case KIND_INT8: go<KIND_INT8>(q, store, grid, stream); break;
        case KIND_FP8: go<KIND_FP8>(q, store, grid, stream); break;
        case KIND_FP16: go<KIND_FP16>(q, store, grid, stream); break;
        case KIND_BF16: go<KIND_BF16>(q, store, grid, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
