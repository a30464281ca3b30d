// Dense MXFP4 x MXFP4 GEMM on 128x256 tiles, two workgroups per CU (mainloop: pair_loop.h).
//
// Bound: MFMA at the clock the power limit leaves, and for short K the start and the end of a tile.  us, 256x256 tiles of eight wavefronts / these, weights in
// memory: 4096x7168x2048 42.9 / 39.4, 4096x4096x4096 38.8 / 36.9, 8192x8192x1024 59.6 / 50.9, 6000x3584x4608 68 / 54, 8192x4096x8192 128.6 / 123.1, each in
// its best tile order; 128x256 tiles of one workgroup a CU / these: 1000x7168x2048 15.4 / 13.1.
// Scales off 16 bytes (three DMAs of a wavefront a step instead of one) cost 0 to 5 %; us 256x256 tiles / 64x256 tiles / these: 4096x7168x2048 44.6 / 51.4 / 41.3, 8192x4096x8192 126 /
// 163 / 121, 1024x8192x8192 41.1 / 52.6 / 37.1, 300x28672x1024 16.0 / 17.9 / 15.9.
#include "pair_loop.h"

namespace {

// STORE_ACC: raw accumulators of the K range blockIdx.y -> slice blockIdx.y of p.c ([splits][M][N] floats)
// SCB: bytes of scales a lane fetches, 16 or, where they are not on 16 bytes, 4
template <int STORE, int OUT, int SCB>
__global__ void __launch_bounds__(256, 2) k_mx_pair(A8W8Params p) {
    constexpr int MR = MxPair::MR, NR = MxPair::NR, TM = MxPair::TM, TN = MxPair::TN;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[MxPair::LDS_BYTES];
    static_assert(MxPair::fits(0), "two workgroups a CU");
    const int tid = threadIdx.x;
    const int wave = wave_id();
    const int lane = tid & 63, li = lane & 15, lg = lane >> 4;
    int tm, tn;
    tile_coords((int)blockIdx.x, (p.M + TM - 1) / TM, (p.N + TN - 1) / TN, p.group_m, tm, tn);
    const int m0 = tm * TM, n0 = tn * TN;
    const uint32_t row_bytes = (uint32_t)p.K >> 1;
    const uint32_t chunk_bytes = (uint32_t)(p.K >> 8) * 256u;  // one 32-row chunk of shuffled scales
    const int steps = p.K >> 8, per = STORE == STORE_ACC ? (steps + p.splits - 1) / p.splits : steps;
    const int kt0 = STORE == STORE_ACC ? (int)blockIdx.y * per : 0, left = steps - kt0;
    const int KT = left < per ? (left > 0 ? left : 0) : per, at = KT ? kt0 : 0;

    // rows >= M and weight rows >= N lie behind the descriptors' bounds and read as zero
    const __amdgpu_buffer_rsrc_t ra = make_rsrc_uniform(p.a + (uint64_t)m0 * row_bytes + (uint32_t)at * TK, (uint64_t)(p.M - m0) * row_bytes - (uint32_t)at * TK);
    const __amdgpu_buffer_rsrc_t rb = make_rsrc_uniform(p.b + (uint64_t)n0 * row_bytes + (uint32_t)at * 2048u, (uint64_t)(p.N - n0) * row_bytes - (uint32_t)at * 2048u);
    uint32_t a_voff[4], b_voff[NR];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = (wave * 4 + j) * 8 + (lane >> 3);
        a_voff[j] = (uint32_t)row * row_bytes + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
#pragma unroll
    for (int ni = 0; ni < NR; ni++) b_voff[ni] = (uint32_t)(wave * NR + ni) * 16u * row_bytes + (uint32_t)lane * 16u;
    const uint8_t *sa = p.mx_sa + (uint64_t)(m0 >> 5) * chunk_bytes + (uint32_t)at * 256u, *sb = p.mx_sb + (uint64_t)(n0 >> 5) * chunk_bytes + (uint32_t)at * 256u;
    const uint64_t sa_bytes = (uint64_t)(((p.M + 31) >> 5) - (m0 >> 5)) * chunk_bytes - (uint32_t)at * 256u, sb_bytes = (uint64_t)((p.N >> 5) - (n0 >> 5)) * chunk_bytes - (uint32_t)at * 256u;

    v4f acc[MR][NR];
    if constexpr (SCB == 16) {
        const bool a_side = wave == 0 || wave == 3;
        const uint32_t s_voff = (uint32_t)((a_side ? 0 : (wave - 1) * 4) + (lane >> 4)) * chunk_bytes + (uint32_t)(lane & 15) * 16u;
        const __amdgpu_buffer_rsrc_t rs = make_rsrc_uniform(a_side ? sa : sb, a_side ? sa_bytes : sb_bytes);
        pair_loop<KIND_MXFP4>(acc, lds, ra, a_voff, rb, b_voff, KT * TK, wave, lane, 2048u, 1024u, rs, rs, s_voff, wave * 2, wave * 2 + 1);
    } else {
        pair_loop<KIND_MXFP4, 4>(acc, lds, ra, a_voff, rb, b_voff, KT * TK, wave, lane, 2048u, 1024u, make_rsrc_uniform(sa, sa_bytes), make_rsrc_uniform(sb, sb_bytes),
                                 (uint32_t)wave * chunk_bytes + (uint32_t)lane * 4u, wave * 2, wave * 2 + 1, chunk_bytes);
    }

    if constexpr (STORE == STORE_ACC) {
        static_for<MR>([&](auto MI) {
            constexpr int mi = decltype(MI)::value;
            const int m = m0 + mi * 16 + li;
            if (m < p.M) {
                static_for<NR>([&](auto NI) {
                    constexpr int ni = decltype(NI)::value;
                    const int n = n0 + (wave * NR + ni) * 16 + lg * 4;
                    if (n < p.N) *reinterpret_cast<v4f*>(static_cast<float*>(p.c) + ((size_t)blockIdx.y * (size_t)p.M + (size_t)m) * (size_t)p.N + (size_t)n) = acc[mi][ni];
                });
            }
        });
    } else {
        // C through LDS, in halves: the stores of one are under way while the other is converted
        const __amdgpu_buffer_rsrc_t rc = make_rsrc(static_cast<uint16_t*>(p.c) + (size_t)m0 * (size_t)p.N, (uint64_t)(p.M - m0) * (uint64_t)p.N * 2ull);
        static_for<2>([&](auto HALF) {
            constexpr int half = decltype(HALF)::value;
            static_for<MR / 2>([&](auto MI) {
                constexpr int mi = half * (MR / 2) + decltype(MI)::value;
                static_for<NR>([&](auto NI) {
                    constexpr int ni = decltype(NI)::value;
                    const v4f x = acc[mi][ni];
                    *reinterpret_cast<v2i*>(pair_c_at(lds, mi, wave * NR + ni, li, lg)) = pack4_out16<OUT>(x[0], x[1], x[2], x[3]);
                });
            });
            __syncthreads();
            pair_store_rows(lds, half, rc, n0, p.N, tid);
        });
    }
}

template <int SCB>
void go(const A8W8Params& p, int store, dim3 grid, hipStream_t stream) {
    if (store == STORE_ACC) hipLaunchKernelGGL((k_mx_pair<STORE_ACC, OUT_BF16, SCB>), grid, dim3(256), 0, stream, p);
    else if (p.out == OUT_BF16) hipLaunchKernelGGL((k_mx_pair<STORE_C, OUT_BF16, SCB>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((k_mx_pair<STORE_C, OUT_FP16, SCB>), grid, dim3(256), 0, stream, p);
}

}  // namespace

// store: STORE_ACC (p.splits slices) or C in p.out
hipError_t psg_launch_mx_pair(const A8W8Params& p, int store, hipStream_t stream) {
    A8W8Params q = p;
    q.splits = store == STORE_ACC && p.splits > 1 ? p.splits : 1;
    const dim3 grid((unsigned)(((p.M + MxPair::TM - 1) / MxPair::TM) * ((p.N + MxPair::TN - 1) / MxPair::TN)), (unsigned)q.splits);
    if ((reinterpret_cast<uintptr_t>(p.mx_sa) | reinterpret_cast<uintptr_t>(p.mx_sb)) % 16 == 0) go<16>(q, store, grid, stream);
    else go<4>(q, store, grid, stream);
    return hipGetLastError();
}
