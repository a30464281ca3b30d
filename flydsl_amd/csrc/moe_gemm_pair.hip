// MoE grouped GEMMs on 128x256 tiles, two workgroups per CU (mainloop: pair_loop.h), over blocks of 128 sorted rows of one expert, for int8 and fp8
// operands with one fp32 scale per row.
//
// Tile = one block x 256 weight rows: in stage 1 the gate and the up rows of 128 columns, so that a wavefront holds both and silu(g) * u happens in
// registers; in stage 2 256 output columns.  The A rows are gathered by the DMA itself: a lane's source address is its row's.
//
// Bound: MFMA, at the clock the power limit leaves.  The tiles of k_moe_gemm (128 rows x 64 or 128 columns) are bound by their operand traffic, 128 flop per
// byte against 171 here; 256-row tiles of two blocks, one workgroup a CU, move less (256 flop per byte) but have nothing beside a tile's start and end, which with the
// 12 K steps of stage 2 are a third of it, and leave half a tile empty where an expert has an odd number of blocks.  Measured, 4096 tokens x top-8 on 32
// experts, 4096 x 1536, fp8 (rocprofv3, 256-row tiles / these): stage 1 389 / 373 us, stage 2 261 / 254 and no launch for the rows' lists (8); the layer 798 / 739;
// 1024 tokens 300 / 268, 1500 x top-8 on 64 experts, 1280 x 1792 244 / 204.  The bits are those of k_moe_gemm.
#include "moe_rows.h"
#include "pair_loop.h"

namespace {

typedef __fp16 v2h_a __attribute__((ext_vector_type(2)));
typedef __bf16 v2b_a __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float silu(float g) { return g / (1.0f + __expf(-g)); }

template <int KIND, int STAGE>
__global__ void __launch_bounds__(256, 2) k_moe_pair(MoeParams p, MoeRowsParams rows) {
    using acc_t = typename Acc<KIND>::type;
    using P = Pair<KIND>;
    constexpr int MR = P::MR, NR = P::NR, TM = P::TM;
    constexpr int TN = STAGE == 1 ? 128 : 256;  // output columns
    __shared__ __attribute__((aligned(1024))) uint8_t lds[P::LDS_BYTES];
    __shared__ int ids[TM];
    __shared__ float s_sx[TM], s_rw[TM], s_sw[256];  // per row: scale of its x row, routing weight; per weight row of the tile: scale
    static_assert(P::fits(TM * 12 + 256 * 4), "two workgroups a CU");

    if constexpr (STAGE == 2) {
        if ((int)blockIdx.x < rows.wgs) {
            moe_rows_index_share<16>(rows, (int)blockIdx.x, rows.wgs, reinterpret_cast<int*>(lds), P::LDS_BYTES / 4);
            return;
        }
    }
    const int wg = (int)blockIdx.x - (STAGE == 2 ? rows.wgs : 0);
    const int used = p.num_valid[0];
    int units = used > 0 ? (used - 1) / TM + 1 : 0;
    units = units < p.blocks ? units : p.blocks;
    const int n_tiles = (p.n_out + TN - 1) / TN;
    if (wg >= units * n_tiles) return;
    int blk, n_tile;
    tile_coords(wg, units, n_tiles, 8, blk, n_tile);
    const int e = __builtin_amdgcn_readfirstlane(p.expert_ids[blk]);
    if ((unsigned)e >= (unsigned)p.experts) return;
    const int tid = threadIdx.x;
    const int wave = wave_id();
    const int lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int n0 = n_tile * TN;
    const int K = p.K;

    // row of x (and of its scale) a sorted row reads, or -1 for a padding row
    auto x_row = [&](int id) {
        const int t = (int)((uint32_t)id & 0xFFFFFFu), s = (int)((uint32_t)id >> 24);
        if (t >= p.tokens || s >= p.topk) return -1;
        if constexpr (STAGE == 1) return p.x_slot_major ? s * p.tokens + t : t;
        return t * p.topk + s;
    };
    const uint64_t rows_x = (STAGE == 1 && !p.x_slot_major) ? (uint64_t)p.tokens : (uint64_t)p.tokens * (uint64_t)p.topk;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc_uniform(p.x, rows_x * (uint64_t)K);
    uint32_t a_voff[4], b_voff[NR];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = (wave * 4 + j) * 8 + (lane >> 3), q = blk * TM + row;
        const int xr = x_row(q < p.sorted_size ? p.sorted_ids[q] : p.tokens);
        a_voff[j] = xr >= 0 ? (uint32_t)xr * (uint32_t)K + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16) : OOB;
    }
    // W: the wavefront's four 16-row blocks, in stage 1 two of gate and two of up rows; a block past the width reads zeros
    const int rows_e = STAGE == 1 ? 2 * p.n_out : p.n_out;
    const __amdgpu_buffer_rsrc_t rb = make_rsrc_uniform(p.w + (uint64_t)e * (uint64_t)rows_e * (uint64_t)K, (uint64_t)rows_e * (uint64_t)K);
#pragma unroll
    for (int ni = 0; ni < NR; ni++) {
        const int col = STAGE == 1 ? n0 + wave * 32 + (ni & 1) * 16 : n0 + (wave * NR + ni) * 16;
        const int row = STAGE == 1 && ni >= 2 ? p.n_out + col : col;
        b_voff[ni] = col < p.n_out ? (uint32_t)row * (uint32_t)K + (uint32_t)lane * 16u : OOB;
    }
    if (tid < TM) {
        const int q = blk * TM + tid, id = q < p.sorted_size ? p.sorted_ids[q] : p.tokens, xr = x_row(id);
        ids[tid] = id;
        s_sx[tid] = xr >= 0 ? p.sx[xr] : 0.f;
        s_rw[tid] = xr >= 0 && p.doweight ? p.sorted_w[q] : 1.f;
    }
    {
        const int col = n0 + (STAGE == 1 ? (tid & 127) : tid);
        s_sw[tid] = col < p.n_out ? p.sw[(size_t)e * rows_e + (STAGE == 1 && tid >= 128 ? p.n_out : 0) + col] : 0.f;
    }

    acc_t acc[MR][NR];
    pair_loop<KIND>(acc, lds, ra, a_voff, rb, b_voff, K, wave, lane, 2048u, 1024u, ra, ra);

    // ---- 16-bit rows through LDS (16-byte granules XORed with the row), in halves, then out row by row ----
    constexpr int ROWB = TN * 2, GR = ROWB / 16, RPP = 256 / GR;  // bytes and granules of a staged row, rows of a store pass
    v4f sw_v[NR];
#pragma unroll
    for (int ni = 0; ni < NR; ni++) sw_v[ni] = *reinterpret_cast<const v4f*>(&s_sw[(STAGE == 1 ? (ni >> 1) * 128 + wave * 32 + (ni & 1) * 16 : (wave * NR + ni) * 16) + lg * 4]);
    const bool bf16 = p.out_dtype == OUT_BF16, atomic = STAGE == 2 && p.accumulate;
    const int g = tid & (GR - 1), r0 = tid / GR, n_st = n0 + g * 8;
    auto put = [&](int r, int cb, v4f y) __attribute__((always_inline)) {  // four values of row r from byte cb on
        *reinterpret_cast<v2i*>(lds + r * ROWB + ((((cb >> 4) ^ r) & (GR - 1)) << 4) + (cb & 15)) = bf16 ? pack4_out16<OUT_BF16>(y[0], y[1], y[2], y[3]) : pack4_out16<OUT_FP16>(y[0], y[1], y[2], y[3]);
    };
    static_for<2>([&](auto HALF) {
        constexpr int half = decltype(HALF)::value;
        static_for<MR / 2>([&](auto MI) {
            constexpr int mi = half * (MR / 2) + decltype(MI)::value;
            const int r = mi * 16 + li;
            const float sx = s_sx[r], rw = s_rw[r];
            if constexpr (STAGE == 1) {
                static_for<2>([&](auto NI) {
                    constexpr int ni = decltype(NI)::value;
                    v4f y;
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const float gt = ((float)acc[mi][ni][v] * sx) * sw_v[ni][v], up = ((float)acc[mi][ni + 2][v] * sx) * sw_v[ni + 2][v];
                        y[v] = silu(gt) * up * rw;
                    }
                    put(r, (wave * 32 + ni * 16 + lg * 4) * 2, y);
                });
            } else {
                static_for<NR>([&](auto NI) {
                    constexpr int ni = decltype(NI)::value;
                    v4f y;
#pragma unroll
                    for (int v = 0; v < 4; v++) y[v] = (((float)acc[mi][ni][v] * sx) * sw_v[ni][v]) * rw;
                    put(r, ((wave * NR + ni) * 16 + lg * 4) * 2, y);
                });
            }
        });
        __syncthreads();
        if (!atomic) {
#pragma unroll
            for (int i = half * (TM / 2 / RPP); i < (half + 1) * (TM / 2 / RPP); i++) {
                const int r = r0 + i * RPP;
                const uint32_t id = (uint32_t)ids[r];
                const int t = (int)(id & 0xFFFFFFu), s = (int)(id >> 24);
                if (t < p.tokens && s < p.topk && n_st < p.n_out) {
                    const size_t orow = STAGE == 2 && p.by_position ? (size_t)(blk * TM + r) : (size_t)t * p.topk + s;
                    const v4i v = *reinterpret_cast<const v4i*>(lds + r * ROWB + (((g ^ r) & (GR - 1)) << 4));
                    v4i* o = reinterpret_cast<v4i*>(static_cast<uint16_t*>(p.out) + orow * (size_t)p.n_out + n_st);
                    if (STAGE == 2 && p.by_position) __builtin_nontemporal_store(v, o);  // read once, by k_moe_rows_add
                    else *o = v;
                }
            }
        } else {
            // packed additions: a wavefront covers 256 contiguous bytes of a row
            for (int q = half * (TM / 2) * (ROWB / 4) + tid; q < (half + 1) * (TM / 2) * (ROWB / 4); q += 256) {
                const int r = q / (ROWB / 4), cb = (q % (ROWB / 4)) * 4, n = n0 + (cb >> 1);
                const uint32_t id = (uint32_t)ids[r];
                const int t = (int)(id & 0xFFFFFFu), s = (int)(id >> 24);
                if (t < p.tokens && s < p.topk && n < p.n_out) {
                    const int bits = *reinterpret_cast<const int*>(lds + r * ROWB + ((((cb >> 4) ^ r) & (GR - 1)) << 4) + (cb & 15));
                    uint16_t* o = static_cast<uint16_t*>(p.out) + (size_t)t * p.n_out + n;
                    if (bf16) __builtin_amdgcn_global_atomic_fadd_v2bf16((__attribute__((address_space(1))) v2b_a*)o, __builtin_bit_cast(v2b_a, bits));
                    else __builtin_amdgcn_global_atomic_fadd_v2f16((__attribute__((address_space(1))) v2h_a*)o, __builtin_bit_cast(v2h_a, bits));
                }
            }
        }
    });
}

template <int KIND, int STAGE>
hipError_t go(MoeParams p, MoeRowsParams rows, int blocks, hipStream_t stream) {
    constexpr int TN = STAGE == 1 ? 128 : 256;
    p.blocks = blocks;
    rows.wgs = p.by_position ? ROWS_INDEX_WGS : 0;
    hipLaunchKernelGGL((k_moe_pair<KIND, STAGE>), dim3((unsigned)blocks * (unsigned)((p.n_out + TN - 1) / TN) + (unsigned)rows.wgs), dim3(256), 0, stream, p, rows);
    return hipGetLastError();
}

}  // namespace

hipError_t psg_launch_moe_pair(const MoeParams& p, const MoeRowsParams& rows, int kind, int stage, int blocks, hipStream_t stream) {
    if (kind == KIND_INT8) return stage == 1 ? go<KIND_INT8, 1>(p, rows, blocks, stream) : go<KIND_INT8, 2>(p, rows, blocks, stream);
    return stage == 1 ? go<KIND_FP8, 1>(p, rows, blocks, stream) : go<KIND_FP8, 2>(p, rows, blocks, stream);
}
