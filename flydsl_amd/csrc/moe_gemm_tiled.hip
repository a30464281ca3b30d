// MoE grouped GEMMs on 256-row tiles (gfx950): the mainloop of the 256x256 GEMM tile (gemm_tiled8.h) over two consecutive blocks
// of 128 sorted rows of one expert, for int8 and fp8 operands with one fp32 scale per row.
//
// Tile = 256 sorted rows x 256 weight rows (stage 1: the gate and the up rows of 128 columns, so that a wavefront holds both of
// its 16 columns and silu(g) * u happens in registers; stage 2: 256 output columns), eight wavefronts side by side along N, one
// workgroup per CU.  The A rows are gathered by the DMA itself: a lane's source address is its row's.  Everything about the
// pipeline (four LDS stages of A by DMA, W fragments one step ahead in registers, one barrier per step) is as in gemm_tiled8.h.
//
// Bound: MFMA, at the clock the power limit leaves (1.87 GHz in the loop, 2,490 cycles a K step of 2,048 issue cycles).  The tiles of
// k_moe_gemm (128 rows x 64 or 128 columns) are bound by their operand traffic: 128 flop per byte against 256 here.  Measured, 4096
// tokens x top-8 on 32 experts, 4096 x 1536, fp8: stage 1 473 -> 391 us, stage 2 (one row per sorted position) 360 -> 273; int8 528 ->
// 423 (loops of launches; under the profiler, on other boxes, 394 to 414 and 274 to 293).  Of the 56 us of a stage-1 tile 43 are the loop, 7 the epilogue and the rest its start.  The bits are those of k_moe_gemm.
// Registers: all 256 vector registers a lane are in use; 4 to 20 of them and about 40 scalar registers spill, none inside the unchecked
// loop (scratch stores between the loops and the epilogue, scalars into lanes of a vector register around the prologue).
//
// The tiles: blocks pair up from the start of each run of equal expert ids; the last block of an odd run is a tile of its own, for
// which only the lower eight 16-row blocks are multiplied.  How many tiles there are is only known on the device, so every
// workgroup scans the expert ids (64 a ballot), takes its tile in the XCD-aware order of the GEMM tiles over the real count, and
// leaves when its id is past that.
#include "gemm_tiled8.h"
#include "moe_rows.h"

namespace {

typedef __fp16 v2h_a __attribute__((ext_vector_type(2)));
typedef __bf16 v2b_a __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float silu(float g) { return g / (1.0f + __expf(-g)); }

template <int KIND, int STAGE>
__global__ void __launch_bounds__(512, 1) k_moe_tiled(MoeParams p) {
    using acc_t = typename Acc<KIND>::type;
    constexpr int MR = 16, NR = 2, WAVES = 8, NS = 4, NB = 2;
    constexpr int TM = 256, BLK = 128;
    constexpr int TN = STAGE == 1 ? 128 : 256;       // output columns
    constexpr int STG = TM * TK;                     // bytes of one A stage
    constexpr int A_DMA = STG / 1024 / WAVES;        // 1 KB blocks of a stage this wavefront fills
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NS * STG];
    __shared__ int ids[TM];
    __shared__ float s_sx[TM], s_rw[TM], s_sw[256];  // per row: scale of its x row, routing weight; per weight row of the tile: scale

    const int wave = wave_id();
    const int used = p.num_valid[0];

    // one pass for every list whose blocks are grouped by expert (the grid covers those); more only where runs are cut up
    for (int id = (int)blockIdx.x;; id += (int)gridDim.x) {
    // thread indices are derived afresh for every tile and again in its epilogue: kept alive through the mainloop, where no
    // register is free, they were spilled
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    const int tid = wave * 64 + lane, li = lane & 15, lg = lane >> 4;
    // ---- which tile: every wavefront for itself, 512 blocks a pass ----
    const int n_tiles = (p.n_out + TN - 1) / TN;
    int carry_id = -2, carry_par = 0, total = 0;
    uint64_t heads[8];
    auto scan = [&](int base, int (&v)[8]) __attribute__((always_inline)) {  // -> heads of blocks [base, base + 512)
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int b = base + c * 64 + lane;
            v[c] = b < p.blocks && b * BLK < used ? p.expert_ids[b] : -1;
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
            int prev = __shfl_up(v[c], 1);
            if (lane == 0) prev = carry_id;
            const uint64_t below = __ballot(v[c] != prev) & (~0ull >> (63 - lane));  // run starts up to this lane
            const int par = (below ? lane - (63 - __builtin_clzll(below)) : carry_par + lane) & 1;
            heads[c] = __ballot((unsigned)v[c] < (unsigned)p.experts && par == 0);
            carry_id = __builtin_amdgcn_readlane(v[c], 63);
            carry_par = (__builtin_amdgcn_readlane(par, 63) + 1) & 1;
        }
    };
    int ev[8];
    for (int base = 0; base < p.blocks; base += 512) {
        scan(base, ev);
#pragma unroll
        for (int c = 0; c < 8; c++) total += __builtin_popcountll(heads[c]);
    }
    if (id >= total * n_tiles) return;  // uniform
    int unit, n_tile;
    tile_coords(id, total, n_tiles, p.group_m, unit, n_tile);
    int blk = 0, e = 0;
    {
        int seen = 0;
        bool found = false;
        carry_id = -2, carry_par = 0;
        for (int base = 0; base < p.blocks && !found; base += 512) {
            if (p.blocks > 512) scan(base, ev);  // (up to 512 blocks the first pass's masks are still there)
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const int cnt = __builtin_popcountll(heads[c]);
                if (!found && unit < seen + cnt) {
                    const int rank = __builtin_popcountll(heads[c] & ((1ull << lane) - 1));
                    const int at = __builtin_ctzll(__ballot((heads[c] >> lane & 1) && rank == unit - seen));
                    blk = base + c * 64 + at;
                    e = __builtin_amdgcn_readlane(ev[c], at);
                    found = true;
                }
                seen += cnt;
            }
        }
    }
    blk = __builtin_amdgcn_readfirstlane(blk);
    e = __builtin_amdgcn_readfirstlane(e);

    const int n0 = n_tile * TN;
    const int K = p.K, KT = K >> 7;
    const int rows_e = STAGE == 1 ? 2 * p.n_out : p.n_out;
    const uint8_t* w_e = p.w + (uint64_t)e * (uint64_t)rows_e * (uint64_t)K;
    // one descriptor per 16-row weight block of the wavefront; a block past the width reads zeros
    auto w_rsrc = [&](int ni) {
        const int col = STAGE == 1 ? n0 + wave * 16 : n0 + (wave * NR + ni) * 16;
        const int row = STAGE == 1 ? col + ni * p.n_out : col;
        const bool in = col < p.n_out;
        return make_rsrc_uniform(w_e + (in ? (uint64_t)row * (uint64_t)K : 0), in ? 16ull * (uint64_t)K : 0);
    };
    const __amdgpu_buffer_rsrc_t rb0 = w_rsrc(0), rb1 = w_rsrc(1);
    const uint32_t b_lane_off = (uint32_t)lane * 16u;
    v4i blo[NB][NR], bhi[NB][NR];
    auto load_b1 = [&](int kt, int idx, v4i* lo, v4i* hi, auto CHK) __attribute__((always_inline)) {
        const int ni = idx >> 1;
        const bool has = !decltype(CHK)::value || kt < KT;
        const v4i v = buf_load16(ni ? rb1 : rb0, has ? b_lane_off : 0xFFFFFFF0u, has ? (uint32_t)kt * 2048u + (uint32_t)(idx & 1) * 1024u : 0u);
        if (idx & 1) hi[ni] = v; else lo[ni] = v;
    };

    // ---- the sorted rows of the tile ----
    const bool paired = blk + 1 < p.blocks && (blk + 1) * BLK < used && p.expert_ids[blk + 1] == e;  // uniform
    const int rows_live = paired ? TM : BLK;
    int my_id = p.tokens;  // padding
    if (tid < TM) {
        const int q = blk * BLK + tid;
        if (tid < rows_live && q < p.sorted_size) my_id = p.sorted_ids[q];
        ids[tid] = my_id;
    }
    // row of x (and of its scale) a sorted row reads, or -1 for a padding row
    auto x_row = [&](int id) {
        const int t = (int)((uint32_t)id & 0xFFFFFFu), s = (int)((uint32_t)id >> 24);
        if (t >= p.tokens || s >= p.topk) return -1;
        if constexpr (STAGE == 1) return p.x_slot_major ? s * p.tokens + t : t;
        return t * p.topk + s;
    };
    __syncthreads();
    const uint64_t rows_x = (STAGE == 1 && !p.x_slot_major) ? (uint64_t)p.tokens : (uint64_t)p.tokens * (uint64_t)p.topk;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc_uniform(p.x, rows_x * (uint64_t)K);
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    uint32_t a_voff[A_DMA];
#pragma unroll
    for (int j = 0; j < A_DMA; j++) {
        const int row = (wave * A_DMA + j) * 8 + (lane >> 3);
        const int xr = x_row(ids[row]);
        a_voff[j] = xr >= 0 ? (uint32_t)xr * (uint32_t)K + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16) : 0xFFFFFFF0u;
    }
    auto dma_a1 = [&](int kt, int stage, int j, auto CHK) __attribute__((always_inline)) {
        const uint32_t dst = lds_base + (uint32_t)(stage * STG + (wave * A_DMA + j) * 1024);
        const bool has = !decltype(CHK)::value || kt < KT;
        dma16(ra, dst, has ? a_voff[j] : 0xFFFFFFF0u, has ? (uint32_t)kt * TK : 0u);
    };

    acc_t acc[MR][NR];
#pragma unroll
    for (int mi = 0; mi < MR; mi++)
#pragma unroll
        for (int ni = 0; ni < NR; ni++) acc[mi][ni] = (acc_t){0, 0, 0, 0};

    const int f_lo = li * TK + ((lg ^ ((li >> 1) & 7)) << 4);
    const int f_hi = li * TK + (((4 + lg) ^ ((li >> 1) & 7)) << 4);
    auto read_frag = [&](int stage, int mi, v4i& flo, v4i& fhi) __attribute__((always_inline)) {
        flo = *reinterpret_cast<const v4i*>(&lds[stage * STG + mi * 16 * TK + f_lo]);
        fhi = *reinterpret_cast<const v4i*>(&lds[stage * STG + mi * 16 * TK + f_hi]);
    };
    constexpr int FRAG_AHEAD = 2, FRAG_BUFS = 4;
    v4i flo[FRAG_BUFS], fhi[FRAG_BUFS];

    // one K step over ML 16-row blocks (all sixteen, or the lower eight of a tile without a second block).  END: it may be the last one, so
    // the wait states between its last MFMA and the first ordinary read of an accumulator stand in the statement that ends it: behind
    // the loops the compiler may spill accumulators before it comes to any statement of ours (it stores up to 20 registers there)
    constexpr int N_W = 2 * NR;
    auto step = [&](int kt, auto SP, auto CHK, auto MLP, auto END) __attribute__((always_inline)) {
        constexpr int S = decltype(SP)::value, ML = decltype(MLP)::value;
        constexpr int SB = S % NB, SN = (SB + 1) % NB;
        constexpr int N_OPS = A_DMA + N_W, OPS_PER = (N_OPS + ML - 2) / (ML - 1);
        static_for<ML>([&](auto MI) {
            constexpr int mi = decltype(MI)::value;
            if constexpr (mi + FRAG_AHEAD < ML)
                read_frag(S, mi + FRAG_AHEAD, flo[(mi + FRAG_AHEAD) % FRAG_BUFS], fhi[(mi + FRAG_AHEAD) % FRAG_BUFS]);
            else
                read_frag((S + 1) % NS, mi + FRAG_AHEAD - ML, flo[(mi + FRAG_AHEAD) % FRAG_BUFS], fhi[(mi + FRAG_AHEAD) % FRAG_BUFS]);
            if constexpr (mi >= 1) {
                static_for<OPS_PER>([&](auto Q) {
                    constexpr int op = (mi - 1) * OPS_PER + decltype(Q)::value;
                    if constexpr (op < A_DMA) dma_a1(kt + NS - 1, (S + NS - 1) % NS, op, CHK);
                    else if constexpr (op < N_OPS) load_b1(kt + 1, op - A_DMA, blo[SN], bhi[SN], CHK);
                });
            }
            __builtin_amdgcn_sched_barrier(0);
            const v4i alo = flo[mi % FRAG_BUFS], ahi = fhi[mi % FRAG_BUFS];
            if constexpr (KIND == KIND_INT8) {
#pragma unroll
                for (int ni = 0; ni < NR; ni++) mfma_i8(acc[mi][ni], blo[SB][ni], alo);
#pragma unroll
                for (int ni = 0; ni < NR; ni++) mfma_i8(acc[mi][ni], bhi[SB][ni], ahi);
            } else {
                const v8i af = {alo[0], alo[1], alo[2], alo[3], ahi[0], ahi[1], ahi[2], ahi[3]};
#pragma unroll
                for (int ni = 0; ni < NR; ni++) {
                    const v8i bf = {blo[SB][ni][0], blo[SB][ni][1], blo[SB][ni][2], blo[SB][ni][3],
                                    bhi[SB][ni][0], bhi[SB][ni][1], bhi[SB][ni][2], bhi[SB][ni][3]};
                    mfma_f8(acc[mi][ni], bf, af);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (decltype(END)::value) asm volatile("s_nop 15\n\ts_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N_W + (NS - 3) * (A_DMA + N_W)) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N_W + (NS - 3) * (A_DMA + N_W)) : "memory");
    };

    // prologue: the epilogue's factors, A(0..2) by DMA, W(0)
    float ep_sx = 0.f, ep_rw = 1.f, ep_sw = 0.f;
    if (tid < TM) {
        const int xr = x_row(my_id);
        if (xr >= 0) {
            ep_sx = p.sx[xr];
            if (p.doweight) ep_rw = p.sorted_w[blk * BLK + tid];
        }
        const int col = n0 + (STAGE == 1 ? (tid & 127) : tid);
        if (col < p.n_out) ep_sw = p.sw[(size_t)e * rows_e + (STAGE == 1 && tid >= 128 ? p.n_out : 0) + col];
    }
#pragma unroll
    for (int s = 0; s < NS - 1; s++)
#pragma unroll
        for (int j = 0; j < A_DMA; j++) dma_a1(s, s, j, std::true_type{});
#pragma unroll
    for (int idx = 0; idx < N_W; idx++) load_b1(0, idx, blo[0], bhi[0], std::true_type{});
    if (tid < TM) {
        s_sx[tid] = ep_sx;
        s_rw[tid] = ep_rw;
        s_sw[tid] = ep_sw;
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N_W) : "memory");
    static_for<FRAG_AHEAD>([&](auto I) { read_frag(0, decltype(I)::value, flo[decltype(I)::value], fhi[decltype(I)::value]); });

    auto mainloop = [&](auto MLP) __attribute__((always_inline)) {
        int kt = 0;
        for (; kt + 2 * NS - 1 <= KT; kt += NS)
            static_for<NS>([&](auto I) { step(kt + decltype(I)::value, I, std::false_type{}, MLP, std::false_type{}); });
        for (; kt + NS <= KT; kt += NS)
            static_for<NS>([&](auto I) { step(kt + decltype(I)::value, I, std::true_type{}, MLP, std::bool_constant<decltype(I)::value == NS - 1>{}); });
        static_for<NS - 1>([&](auto I) {
            if (kt + decltype(I)::value < KT) step(kt + decltype(I)::value, I, std::true_type{}, MLP, std::true_type{});
        });
    };
    if (paired) mainloop(std::integral_constant<int, 16>{});
    else mainloop(std::integral_constant<int, 8>{});
    // every DMA still on its way must land before the stages are reused
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    // ---- epilogue: 16-bit rows through LDS (16-byte granules XOR-swizzled by the row), then out row by row ----
    int lane_e;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_e));
    const int tid_e = wave * 64 + lane_e, li_e = lane_e & 15, lg_e = lane_e >> 4;
    constexpr int ROWB = TN * 2, GR = ROWB / 16, RPP = 512 / GR;  // bytes and granules of a staged row, rows per store pass
    constexpr int NC = STAGE == 1 ? 1 : NR;                       // column blocks a wavefront puts out
    uint8_t* st_base[NC];
    v4f sw_v[NR];
#pragma unroll
    for (int ni = 0; ni < NC; ni++) st_base[ni] = lds + li_e * ROWB + (((((wave * NC + ni) * 2 + (lg_e >> 1)) ^ li_e) & (GR - 1)) << 4) + (lg_e & 1) * 8;
#pragma unroll
    for (int ni = 0; ni < NR; ni++) sw_v[ni] = *reinterpret_cast<const v4f*>(&s_sw[(STAGE == 1 ? ni * 128 + wave * 16 : (wave * NR + ni) * 16) + lg_e * 4]);
    const bool bf16 = p.out_dtype == OUT_BF16;
    const int g = tid_e & (GR - 1), r0 = tid_e / GR;
    const uint8_t* src = lds + r0 * ROWB + ((g ^ (r0 & 15)) << 4);
    const int n_st = n0 + g * 8;
    const bool atomic = STAGE == 2 && p.accumulate;
    static_for<2>([&](auto HALF) {
        constexpr int half = decltype(HALF)::value;
        if (half == 1 && !paired) return;  // uniform (out of this half, not of the kernel)
        static_for<MR / 2>([&](auto MI) {
            constexpr int mi = half * (MR / 2) + decltype(MI)::value;
            const float sx = s_sx[mi * 16 + li_e], rw = s_rw[mi * 16 + li_e];
            if constexpr (STAGE == 1) {
                v4f y;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float gt = ((float)acc[mi][0][v] * sx) * sw_v[0][v], up = ((float)acc[mi][1][v] * sx) * sw_v[1][v];
                    y[v] = silu(gt) * up * rw;
                }
                *reinterpret_cast<v2i*>(st_base[0] + mi * 16 * ROWB) = bf16 ? pack4_out16<OUT_BF16>(y[0], y[1], y[2], y[3]) : pack4_out16<OUT_FP16>(y[0], y[1], y[2], y[3]);
            } else {
                static_for<NR>([&](auto NI) {
                    constexpr int ni = decltype(NI)::value;
                    v4f y;
#pragma unroll
                    for (int v = 0; v < 4; v++) y[v] = (((float)acc[mi][ni][v] * sx) * sw_v[ni][v]) * rw;
                    *reinterpret_cast<v2i*>(st_base[ni < NC ? ni : 0] + mi * 16 * ROWB) = bf16 ? pack4_out16<OUT_BF16>(y[0], y[1], y[2], y[3]) : pack4_out16<OUT_FP16>(y[0], y[1], y[2], y[3]);
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
                    const size_t orow = STAGE == 2 && p.by_position ? (size_t)(blk * BLK + r) : (size_t)t * p.topk + s;
                    *reinterpret_cast<v4i*>(static_cast<uint16_t*>(p.out) + orow * (size_t)p.n_out + n_st) = *reinterpret_cast<const v4i*>(src + i * RPP * ROWB);
                }
            }
        } else {
            // packed additions: a wavefront covers 256 contiguous bytes of a row
            for (int q = half * (TM / 2) * (ROWB / 4) + tid_e; q < (half + 1) * (TM / 2) * (ROWB / 4); q += 512) {
                const int r = q / (ROWB / 4), cb = (q % (ROWB / 4)) * 4, n = n0 + (cb >> 1);
                const uint32_t id = (uint32_t)ids[r];
                const int t = (int)(id & 0xFFFFFFu), s = (int)(id >> 24);
                if (t < p.tokens && s < p.topk && n < p.n_out) {
                    const int bits = *reinterpret_cast<const int*>(lds + r * ROWB + ((((cb >> 4) ^ (r & 15)) & (GR - 1)) << 4) + (cb & 15));
                    uint16_t* o = static_cast<uint16_t*>(p.out) + (size_t)t * p.n_out + n;
                    if (bf16) __builtin_amdgcn_global_atomic_fadd_v2bf16((__attribute__((address_space(1))) v2b_a*)o, __builtin_bit_cast(v2b_a, bits));
                    else __builtin_amdgcn_global_atomic_fadd_v2f16((__attribute__((address_space(1))) v2h_a*)o, __builtin_bit_cast(v2h_a, bits));
                }
            }
        }
    });
    __syncthreads();  // the LDS is free for another tile
    }
}

template <int KIND, int STAGE>
hipError_t go(MoeParams p, const MoeRowsParams& rows, int blocks, hipStream_t stream) {
    constexpr int TN = STAGE == 1 ? 128 : 256;
    p.blocks = blocks;
    p.group_m = 8;
    if (p.by_position) {
        const hipError_t e = psg_launch_moe_rows_index(rows, stream);
        if (e != hipSuccess) return e;
    }
    // a list grouped by expert has at most one tile per two blocks and half a tile more per expert
    const long runs = (blocks + (long)p.experts + 1) / 2;
    const unsigned units = (unsigned)(runs < blocks ? runs : blocks);
    hipLaunchKernelGGL((k_moe_tiled<KIND, STAGE>), dim3(units * (unsigned)((p.n_out + TN - 1) / TN)), dim3(512), 0, stream, p);
    return hipGetLastError();
}

}  // namespace

hipError_t psg_launch_moe_tiled(const MoeParams& p, const MoeRowsParams& rows, int kind, int stage, int blocks, hipStream_t stream) {
    if (kind == KIND_INT8) return stage == 1 ? go<KIND_INT8, 1>(p, rows, blocks, stream) : go<KIND_INT8, 2>(p, rows, blocks, stream);
    return stage == 1 ? go<KIND_FP8, 1>(p, rows, blocks, stream) : go<KIND_FP8, 2>(p, rows, blocks, stream);
}
