// MoE grouped GEMMs for gfx950 over expert-sorted token blocks, int8 or OCP fp8 operands with per-row fp32 scales, or int8
// activations against packed int4 weights (W4A8).
//
// The sorted row list (one entry per routed (token, slot), padded per expert to whole blocks of BM rows) says which
// row of x each tile row reads; one expert id per block says which slab of the preshuffled weights it multiplies.
//   stage 1 (gate-up): y[t, slot, n] = silu(g) * u with g = x[t] . W1[e, n], u = x[t] . W1[e, inter + n]
//   stage 2 (down):    y[n] = a2[t, slot] . W2[e, n] (* routing weight); added atomically into out[t] or written to
//                      out[t*topk + slot]
// Workgroup = four wavefronts side by side along N, tile BM x 64*NR, 128 bytes of K per step.  The A rows are
// gathered (per-row offsets through a bounds-checked buffer descriptor: padding rows read zeros) into a two-stage
// XOR-swizzled LDS tile; W fragments go straight from the expert's slab into MFMA operand registers (lane l reads
// bytes [16l, 16l+16) of a 1 KB block, the same wire format as the plain GEMM).  Stage 1 keeps two accumulators per
// fragment (gate and up) so silu(g)*u happens in registers.
// W4A8: the weights are the preshuffled int8 bytes with every 8 consecutive values v0..v7 packed into 4 bytes, byte j =
// (v_j & 15) | (v_{j+4} << 4) (tests/kernels/test_moe_gemm_2stage.py:64-80 of the reference), so a lane's 16-byte piece
// of a fragment is 8 bytes at half the offset; it is unpacked with the reference's sign-extending mask-and-multiply
// (kernels/common/mma/mfma_preshuffle_pipeline.py:225-238) into the same int8 fragment and multiplied by the int8 MFMA.
#include "moe_blocks.h"
#include "moe_rows.h"
#include "psg_common.h"

namespace {

typedef __fp16 v2h __attribute__((ext_vector_type(2)));
typedef __bf16 v2b __attribute__((ext_vector_type(2)));

template <int KIND>
struct MoeAcc {
    using type = v4f;
};
template <>
struct MoeAcc<KIND_INT8> {
    using type = v4i;
};
template <>
struct MoeAcc<KIND_INT8W4> {
    using type = v4i;
};

// 8 packed int4 (one dword) -> two dwords of int8: the low nibbles of the four bytes, then the high nibbles
__device__ __forceinline__ void unpack_int4(int packed, int& even, int& odd) {
    even = (packed & 0x0F0F0F0F) | ((packed & 0x08080808) * 0x1E);
    const int t = (int)((unsigned)packed >> 4);
    odd = (t & 0x0F0F0F0F) | ((t & 0x08080808) * 0x1E);
}
__device__ __forceinline__ v4i unpack_int4x16(v2i packed) {
    int e0, o0, e1, o1;
    unpack_int4(packed[0], e0, o0);
    unpack_int4(packed[1], e1, o1);
    return (v4i){e0, o0, e1, o1};
}

__device__ __forceinline__ int moe_lds_off(int row, int kc) { return row * 128 + ((kc ^ ((row >> 1) & 7)) << 4); }

__device__ __forceinline__ float silu(float g) { return g / (1.0f + __expf(-g)); }

// CO = 2: the workgroup's BM rows are TWO consecutive blocks of the sorted list when both belong to the same expert (blocks
// of 16 or 32 rows: an expert with 17 to 32 routed rows would otherwise stream its weights once per block).  Blocks pair up
// from the start of each run of equal expert ids: the workgroup of the second block of a pair ends at once, and the
// first one treats the second half of its tile as padding when the run ends there.
// AHEAD: 0 = operands a step ahead; 1 = three steps (the rule and its figures: takes_deep; a stage by rows never, having more workgroups than that); 2 = three steps,
// and W past the caches where a tile is the only one to read it (takes_nt, moe_reads_once).
// ROWS = MoeRowsParams: the down stage by rows, whose first `rows.wgs` rows of the grid make the lists of the tokens' rows.  A build of
// its own: the decode layers, which add directly, lost 0.4 to 0.8 us of 55 to 140 to the longer arguments and the branch.
template <int KIND, int MR, int NR, int STAGE, int CO, int AHEAD, class... ROWS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(AHEAD != 2 || KIND == KIND_INT8W4 ? 1 : MR <= 2 ? 4 : 3))) k_moe_gemm(MoeParams p, ROWS... rows) {
    using acc_t = typename MoeAcc<KIND>::type;
    constexpr int BM = 16 * MR, TN = 64 * NR;
    constexpr int BLK = BM / CO;                        // rows of one block of the sorted list
    constexpr int NSET = STAGE == 1 ? 2 : 1;           // gate and up
    constexpr int A_LOADS = (BM * 8 + 255) / 256;      // 16-byte chunks of the A tile per thread
    constexpr bool W4 = KIND == KIND_INT8W4;           // packed int4 weights
    constexpr int WSH = W4 ? 1 : 0;                    // weight byte offsets are halved
    constexpr bool DEEP = AHEAD != 0;
    __shared__ __attribute__((aligned(16))) uint8_t lds[2][BM * 128];
    __shared__ int ids[BM];
    __shared__ float s_sx[BM], s_rw[BM];  // per tile row: scale of its x row and routing weight, fetched before the K loop

    const int tid = threadIdx.x;
    const int wave = wave_id();
    const int lane = tid & 63, li = lane & 15, lg = lane >> 4;
    int blk = (int)blockIdx.y;
    if constexpr (sizeof...(ROWS) == 1) {
        const MoeRowsParams& r = (rows, ...);
        if (blk < r.wgs) {
            moe_rows_index_share<4>(r, (int)(blockIdx.y * gridDim.x + blockIdx.x), r.wgs * (int)gridDim.x, reinterpret_cast<int*>(lds), BM * 64);
            return;
        }
        blk -= r.wgs;
    }
    const int n0 = (int)blockIdx.x * TN;
    const int used = p.num_valid[0];
    // what is looked at of the list's experts, in one go
    MoeNeighbours around;
    int back = 0;  // of block blk - 1 - lane (not in the builds that look at nothing else: it takes four of their registers, and the pairs of 16 a wavefront)
    if constexpr (AHEAD == 2) around = moe_neighbours(p.expert_ids, (int)gridDim.y, blk, CO, lane);
    if constexpr (CO == 2 && AHEAD == 2) back = p.expert_ids[blk - 1 - lane > 0 ? blk - 1 - lane : 0];
    auto sorted_row = [&]() { return tid < BM && blk * BLK + tid < p.sorted_size ? p.sorted_ids[blk * BLK + tid] : p.tokens; };  // past the list = a padding row
    int my_id = 0;
    if constexpr (AHEAD == 2) my_id = sorted_row();
    if (blk * BLK >= used) return;                     // uniform: blocks past the sorted rows in use
    const int e = p.expert_ids[blk];
    if (e < 0 || e >= p.experts) return;               // uniform: a block without an expert
    int rows_live = BLK;                               // rows of the tile that belong to this workgroup's expert
    if constexpr (CO == 2) {
        // position of this block in its run of equal expert ids: 64 earlier ids at a time, one per lane
        int before = 0;
        for (int base = blk - 1; base >= 0; base -= 64) {
            const int j = base - lane;
            const int v = AHEAD == 2 && base == blk - 1 ? back : p.expert_ids[j > 0 ? j : 0];
            const unsigned long long same = __ballot(j >= 0 && v == e);
            const int run = same == ~0ull ? 64 : __builtin_ctzll(~same);
            before += run;
            if (run < 64) break;
        }
        before = __builtin_amdgcn_readfirstlane(before);
        if (before & 1) return;                        // uniform: the second block of a pair
        if (blk + 1 < (int)gridDim.y && (blk + 1) * BLK < used && p.expert_ids[blk + 1] == e) rows_live = BM;  // (gridDim.y = entries of expert_ids)
    }

    const int K = p.K, KT = K >> 7;
    const int rows_x = (STAGE == 1 && !p.x_slot_major) ? p.tokens : p.tokens * p.topk;
    const int rows_e = STAGE == 1 ? 2 * p.n_out : p.n_out;            // weight rows per expert
    __amdgpu_buffer_rsrc_t ra = make_rsrc(p.x, (uint64_t)rows_x * (uint64_t)K);
    const uint8_t* w_e = p.w + (((uint64_t)e * (uint64_t)rows_e * (uint64_t)K) >> WSH);
    __amdgpu_buffer_rsrc_t rb = make_rsrc(w_e, ((uint64_t)rows_e * (uint64_t)K) >> WSH);

    // n-blocks of this wavefront inside the expert's slab: set 0 = gate (or the only set), set 1 = up
    uint32_t b_voff[NSET][NR];
#pragma unroll
    for (int s = 0; s < NSET; s++)
#pragma unroll
        for (int ni = 0; ni < NR; ni++) {
            const int n = n0 + (ni * 4 + wave) * 16;                  // first column of the block: the four wavefronts of pass ni
                                                                      // cover 64 consecutive columns
            const int nb = (n + s * p.n_out) >> 4;
            b_voff[s][ni] = n < p.n_out ? ((uint32_t)nb * 16u * (uint32_t)K + (uint32_t)lane * 16u) >> WSH : OOB;
        }

    uint32_t a_voff[A_LOADS];
    int a_ldsoff[A_LOADS];
    constexpr int NAS = DEEP ? 4 : 1;  // register sets of the A tile on its way to LDS
    v4i areg[NAS][A_LOADS];
    auto load_a = [&](int kt, int set) {
#pragma unroll
        for (int j = 0; j < A_LOADS; j++) {
            const bool ok = kt < KT;
            areg[set][j] = buf_load16(ra, ok ? a_voff[j] : OOB, ok ? (uint32_t)kt * 128u : 0u);
        }
    };
    auto store_a = [&](int stage, int set) {
#pragma unroll
        for (int j = 0; j < A_LOADS; j++)
            if (a_ldsoff[j] >= 0) *reinterpret_cast<v4i*>(&lds[stage][a_ldsoff[j]]) = areg[set][j];
    };
    using wreg_t = typename std::conditional<W4, v2i, v4i>::type;  // a lane's piece of a W fragment as it is loaded
    // W register sets: the fragments of step kt live in set kt % NWS and are requested WPF steps ahead; loads return in order, so A has to be as far ahead as W.
    constexpr int WPF = DEEP ? 3 : 1;
    constexpr int NWS = WPF + 1;
    wreg_t blo[NWS][NSET][NR], bhi[NWS][NSET][NR];
    __builtin_assume(KT > 0);  // (otherwise the first loads stand behind branches)
    auto load_b = [&](int kt, int set, auto NTP) __attribute__((always_inline)) {
        constexpr int POLICY = decltype(NTP)::value ? 2 : 0;  // non-temporal or none
        auto w8 = [&](uint32_t voff, uint32_t soff) { return (v2i)__builtin_amdgcn_raw_buffer_load_b64(rb, (int)voff, (int)soff, POLICY); };
        auto w16 = [&](uint32_t voff, uint32_t soff) { return (v4i)__builtin_amdgcn_raw_buffer_load_b128(rb, (int)voff, (int)soff, POLICY); };
#pragma unroll
        for (int s = 0; s < NSET; s++)
#pragma unroll
            for (int ni = 0; ni < NR; ni++) {
                const bool ok = kt < KT;
                if constexpr (W4) {
                    blo[set][s][ni] = w8(ok ? b_voff[s][ni] : OOB, ok ? (uint32_t)kt * 1024u : 0u);
                    bhi[set][s][ni] = w8(ok ? b_voff[s][ni] + 512u : OOB, ok ? (uint32_t)kt * 1024u : 0u);
                } else {
                    blo[set][s][ni] = w16(ok ? b_voff[s][ni] : OOB, ok ? (uint32_t)kt * 2048u : 0u);
                    bhi[set][s][ni] = w16(ok ? b_voff[s][ni] + 1024u : OOB, ok ? (uint32_t)kt * 2048u : 0u);
                }
            }
    };

    // the weight scales of the lane's columns (pass ni: columns ni*64 + wave*16 + lg*4 + 0..3), also ahead of the K loop
    v4f swa_[NR], swb_[STAGE == 1 ? NR : 1];
#pragma unroll
    for (int ni = 0; ni < NR; ni++) {
        const int ncol = n0 + ni * 64 + wave * 16 + lg * 4;
        const bool in = ncol < p.n_out;
        swa_[ni] = in ? *reinterpret_cast<const v4f*>(p.sw + (size_t)e * rows_e + ncol) : (v4f){0.f, 0.f, 0.f, 0.f};
        if constexpr (STAGE == 1) swb_[ni] = in ? *reinterpret_cast<const v4f*>(p.sw + (size_t)e * rows_e + p.n_out + ncol) : (v4f){0.f, 0.f, 0.f, 0.f};
    }

    acc_t acc[MR][NSET][NR];
#pragma unroll
    for (int mi = 0; mi < MR; mi++)
#pragma unroll
        for (int s = 0; s < NSET; s++)
#pragma unroll
            for (int ni = 0; ni < NR; ni++) acc[mi][s][ni] = (acc_t){0, 0, 0, 0};

    auto step = [&](int kt, auto SP, auto WP, auto NTP) __attribute__((always_inline)) {
        constexpr int S = decltype(SP)::value;    // LDS stage of this step's A tile
        constexpr int WS = decltype(WP)::value;   // register set of this step's W fragments
        load_a(kt + (DEEP ? 3 : 1), DEEP ? (WS + 3) % NAS : 0);
        load_b(kt + WPF, (WS + WPF) % NWS, NTP);
        // packed int4: this step's fragments unpacked once, in front of the row blocks that share them
        v4i ulo[W4 ? NSET : 1][W4 ? NR : 1], uhi[W4 ? NSET : 1][W4 ? NR : 1];
        if constexpr (W4) {
#pragma unroll
            for (int s = 0; s < NSET; s++)
#pragma unroll
                for (int ni = 0; ni < NR; ni++) {
                    ulo[s][ni] = unpack_int4x16(blo[WS][s][ni]);
                    uhi[s][ni] = unpack_int4x16(bhi[WS][s][ni]);
                }
        }
        static_for<MR>([&](auto MI) {
            constexpr int mi = decltype(MI)::value;
            const int row = mi * 16 + li;
            const v4i alo = *reinterpret_cast<const v4i*>(&lds[S][moe_lds_off(row, lg)]);
            const v4i ahi = *reinterpret_cast<const v4i*>(&lds[S][moe_lds_off(row, 4 + lg)]);
            static_for<NSET>([&](auto SI) {
                constexpr int s = decltype(SI)::value;
                static_for<NR>([&](auto NI) {
                    constexpr int ni = decltype(NI)::value;
                    if constexpr (W4) {
                        acc[mi][s][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ulo[s][ni], alo, acc[mi][s][ni], 0, 0, 0);
                        acc[mi][s][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(uhi[s][ni], ahi, acc[mi][s][ni], 0, 0, 0);
                    } else if constexpr (KIND == KIND_INT8) {
                        acc[mi][s][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(blo[WS][s][ni], alo, acc[mi][s][ni], 0, 0, 0);
                        acc[mi][s][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bhi[WS][s][ni], ahi, acc[mi][s][ni], 0, 0, 0);
                    } else {
                        const v8i w8 = __builtin_shufflevector(blo[WS][s][ni], bhi[WS][s][ni], 0, 1, 2, 3, 4, 5, 6, 7);
                        const v8i a8 = __builtin_shufflevector(alo, ahi, 0, 1, 2, 3, 4, 5, 6, 7);
                        acc[mi][s][ni] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w8, a8, acc[mi][s][ni], 0, 0, 0, 0, 0, 0);
                    }
                });
            });
        });
        store_a(S ^ 1, DEEP ? (WS + 1) % NAS : 0);
        __syncthreads();
    };

    // the product, W past the caches (NTP) or through them
    auto product = [&](auto NTP) __attribute__((always_inline)) {
        // W first: its addresses need only the expert, so these requests are in flight while the sorted row list is fetched (which is here already where W waited for the
        // experts of the list)
        static_for<WPF>([&](auto I) { load_b(decltype(I)::value, decltype(I)::value, NTP); });
        if constexpr (AHEAD != 2) my_id = sorted_row();
        if (tid < BM) ids[tid] = tid < rows_live ? my_id : p.tokens;  // past the pair = a padding row
        __syncthreads();

        // row of x (and of its scale) a tile row reads, or -1 for a padding row
        auto x_row = [&](int r) {
            const uint32_t sid = (uint32_t)ids[r];
            const int t = (int)(sid & 0xFFFFFFu), s = (int)(sid >> 24);
            if (t >= p.tokens || s >= p.topk) return -1;
            if constexpr (STAGE == 1) return p.x_slot_major ? s * p.tokens + t : t;
            return t * p.topk + s;
        };
        // the epilogue's per-row factors now, so that their memory latency runs under the K loop (whose barriers also make them
        // visible to every wavefront)
        if (tid < BM) {
            const int xr = x_row(tid);
            s_sx[tid] = xr >= 0 ? p.sx[xr] : 0.f;
            s_rw[tid] = (p.doweight && xr >= 0) ? p.sorted_w[blk * BLK + tid] : 1.0f;
        }

#pragma unroll
        for (int j = 0; j < A_LOADS; j++) {
            const int c = tid + 256 * j, row = c >> 3, kc = c & 7;
            const int xr = row < BM ? x_row(row) : -1;
            a_voff[j] = xr >= 0 ? (uint32_t)xr * (uint32_t)K + (uint32_t)kc * 16u : OOB;
            a_ldsoff[j] = row < BM ? moe_lds_off(row, kc) : -1;
        }
        static_for<DEEP ? 3 : 1>([&](auto I) { load_a(decltype(I)::value, decltype(I)::value); });
        store_a(0, 0);
        __syncthreads();
        // unrolled over lcm(2 LDS stages, NWS register sets) steps so that both indices are compile-time
        constexpr int UN = NWS % 2 == 0 ? NWS : 2 * NWS;
        int kt0 = 0;
        if constexpr (DEEP)  // whole rounds without a condition: the compiler's count of the loads on their way is then exact
            for (; kt0 + UN <= KT; kt0 += UN)
                static_for<UN>([&](auto I) { step(kt0 + decltype(I)::value, std::integral_constant<int, decltype(I)::value & 1>{}, std::integral_constant<int, decltype(I)::value % NWS>{}, NTP); });
        for (; kt0 < KT; kt0 += UN) {
            static_for<UN>([&](auto I) {
                constexpr int i = decltype(I)::value;
                if (kt0 + i < KT) step(kt0 + i, std::integral_constant<int, i & 1>{}, std::integral_constant<int, i % NWS>{}, NTP);
            });
        }
    };
    if constexpr (AHEAD == 2) {
        const int n = (used + BLK - 1) / BLK;
        if (moe_reads_once(around, p.expert_ids, n < (int)gridDim.y ? n : (int)gridDim.y, blk, CO, e, p.experts, p.cached, lane)) product(std::true_type{});
        else product(std::false_type{});
    } else {
        product(std::false_type{});
    }

    // Epilogue, one pass per ni (64 consecutive columns of the tile): every lane finishes its own fragments (rows
    // mi*16 + li, columns ni*64 + wave*16 + lg*4 + 0..3) into an LDS tile of BM rows (free after the loop's last
    // barrier; 16-byte granules XOR-swizzled by the row), then the workgroup walks the tile row by row so that one
    // store or atomic instruction covers whole 128- or 256-byte rows of the output instead of 16 rows x 16 bytes.
    const bool f32_out = p.out_dtype == OUT_F32;
    const int esize = f32_out ? 4 : 2;
    const int row_bytes = 64 * esize;                  // one pass's row in LDS: 128 or 256 bytes (both stages hold BM*256)
    const int gmask = (row_bytes >> 4) - 1;            // granules per row - 1 (7 or 15)
    uint8_t* stage = &lds[0][0];
    static_for<NR>([&](auto NI) {
        constexpr int ni = decltype(NI)::value;
        const int ncol = n0 + ni * 64 + wave * 16 + lg * 4;   // first of the lane's four columns
        const v4f swa = swa_[ni], swb = swb_[STAGE == 1 ? ni : 0];
        static_for<MR>([&](auto MI) {
            constexpr int mi = decltype(MI)::value;
            const int r = mi * 16 + li;
            const float sx = s_sx[r];
            const float rw = s_rw[r];
            v4f y;
            if constexpr (STAGE == 1) {
                const acc_t ag = acc[mi][0][ni], au = acc[mi][NSET - 1][ni];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float g = ((float)ag[v] * sx) * swa[v], u = ((float)au[v] * sx) * swb[v];
                    y[v] = silu(g) * u * rw;
                }
            } else {
                const acc_t a = acc[mi][0][ni];
#pragma unroll
                for (int v = 0; v < 4; v++) y[v] = (((float)a[v] * sx) * swa[v]) * rw;
            }
            const int cb = (wave * 16 + lg * 4) * esize;      // byte column inside the pass's row
            uint8_t* dst = stage + r * row_bytes + ((((cb >> 4) ^ r) & gmask) << 4) + (cb & 15);
            if (f32_out) {
                *reinterpret_cast<v4f*>(dst) = y;
            } else {
                *reinterpret_cast<v2i*>(dst) = p.out_dtype == OUT_BF16 ? pack4_out16<OUT_BF16>(y[0], y[1], y[2], y[3]) : pack4_out16<OUT_FP16>(y[0], y[1], y[2], y[3]);
            }
        });
        __syncthreads();
        const bool atomic = STAGE == 2 && p.accumulate;
        // trips of the workgroup over the pass, 4 or 16 bytes a thread; four of them together (two on larger tiles, whose builds it would cost a wavefront a SIMD), so that their row ids and values come out of LDS side by side
        // (and shifts instead of a division for every unit, the units of a row being a power of two known at build time; layers, us before / now: fp8 64 tokens x top-8 on 32 experts, 4096 x 1536, 120.7 / 119.8, 98 x top-4 on 8, 1280 x
        // 1024, 31.3 / 29.1, 433 x top-2 on 16, 4096 x 1792, 103.0 / 100.7; int8 226 x top-4 on 32, 1280 x 768, 45.2 / 44.1; int4 2000 x top-8, 4096 x 1536, 475 / 470)
        auto walk = [&](auto SH, auto&& put) __attribute__((always_inline)) {
            constexpr int sh = decltype(SH)::value, TRIPS = ((BM << sh) + 255) / 256;  // log2 of the units of a row
            const int unit_sh = (f32_out ? 8 : 7) - sh, cb = (tid & ((1 << sh) - 1)) << unit_sh, n = n0 + ni * 64 + (cb >> (f32_out ? 2 : 1));
            constexpr int MOST = MR <= 2 ? 4 : 2;
            static_for<(TRIPS + MOST - 1) / MOST>([&](auto I) {
                constexpr int at = decltype(I)::value * MOST, B = TRIPS - at < MOST ? TRIPS - at : MOST;
                uint32_t sid[B];
                const uint8_t* src[B];
#pragma unroll
                for (int j = 0; j < B; j++) {
                    const int r = (tid >> sh) + ((at + j) * 256 >> sh);
                    sid[j] = r < BM ? (uint32_t)ids[r] : 0xFFFFFFu;
                    src[j] = stage + r * row_bytes + ((((cb >> 4) ^ r) & gmask) << 4) + (cb & 15);
                }
                put(sid, src, n, at, std::integral_constant<int, B>{});
            });
        };
        auto live = [&](uint32_t sid, int n) { return (int)(sid & 0xFFFFFFu) < p.tokens && (int)(sid >> 24) < p.topk && n < p.n_out; };
        if (!atomic) {
            walk(std::integral_constant<int, 3>{}, [&](const auto& sid, const auto& src, int n, int at, auto B) __attribute__((always_inline)) {
                v4i v[decltype(B)::value];
#pragma unroll
                for (int j = 0; j < decltype(B)::value; j++) v[j] = *reinterpret_cast<const v4i*>(src[j]);
#pragma unroll
                for (int j = 0; j < decltype(B)::value; j++) {
                    const size_t t = sid[j] & 0xFFFFFFu, orow = p.by_position ? (size_t)(blk * BLK + (tid >> 3) + (at + j) * 32) : t * p.topk + (sid[j] >> 24);
                    if (live(sid[j], n)) *reinterpret_cast<v4i*>(static_cast<uint16_t*>(p.out) + orow * (size_t)p.n_out + n) = v[j];
                }
            });
        } else if (f32_out) {
            walk(std::integral_constant<int, 6>{}, [&](const auto& sid, const auto& src, int n, int, auto B) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < decltype(B)::value; j++)
                    if (live(sid[j], n)) unsafeAtomicAdd(static_cast<float*>(p.out) + (size_t)(sid[j] & 0xFFFFFFu) * (size_t)p.n_out + n, *reinterpret_cast<const float*>(src[j]));
            });
        } else {
            walk(std::integral_constant<int, 5>{}, [&](const auto& sid, const auto& src, int n, int, auto B) __attribute__((always_inline)) {
                int v[decltype(B)::value];
#pragma unroll
                for (int j = 0; j < decltype(B)::value; j++) v[j] = *reinterpret_cast<const int*>(src[j]);
#pragma unroll
                for (int j = 0; j < decltype(B)::value; j++) {
                    if (!live(sid[j], n)) continue;
                    uint16_t* o = static_cast<uint16_t*>(p.out) + (size_t)(sid[j] & 0xFFFFFFu) * (size_t)p.n_out + n;
                    if (p.out_dtype == OUT_FP16) __builtin_amdgcn_global_atomic_fadd_v2f16((__attribute__((address_space(1))) v2h*)o, __builtin_bit_cast(v2h, v[j]));
                    else __builtin_amdgcn_global_atomic_fadd_v2bf16((__attribute__((address_space(1))) v2b*)o, __builtin_bit_cast(v2b, v[j]));
                }
            });
        }
        if constexpr (ni + 1 < NR) __syncthreads();
    });
}

// Whether a stage takes the build that asks for its operands three steps ahead (the builds that read W past the caches and those on two paired blocks always do).  Tiles of up to 32
// rows are bound by the bytes of W on their way, and it gains (us, 32 experts, 4096 x 1536, one step ahead / three: 8 tokens x top-8 fp8 stage 1 66.6 / 64.9, there with W alone
// ahead before, stage 2 36.1 / 33.3, int4 42.2 / 35.6 and 23.1 / 21.7; 4 x top-2 on 8, 4096 x 2048, fp8 30.5 / 21.8 and 16.9 / 13.4, int4 25.1 / 15.8 and 13.5 / 9.7) but in stage 2 with
// more than 11 workgroups a CU (128 experts, 2048 x 768, 600 x top-8 in blocks of 32 51.6 / 56.6; 2048 x 512, 384 in blocks of 16 36.9 / 38.5) and with int4 weights in blocks of 16 with more
// than four in stage 1, three in stage 2 (64 tokens 46.8 / 46.9 and 26.8 / 29.1, 200 x top-8 on 128, 2048 x 512 29.9 / 31.2 and 22.6 / 23.9).  On 64- and 128-row tiles: with few workgroups on a CU nothing else
// covers a load: up to two of them per CU that build is the faster one in either stage.  With more of them stage 2 is better off with the
// registers of more workgroups (683 to 1,891 workgroups), stage 1 only where the rows are short.  Workgroups on average over routings.  Measured,
// us one step ahead / three: stage 1, 1086 tokens x top-4 on 17 experts, 4096 x 256 (170 workgroups of 128 rows) fp8 41.4 / 26.8, int4 47.6 / 29.6; 813 x
// top-4 on 32, 4096 x 512 (331) 49.8 / 34.3; 600 x top-1 on 8, 3072 x 768, 64 rows (160) 23.9 / 17.6; 1024 x top-8, 4096 x 1536 (1,920) fp8 170 / 156, int8
// 190 / 164, int4 161 / 143; 400 x top-6, 4096 x 1536, 64 rows (1,284) 96.7 / 93.1; but 1052 x top-8, 1536 x 1024 (1,180) fp8 43.3 / 45.2, 1726 x top-2,
// 2816 x 512, 64 rows (688) 39.3 / 40.9.  Stage 2: 339 x top-4 on 16, 1024 x 2048 (234) 19.9 / 15.7; 200 x top-2 on 8, 4096 x 2048 (328) 26.8 / 20.9; but
// 1086 x top-4, 4096 x 256 (1,358) 24.0 / 29.6.  Two blocks of 32 rows in one tile (stage 1) have that build alone: of 54 layers of 8 to 128 experts, 72 to 3,108 such workgroups,
// 50 are faster with it, weights in memory or in the last-level cache (int8 45 x top-6 on 8, 3072 x 768 28.7 / 17.8, fp8 100 x top-2 on 8, 4096 x 2048 36.9 / 30.7, 564 x
// top-6 on 128, 1280 x 768 58.9 / 55.3), and four 1 to 6 % slower (150 x top-4 on 16, 4096 x 2048 59.4 / 60.6; from the cache 49.8 / 52.8).
template <int KIND, int STAGE>
bool takes_deep(const MoeParams& p, int block_m, int blocks, int nx) {
    const long pairs = (long)p.tokens * p.topk, likely = pairs / block_m + p.experts / 2;
    const long wgs = (likely < blocks ? likely : blocks) * nx;
    if (wgs <= 2L * psg_cu_count()) return true;
    if (block_m <= 32) return KIND == KIND_INT8W4 ? block_m == 32 || wgs <= (STAGE == 1 ? 4L : 3L) * psg_cu_count() : STAGE == 1 || wgs <= 11L * psg_cu_count();
    if (STAGE == 2) return false;
    return p.K >= 4096 || (block_m == 128 && (p.K >= 2048 || KIND == KIND_INT8W4));
}

// Whether a stage on tiles of up to 32 rows, or on two paired blocks of 32, reads W past the caches (non-temporal): where an expert's rows mostly make one tile, so that nothing
// is read twice, and the weights of both stages together are more than the last-level cache holds (256 MB).  Streamed like this they come at 5.5 to 6.6 TB/s
// instead of 5.0 to 6.0, us plain / non-temporal, weights in memory: stage 1, 32 experts, 4096 x 1536, fp8 8 tokens x top-8 64.9 / 59.2, 64 75.3 / 67.9, 96 75.8 /
// 68.5; blocks of 32 110 80.7 / 73.0, 192 80.3 / 73.1; int4 8 tokens 35.6 / 32.7; 64 experts, 2048 x 768, 128 x top-4 39.1 / 35.9.  Stage 2 8 tokens 33.3 / 30.5, 128 x top-4 23.4 /
// 21.3, but 96 x top-8 in blocks of 16 (one and a half tiles an expert) 45.6 / 50.9, 100 x top-6 on 16, 3072 x 512 11.6 / 12.3.  The
// cache keeps nothing that was read like this: a layer of 226 MB (128 experts, 2304 x 256, 160 x top-8) took 73.7 / 69.4 from memory, 60.8 / 68.9 from the cache.
// That is the rule for the routings that a call can have; which tiles of its own do is for the workgroups to say (moe_reads_once), because a router that prefers some experts leaves the others'
// weights unread, so that what is read fits the cache, and gives the busy ones several tiles.  Layers, us through the caches / past them everywhere / as it is, weights in memory; in the
// cache, expert preferences N(0, 4^2) beside N(0, 1) logits, 32 experts, 4096 x 1536, top-8, fp8: 64 tokens 94.8 / 96.8 / 89.5; 70.9 / 92.9 / 69.3, 96 98.4 / 102.8 / 91.2; 80.6 / 101.5 / 76.1,
// int4 64 74.0 / 72.5 / 70.6; 58.1 / 69.6 / 56.6; 64 experts, 2048 x 2048, 128 x top-4 56.9 / 62.8 / 52.8; 45.5 / 56.0 / 42.9.  Without preferences within 0.5 % of past them everywhere.
template <int STAGE>
bool takes_nt(const MoeParams& p, int tile_m) {
    return p.experts > p.cached && 4ll * p.tokens * p.topk <= 3ll * p.experts * tile_m;
}

// Whether a stage multiplies two consecutive blocks of an expert in one workgroup.  Stage 1 with one-byte weights always does with blocks of up to 32 rows (64 tokens x
// top-8 on 32 experts, blocks of 16: 107 -> 92 us).  The other stages stream half the bytes and have fewer workgroups from the start: they do with blocks of 16 where
// most experts have two and the pairs still make three workgroups a CU (us single / paired, weights in memory, 32 experts, 4096 x 1536: int4 stage 1 64 tokens x
// top-8 46.5 / 41.7, 96 53.9 / 41.7, but 51 42.4 / 41.8; 128 experts, 2048 x 512, 256 tokens 36.1 / 31.6, 204 29.8 / 31.3; stage 2 fp8 51 tokens 40.7 / 35.4, 64 41.3 /
// 36.2, 96 45.5 / 41.1, int4 64 26.7 / 24.8, 96 36.0 / 28.3, but K = 512 33.9 / 34.4, two workgroups a CU 17.3 / 18.9, one 18.8 / 20.8).
template <int KIND, int STAGE>
bool takes_pairs(const MoeParams& p, int block_m) {
    if (!p.pair_blocks || block_m > 32) return false;
    if (STAGE == 1 && KIND != KIND_INT8W4) return true;
    const int64_t pairs = (int64_t)p.tokens * p.topk, rows = 16ll * p.experts, tn = STAGE == 1 ? 64 : 128;
    if (block_m != 16 || p.by_position || p.experts * ((p.n_out + tn - 1) / tn) < 3ll * psg_cu_count()) return false;
    return STAGE == 1 ? 10 * pairs >= 9 * rows : p.K >= 1024 && 4 * pairs > 3 * rows;
}

template <int KIND, int STAGE, int NR>
hipError_t launch_nr(MoeParams p, MoeRowsParams rows, int block_m, int blocks, bool pair, hipStream_t stream) {
    const unsigned nx = (unsigned)((p.n_out + 64 * NR - 1) / (64 * NR));
    rows.wgs = 0;
    p.cached = moe_experts_cached(STAGE, ((STAGE == 1 ? 2ll * p.n_out : p.n_out) * p.K) >> (KIND == KIND_INT8W4 ? 1 : 0));
    // rows of the grid for the lists, as far as it has any left (65535 of them)
    const int list_rows = (int)((ROWS_INDEX_WGS + nx - 1) / nx);
    const bool lists = STAGE == 2 && p.by_position && rows.sorted_size <= moe_rows_share_max(block_m) && blocks + list_rows <= 65535;
    if (lists) {
        rows.wgs = list_rows;
    } else if (STAGE == 2 && p.by_position) {
        const hipError_t e = psg_launch_moe_rows_index(rows, stream);
        if (e != hipSuccess) return e;
    }
    const bool deep = takes_deep<KIND, STAGE>(p, block_m, blocks, (int)nx);
    const dim3 grid(nx, blocks + rows.wgs, 1);
#define PSG_MOE(MR_, CO_)                                                                                \
    {                                                                                                    \
        constexpr bool kOnly = CO_ == 2 || (MR_ <= 2 && STAGE == 1 && KIND != KIND_INT8W4); /* always deep */ \
        constexpr bool kNt = MR_ <= 2 || CO_ == 2;                             /* may read W past the caches */ \
        if constexpr (STAGE == 2 && CO_ == 1) {  /* (a stage by rows takes no pairs) */                   \
            if (lists) {                                                                                 \
                hipLaunchKernelGGL((k_moe_gemm<KIND, MR_, NR, STAGE, CO_, 0, MoeRowsParams>), grid, dim3(256), 0, stream, p, rows); \
                return hipGetLastError();                                                                \
            }                                                                                            \
        }                                                                                                \
        if (kNt && takes_nt<STAGE>(p, block_m * CO_)) hipLaunchKernelGGL((k_moe_gemm<KIND, MR_, NR, STAGE, CO_, kNt ? 2 : 1>), grid, dim3(256), 0, stream, p); \
        else if (deep || kOnly) hipLaunchKernelGGL((k_moe_gemm<KIND, MR_, NR, STAGE, CO_, 1>), grid, dim3(256), 0, stream, p); \
        else hipLaunchKernelGGL((k_moe_gemm<KIND, MR_, NR, STAGE, CO_, kOnly ? 1 : 0>), grid, dim3(256), 0, stream, p); \
        return hipGetLastError();                                                                        \
    }
    if (pair && block_m == 16) PSG_MOE(2, 2)
    if constexpr (STAGE == 1 && KIND != KIND_INT8W4) {
        if (pair && block_m == 32) PSG_MOE(4, 2)
    }
    if (block_m == 16) PSG_MOE(1, 1)
    if (block_m == 32) PSG_MOE(2, 1)
    if (block_m == 64) PSG_MOE(4, 1)
    if (block_m == 128) PSG_MOE(8, 1)
#undef PSG_MOE
    return hipErrorInvalidValue;
}

template <int KIND, int STAGE>
hipError_t launch_kind(const MoeParams& p, const MoeRowsParams& rows, int block_m, int blocks, hipStream_t stream) {
    const bool pair = takes_pairs<KIND, STAGE>(p, block_m);
    // Stage 2 on 128 columns per workgroup where they divide the output, stage 1, which has two accumulator sets, on 64: measured at 4096 tokens x top-8, blocks of 128: stage 1 488 us with
    // 64 columns against 800 with 128, stage 2 442 against 412 (stage 2 with 256 columns: 805 with one workgroup per CU, 492 when held to two).
    if constexpr (STAGE == 2) {
        if (p.n_out % 128 == 0) return launch_nr<KIND, STAGE, 2>(p, rows, block_m, blocks, pair, stream);
    }
    return launch_nr<KIND, STAGE, 1>(p, rows, block_m, blocks, pair, stream);
}

}  // namespace

hipError_t psg_launch_moe_pair(const MoeParams& p, const MoeRowsParams& rows, int kind, int stage, int blocks, hipStream_t stream);

// Whether the 128x256 tiles (moe_gemm_pair.hip) are the better way for blocks of 128 rows: where there are about as many of them as CUs, blocks counted as
// a routing needs them on average (the pairs' and half a block for every expert), and in stage 1, whose weights are the larger ones, more than a block an expert.
// Measured, us k_moe_gemm / 128x256 tiles (fp8; int8 the same or a few per cent better), tiles by that count: stage 1 120 16.7 / 19.9, 136 15.7 / 16.3, 144 40.0 /
// 39.9, 192 16.5 / 17.4, 198 19.5 / 17.7, 240 43.5 / 40.3, 984 75.6 / 55.6; but 128 rows an expert, 576 tiles, 107.5 / 111.3.  Stage 2 97 19.3 / 20.5, 128 21.1 / 23.4,
// 160 18.6 / 18.3, 165 22.9 / 19.7, 192 26.6 / 24.5, 428 38.5 / 27.4, 656 76.1 / 61.1.  The same where stage 2 adds directly (no scratch, few slots, under capture: 4096 x
// top-8 379 / 326, 2048 x top-3 75.5 / 67.5, 4096 x top-1 56.1 / 55.2).
bool takes_pair(const MoeParams& p, int stage, int blocks) {
    const long pairs = (long)p.tokens * p.topk, cus = psg_cu_count(), tn = stage == 1 ? 128 : 256;
    const long expected = pairs / 128 + p.experts / 2, tiles = (expected < blocks ? expected : blocks) * ((p.n_out + tn - 1) / tn);
    return stage == 1 ? tiles * 4 > cus * 3 && pairs >= 144L * p.experts : tiles * 8 >= cus * 5;
}

// kind: KIND_INT8 / KIND_FP8 / KIND_INT8W4; stage 1 or 2; rows: where p.by_position is set; block_m in {16, 32, 64, 128}; blocks = entries of expert_ids
hipError_t psg_launch_moe_gemm(const MoeParams& p, const MoeRowsParams& rows, int kind, int stage, int block_m, int blocks, hipStream_t stream) {
    if (block_m == 128 && kind != KIND_INT8W4 && p.out_dtype != OUT_F32 && p.pair_blocks && takes_pair(p, stage, blocks)) return psg_launch_moe_pair(p, rows, kind, stage, blocks, stream);
    if (kind == KIND_INT8) return stage == 1 ? launch_kind<KIND_INT8, 1>(p, rows, block_m, blocks, stream) : launch_kind<KIND_INT8, 2>(p, rows, block_m, blocks, stream);
    if (kind == KIND_INT8W4) return stage == 1 ? launch_kind<KIND_INT8W4, 1>(p, rows, block_m, blocks, stream) : launch_kind<KIND_INT8W4, 2>(p, rows, block_m, blocks, stream);
    return stage == 1 ? launch_kind<KIND_FP8, 1>(p, rows, block_m, blocks, stream) : launch_kind<KIND_FP8, 2>(p, rows, block_m, blocks, stream);
}

// sum over the topk slots: y[t, :] = sum_s x[t, s, :] (bf16, fp16 or fp32, the same type in and out; fp32 sum in slot order)
namespace {
// mask != nullptr: slot k of token t only counts when mask[ids[t*topk + k]] != 0 (expert parallelism: the rows of experts
// that live elsewhere were never written by stage 2)
__global__ void __launch_bounds__(256) k_moe_reduce(const uint16_t* x, uint16_t* y, int tokens, int topk, int dim, int out_dtype,
                                                    const int32_t* mask, const int32_t* ids, int experts) {
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;   // one thread per 4 columns
    const size_t quads = (size_t)tokens * (size_t)(dim >> 2);
    if (q >= quads) return;
    const size_t t = q / (size_t)(dim >> 2), c = (q % (size_t)(dim >> 2)) << 2;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    for (int k = 0; k < topk; k++) {
        if (mask) {
            const int e = ids[t * topk + k];
            if ((unsigned)e >= (unsigned)experts || mask[e] == 0) continue;
        }
        if (out_dtype == OUT_F32) {
            const v4f v = *reinterpret_cast<const v4f*>(reinterpret_cast<const float*>(x) + (t * topk + k) * (size_t)dim + c);
            s0 += v[0]; s1 += v[1]; s2 += v[2]; s3 += v[3];
            continue;
        }
        const v2i v = *reinterpret_cast<const v2i*>(x + (t * topk + k) * (size_t)dim + c);
        const uint16_t h0 = (uint16_t)(v[0] & 0xFFFF), h1 = (uint16_t)((uint32_t)v[0] >> 16), h2 = (uint16_t)(v[1] & 0xFFFF), h3 = (uint16_t)((uint32_t)v[1] >> 16);
        if (out_dtype == OUT_BF16) {
            s0 += from_out16<OUT_BF16>(h0); s1 += from_out16<OUT_BF16>(h1); s2 += from_out16<OUT_BF16>(h2); s3 += from_out16<OUT_BF16>(h3);
        } else {
            s0 += from_out16<OUT_FP16>(h0); s1 += from_out16<OUT_FP16>(h1); s2 += from_out16<OUT_FP16>(h2); s3 += from_out16<OUT_FP16>(h3);
        }
    }
    if (out_dtype == OUT_F32) {
        *reinterpret_cast<v4f*>(reinterpret_cast<float*>(y) + t * (size_t)dim + c) = (v4f){s0, s1, s2, s3};
        return;
    }
    const v2i o = out_dtype == OUT_BF16 ? pack4_out16<OUT_BF16>(s0, s1, s2, s3) : pack4_out16<OUT_FP16>(s0, s1, s2, s3);
    *reinterpret_cast<v2i*>(y + t * (size_t)dim + c) = o;
}
}  // namespace

hipError_t psg_launch_moe_reduce(const void* x, void* y, int tokens, int topk, int dim, int out_dtype, const int32_t* mask,
                                 const int32_t* ids, int experts, hipStream_t stream) {
    const size_t quads = (size_t)tokens * (size_t)(dim >> 2);
    hipLaunchKernelGGL(k_moe_reduce, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, stream, static_cast<const uint16_t*>(x),
                       static_cast<uint16_t*>(y), tokens, topk, dim, out_dtype, mask, ids, experts);
    return hipGetLastError();
}

// What moe_reads_once says of every block of a list, by one wavefront each (for tests)
namespace {
__global__ void __launch_bounds__(64) k_moe_reads_once(const int32_t* expert_ids, int blocks, int used, int per_tile, int experts, int cached, int32_t* out) {
    const int blk = (int)blockIdx.x, lane = (int)threadIdx.x, e = expert_ids[blk];
    const bool counts = blk < used && (unsigned)e < (unsigned)experts;
    const int once = moe_reads_once(moe_neighbours(expert_ids, blocks, blk, per_tile, lane), expert_ids, used, blk, per_tile, e, experts, cached, lane);
    if (lane == 0) out[blk] = counts ? once : -1;
}
}  // namespace

hipError_t psg_launch_moe_reads_once(const int32_t* expert_ids, int blocks, int used, int per_tile, int experts, int cached, int32_t* out, hipStream_t stream) {
    hipLaunchKernelGGL(k_moe_reads_once, dim3((unsigned)blocks), dim3(64), 0, stream, expert_ids, blocks, used, per_tile, experts, cached, out);
    return hipGetLastError();
}
