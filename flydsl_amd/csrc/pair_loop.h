// Mainloop of the 128x256 tile that runs two workgroups per CU (gfx950), for fp4 operands with e8m0 scales on both sides, fp8, int8, fp16 and bf16: the dense
// MXFP4 GEMM (gemm_mx_pair.hip), that of the 8- and 16-bit kinds (gemm_pair.hip) and the stages of both MoE pairs on blocks of 128 sorted rows (moe_mx_gemm.hip,
// moe_gemm_pair.hip).
//
// Four wavefronts side by side along N, each 128 rows x 64 weight rows (128 accumulator registers a lane), 128 bytes of K a step:
//   * A goes global -> LDS by DMA into four stages of 16 KB (rows of 128 bytes, 16-byte pieces XORed with row / 2), requested three steps
//     ahead; a lane's source address is its row's, so rows may be gathered.
//   * W never touches LDS: a wavefront's fragments are its own.  They are fetched three half steps (64 bytes of K) ahead into a ring of four
//     half-step register sets; two whole-step sets need the same 64 registers and are ahead by half as much.  (fp8, whose MFMA takes both
//     halves, has those: a step ahead.)
//   * The scale dwords of a step, 4 chunks of 256 bytes on the A side and 8 on the W side, are one 16-byte DMA of three of the wavefronts: a DMA
//     takes 64 lanes anywhere, so 16 lanes bring a chunk and one instruction four of them.  Scales that are not on 16 bytes come 4 bytes a lane, a chunk an instruction, three
//     of every wavefront (SCB = 4).
//   * At most one memory instruction stands behind an MFMA: what is issued between two of them in a row, the matrix cores wait for (one
//     workgroup alone on a CU, zero operands: 1,580 core cycles a step with the instructions in front of each block of four MFMAs, 1,450 like
//     this; 1,088 is what 64 MFMAs take).
//   * Within a half step (fp8: a step) every MFMA has one of its operands in common with the one in front of it, A or W; where a half begins both change, two of 64 times a step (fp8: one of 32). At the power limit what the operands' change costs is clock (a
//     loop of nothing but MFMAs on random data, eight A and four W fragments, us with all W for one A fragment after the other / as here / with both operands changing every
//     time: fp4 3620 / 3508 / 3710, int8 3160 / 3070 / 3290, bf16 3180 / 3090 / 3280, fp8 3000 / 2970 / 3100).  Eight products of two A and four W fragments in a row like a
//     snake; fp8, whose fragments have no registers for two of A and the next two, back through W in every other m-block.  us before / now: fp4 4096x7168x2048 36.1 / 35.5,
//     8192x4096x8192 116.0 / 114.7; bf16 1500x5264x4096 48.5 / 47.5, fp16 49.5 / 48.4; int8 1500x11264x4096 66.2 / 65.3; fp8 the same 66.9 / 66.7; MX layer of 4096 tokens x top-8
//     457 / 452, int8 735 / 729.  The order of an accumulator's own sums is the same.
// Two workgroups on a CU take 2,600 to 3,000 cycles for a step of both, the 256x256 tile of eight wavefronts (gemm_tiled8.h) 2,850 to 3,100 for as much
// work; but they are not in step with each other, so that the start and the end of one, 7 of the 18 us of a tile with K = 2048, stand beside
// MFMAs of the other.
#pragma once
#include "gemm_tiled.h"
#include "lds_dma.h"

namespace {

template <int KIND>
struct Pair {
    static constexpr int MR = 8, NR = 4, NS = 4;  // 16-row blocks of A, of W a wavefront; LDS stages
    static constexpr int TM = 128, TN = 256;
    static constexpr int STAGE = TM * TK;         // bytes of one A stage
    static constexpr int SC_SLOT = KIND == KIND_MXFP4 ? 12 * 256 : 0;  // scale dwords of a step
    static constexpr int LDS_BYTES = NS * (STAGE + SC_SLOT);
    // two workgroups a CU, with `more` bytes each for what a kernel adds
    static constexpr bool fits(int more) { return 2 * (LDS_BYTES + more) <= 160 * 1024; }
};
using MxPair = Pair<KIND_MXFP4>;

// acc[mi][ni] = A (rows 16 mi ..) x W (the wavefront's 16-row block ni) over K bytes of a row (multiples of 64); 0 without any.
//   lds      LDS_BYTES, 1 KB aligned: the A stages, behind them the scale slots; free again at the end
//   a_voff   this lane's offsets into `ra` of the four 1 KB blocks (8 rows) that its wavefront fetches of a stage: of row (4 wave + j) 8 + lane / 8,
//            16-byte piece (lane % 8) ^ (row / 2 % 8); out of the descriptor's bounds for a row that reads as zero
//   b_voff   this lane's offsets into `rb` of the wavefront's four 16-row blocks, b_step and b_half from a step and a half step to the next (2048 and 1024 in the
//            preshuffled order)
// fp4 only (rs and rs_w: any descriptors otherwise):
//   s_voff   this lane's offset into `rs`, the scales of wavefront 0 and 3: A side, 1 and 2: W side chunks 0..3 and 4..7 of the tile: chunk
//            lane / 16, 16-byte piece lane % 16
//   chunk0/1 which of the eight W-side chunks belong to the wavefront's blocks 0, 1 and 2, 3
//   SCB = 4: `rs` the A side, s_voff chunk `wave` of it, 4-byte piece `lane`; `rs_w` the W side, in chunks of chunk_bytes (SCB = 16: any descriptor)
template <int KIND, int SCB = 16, class ACC>
__device__ __forceinline__ void pair_loop(ACC (&acc)[8][4], uint8_t* lds, const __amdgpu_buffer_rsrc_t ra, const uint32_t (&a_voff)[4],
                                          const __amdgpu_buffer_rsrc_t rb, const uint32_t (&b_voff)[4], const int K, const int wave, const int lane,
                                          const uint32_t b_step, const uint32_t b_half, const __amdgpu_buffer_rsrc_t rs, const __amdgpu_buffer_rsrc_t rs_w,
                                          const uint32_t s_voff = 0, const int chunk0 = 0, const int chunk1 = 0, const uint32_t chunk_bytes = 0) {
    using P = Pair<KIND>;
    constexpr int MR = P::MR, NR = P::NR, NS = P::NS, STAGE = P::STAGE, SC_SLOT = P::SC_SLOT;
    constexpr bool MX = KIND == KIND_MXFP4, WHOLE = KIND == KIND_FP8;  // WHOLE: an MFMA takes both halves of a step
    const int li = lane & 15, lg = lane >> 4;
    const int KT = (K + TK - 1) / TK, KF = K / TK;  // steps, whole steps
    // 16-byte piece of its row that this lane fetches, by the parity of the block (the rows of a block count from 8 j)
    const int a_kc[2] = {(lane & 7) ^ (lane >> 4), (lane & 7) ^ (lane >> 4) ^ 4};
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    uint8_t* const lds_x = lds + NS * STAGE;
    // (wavefront 3 brings the bytes of wavefront 0 once more: all of them count the same number of DMAs)
    const uint32_t sc_dst = lds_base + (uint32_t)(NS * STAGE) + (uint32_t)(wave == 3 ? 0 : wave) * 1024u;

    // DMA j of step kt: 0..3 A, from 4 on scales.  Without CHK the step is known to be before the end
    constexpr int N_DMA = !MX ? 4 : SCB == 16 ? 5 : 7;
    auto dma = [&](int kt, int stage, int j, auto CHK) __attribute__((always_inline)) {
        const bool has = !decltype(CHK)::value || kt < KT, in = !decltype(CHK)::value || kt * TK + a_kc[j & 1] * 16 < K;
        if (j < 4) dma16(ra, lds_base + (uint32_t)(stage * STAGE + (wave * 4 + j) * 1024), in ? a_voff[j < 4 ? j : 0] : OOB, has ? (uint32_t)kt * TK : 0u);
        else if (SCB == 16) dma16(rs, sc_dst + (uint32_t)(stage * SC_SLOT), has ? s_voff : OOB, has ? (uint32_t)kt * 256u : 0u);
        else if (j == 4) dma4(rs, lds_base + (uint32_t)(NS * STAGE + stage * SC_SLOT + wave * 256), has ? s_voff : OOB, has ? (uint32_t)kt * 256u : 0u);
        else {
            const int ch = j == 5 ? chunk0 : chunk1;
            dma4(rs_w, lds_base + (uint32_t)(NS * STAGE + stage * SC_SLOT + 1024 + ch * 256), has ? (uint32_t)ch * chunk_bytes + (uint32_t)lane * 4u : OOB, has ? (uint32_t)kt * 256u : 0u);
        }
    };
    v4i bw[4][NR];
    auto load_w = [&](int kt, int half, int ni, v4i* dst, auto CHK) __attribute__((always_inline)) {
        const bool has = !decltype(CHK)::value || kt * TK + half * 64 < K;
        dst[ni] = buf_load16(rb, has ? b_voff[ni] : OOB, has ? (uint32_t)kt * b_step + (uint32_t)half * b_half : 0u);
    };
    const int f_base[2] = {li * TK + ((lg ^ ((li >> 1) & 7)) << 4), li * TK + (((4 + lg) ^ ((li >> 1) & 7)) << 4)};
    constexpr int AHEAD = 2;  // blocks of four MFMAs that an A fragment is read ahead
    static_assert(AHEAD == 2, "a ring of four: two fragments at work, the two behind them on their way");
    v4i fr[4];
    auto read_frag = [&](int stage, int half, int mi, v4i& dst) __attribute__((always_inline)) {
        dst = *reinterpret_cast<const v4i*>(&lds[stage * STAGE + mi * 16 * TK + f_base[half]]);
    };
    int sav[2][4], sbv[2][2];
    auto read_sc = [&](int slot, int q, int set) __attribute__((always_inline)) {
        if (q < 4) sav[set][q < 4 ? q : 0] = *reinterpret_cast<const int*>(lds_x + slot * SC_SLOT + q * 256 + lane * 4);
        else sbv[set][q < 4 ? 0 : q - 4] = *reinterpret_cast<const int*>(lds_x + slot * SC_SLOT + 1024 + (q == 4 ? chunk0 : chunk1) * 256 + lane * 4);
    };

    // fp8: eight m-blocks of four MFMAs of 32 cycles, back through W in every other one; the DMAs of step kt + 3, then the W fragments of the next step into the other set, early in
    // the step, the A fragments an m-block ahead
    auto whole_step = [&](int kt, auto SP, auto CHK) __attribute__((always_inline)) {
        constexpr int S = decltype(SP)::value, B0 = 2 * (S & 1), B1 = 2 - B0;  // sets of W: halves B0, B0 + 1 and B1, B1 + 1
        static_for<MR>([&](auto MI) {
            constexpr int mi = decltype(MI)::value, f = 2 * (mi & 1), fn = 2 - f;
            static_for<NR>([&](auto NI) {
                constexpr int at = decltype(NI)::value, ni = mi & 1 ? NR - 1 - at : at, slot = mi * NR + at;
                const v8i a = {fr[f][0], fr[f][1], fr[f][2], fr[f][3], fr[f + 1][0], fr[f + 1][1], fr[f + 1][2], fr[f + 1][3]};
                const v8i b = {bw[B0][ni][0], bw[B0][ni][1], bw[B0][ni][2], bw[B0][ni][3], bw[B0 + 1][ni][0], bw[B0 + 1][ni][1], bw[B0 + 1][ni][2], bw[B0 + 1][ni][3]};
                if constexpr (WHOLE) mfma_f8(acc[mi][ni], b, a);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (at < 2) {
                    if constexpr (mi + 1 < MR) read_frag(S, at, mi + 1, fr[fn + at]);
                    else read_frag((S + 1) % NS, at, 0, fr[fn + at]);
                }
                if constexpr (slot >= 3 && slot < 7) dma(kt + 3, (S + 3) % NS, slot - 3, CHK);
                if constexpr (slot >= 7 && slot < 15) load_w(kt + 1, slot & 1, (slot - 7) / 2, bw[B1 + (slot & 1)], CHK);
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NR + N_DMA + 2 * NR) : "memory");
    };

    // Step kt (kt % 4 = S): sixteen blocks of four MFMAs, m-blocks by twos, eight of the lower half of K and eight of the upper.  A's stage and scales of the step
    // have landed for everybody a step ago, so its first fragments and scales were read before the barrier in front of it.
    auto half_steps = [&](int kt, auto SP, auto CHK) __attribute__((always_inline)) {
        constexpr int S = decltype(SP)::value, SS = S & 1;
        static_for<16>([&](auto BI) {
            constexpr int b = decltype(BI)::value, half = b >> 3;
            static_for<NR>([&](auto NI) {
                constexpr int at = decltype(NI)::value;
                // two blocks: the products of two A fragments with all of W
                constexpr int q = (b & 1) * 4 + at, fb = (b & 14) + (((q + 1) >> 1) & 1), mi = fb & 7, ni = b & 2 ? NR - 1 - (q >> 1) : q >> 1;
                if constexpr (MX) mfma_mx<half, ni & 1, mi & 1>(acc[mi][ni], bw[(2 * S + half) % 4][ni], fr[fb & 3], sbv[SS][ni / 2], sav[SS][mi / 2]);
                else if constexpr (KIND == KIND_INT8) mfma_i8(acc[mi][ni], bw[(2 * S + half) % 4][ni], fr[fb & 3]);
                else if constexpr (KIND == KIND_BF16) mfma_bf16(acc[mi][ni], bw[(2 * S + half) % 4][ni], fr[fb & 3]);
                else if constexpr (KIND == KIND_FP16) mfma_f16(acc[mi][ni], bw[(2 * S + half) % 4][ni], fr[fb & 3]);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr ((b & 1) == 0 && at < 2) {
                    constexpr int nb = b + AHEAD + at;
                    if constexpr (nb < 16) read_frag(S, nb >> 3, nb & 7, fr[nb & 3]);
                    else read_frag((S + 1) % NS, 0, nb - 16, fr[nb & 3]);
                }
                if constexpr (MX && at == 3 && b >= 10) read_sc((S + 1) % NS, b - 10, SS ^ 1);
                // The DMAs of step kt + 3 and the W fragments three half steps ahead.  The compiler counts only the loads it knows, W's, so its waits
                // for W let as many instructions be on their way as there are W loads behind the awaited one, DMAs among them: in each half the DMAs
                // go first, and both halves have some.
                if constexpr (at == 2) {
                    constexpr int FROM = N_DMA == 7 ? 0 : 1, LOW = 4 - FROM;  // block of the first DMA in a half; DMAs in the lower one
                    if constexpr (b >= FROM && b < 4) dma(kt + 3, (S + 3) % NS, b - FROM, CHK);
                    if constexpr (b >= 4 && b < 8) load_w(kt + 1, 1, b - 4, bw[(2 * S + 3) % 4], CHK);
                    if constexpr (b >= 8 + FROM && b < 8 + FROM + N_DMA - LOW) dma(kt + 3, (S + 3) % NS, b - 8 - FROM + LOW, CHK);
                    if constexpr (b >= 11 && b < 15) load_w(kt + 2, 0, b - 11, bw[(2 * S + 4) % 4], CHK);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        // the DMAs this wavefront issued a step ago (of step kt + 2) have landed before the barrier: behind the last of them it has issued four W
        // loads of that step and everything of this one
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NR + N_DMA + 2 * NR) : "memory");
    };

    auto step = [&](int kt, auto SP, auto CHK) __attribute__((always_inline)) {
        if constexpr (WHOLE) whole_step(kt, SP, CHK);
        else half_steps(kt, SP, CHK);
    };

    // prologue: A and scales of steps 0 and 1, W of the first half step, A and scales of step 2, W of the two half steps behind (fp8: A of steps 0
    // to 2, W of step 0)
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int j = 0; j < N_DMA; j++) dma(s, s, j, std::true_type{});
    if constexpr (!WHOLE) {
#pragma unroll
        for (int ni = 0; ni < NR; ni++) load_w(0, 0, ni, bw[0], std::true_type{});
    }
#pragma unroll
    for (int j = 0; j < N_DMA; j++) dma(2, 2, j, std::true_type{});
    if constexpr (WHOLE) {
#pragma unroll
        for (int ni = 0; ni < NR; ni++) load_w(0, 0, ni, bw[0], std::true_type{});
    }
#pragma unroll
    for (int ni = 0; ni < NR; ni++) load_w(0, 1, ni, bw[1], std::true_type{});
    if constexpr (!WHOLE) {
#pragma unroll
        for (int ni = 0; ni < NR; ni++) load_w(1, 0, ni, bw[2], std::true_type{});
    }
#pragma unroll
    for (int mi = 0; mi < MR; mi++)
#pragma unroll
        for (int ni = 0; ni < NR; ni++) acc[mi][ni] = (ACC){0, 0, 0, 0};
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((WHOLE ? 2 : 3) * NR + N_DMA) : "memory");
    if constexpr (WHOLE) {
        read_frag(0, 0, 0, fr[0]);
        read_frag(0, 1, 0, fr[1]);
    } else {
        static_for<AHEAD>([&](auto I) { read_frag(0, 0, decltype(I)::value, fr[decltype(I)::value]); });
    }
    if constexpr (MX) {
#pragma unroll
        for (int q = 0; q < 6; q++) read_sc(0, q, 0);
    }

    // four steps an iteration (stages and register sets are compile-time); the first loop while every load of it is before the end, then with
    // checks, then what is left
    int kt = 0;
    for (; kt + 7 <= KF; kt += NS) static_for<NS>([&](auto I) { step(kt + decltype(I)::value, I, std::false_type{}); });
    for (; kt + NS <= KT; kt += NS) static_for<NS>([&](auto I) { step(kt + decltype(I)::value, I, std::true_type{}); });
    static_for<NS - 1>([&](auto I) {
        if (kt + decltype(I)::value < KT) step(kt + decltype(I)::value, I, std::true_type{});
    });
    // wait states between the last MFMA and the first ordinary read of an accumulator (the compiler does not know that the asm statements are
    // MFMAs); every DMA still on its way (redirected past the bounds) is done before the stages are reused
    asm volatile("s_nop 15\n\ts_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
}

// A tile of 16-bit C on its way through LDS, as whole rows of 512 bytes, 16-byte granules XORed with the row: where a lane's four columns of row 16 mi + li in the 16-column block `nb` go
__device__ __forceinline__ uint8_t* pair_c_at(uint8_t* lds, int mi, int nb, int li, int lg) { return lds + (mi * 16 + li) * 512 + ((((nb * 2 + (lg >> 1)) ^ li) & 31) << 4) + (lg & 1) * 8; }

// ... and its rows of half `half`, out by all lanes.  `rc` is C from the tile's first row on: rows past the last lie behind its bound, granules past N are redirected there.
__device__ __forceinline__ void pair_store_rows(const uint8_t* lds, int half, const __amdgpu_buffer_rsrc_t rc, int n0, int N, int tid) {
    const int g = tid & 31, r0 = tid >> 5, n = n0 + g * 8;
    const uint32_t off = ((uint32_t)r0 * (uint32_t)N + (uint32_t)n) * 2u, step = 16u * (uint32_t)N;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int i = half * 8 + j, r = r0 + i * 8;
        const v4i v = *reinterpret_cast<const v4i*>(lds + r * 512 + ((g ^ (r & 15)) << 4));
        __builtin_amdgcn_raw_buffer_store_b128((v4u)v, rc, (int)(n < N ? off + (uint32_t)i * step : OOB), 0, 0);
    }
}

}  // namespace
