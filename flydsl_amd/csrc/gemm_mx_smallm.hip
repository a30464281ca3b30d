// Small-M MX preshuffle GEMM (64 rows a workgroup) for every format the general kernel takes: A in fp4 / fp6 / fp8, W in fp4 / fp8, strided
// rows, batches over blockIdx.z.  Operand and scale layouts: gemm_mx_generic.hip.
//
// Bound: the bytes of W and, from 32 rows on, of A, which every workgroup reads whole.  A workgroup owns 32 columns and splits K over
// its wavefronts in steps of 256 elements, so N / 32 workgroups stream W with all their loads in flight, the partial sums meet in LDS in a
// fixed order, and there is neither a partials buffer nor a second launch.  The 64 x 128 tiles of the general kernel gave such
// calls N / 128 workgroups per K split and a finalising launch: fp8 x fp4, 64 x 8192 x 8192, 20.2 -> 12.3 us (37 MB, 7.2 at the rate of
// a large copy), one row of it 12.2 -> 7.7.  Of the 12.3 about 5 go into reading the 512 KB of A through every CU.
#include "lds_dma.h"
#include "psg_common.h"

namespace {

template <int F>
struct MxCode {  // cbsz / blgp format code of the MFMA
    static constexpr int value = F == MXF_FP4 ? 4 : (F == MXF_FP6 ? 2 : 0);
};

template <int AF, int BF, int MB, int NW>
__global__ void __launch_bounds__(NW * 64) k_mx_smallm(MxGenParams p) {
    constexpr int AB = AF == MXF_FP4 ? 64 : 128, BB = BF == MXF_FP4 ? 64 : 128;  // bytes of a row per 128 elements
    constexpr int AL = AB / 64, BL = BB / 64;                                    // 16-byte loads of an operand
    constexpr int MC = (MB + 1) / 2;                                             // 32-row scale chunks of A
    // fp6 / fp8 A (256 bytes of a row per step) travels row by row into a patch of the wavefront's own in LDS: fragment-order loads
    // touch 16 rows an instruction, which cost the texture addresser more than the whole W stream (fp8 x fp4, 64 x 8192 x 8192: 19.0 us).
    // fp4 A (128 bytes) is loaded in fragment order.
    constexpr bool PATCH = AF != MXF_FP4;
    constexpr int PASSES = MB * 4;                                               // 1 KB of the patch (four rows) per DMA instruction
    constexpr int PW = PATCH ? MB * 16 * 256 : MB * 2 * 64 * 16;                 // a wavefront's bytes: patch, then its partial sums
    static_assert(PW >= MB * 2 * 64 * 16, "the partial sums must fit the patch");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[NW * PW];

    const int tid = threadIdx.x;
    const int wave = wave_id();
    const int lane = tid & 63, li = lane & 15, lg = lane >> 4;
    // workgroups go round-robin over the 8 XCDs: each XCD gets one contiguous range of columns, so the lines of C that two
    // neighbours share are completed in one L2
    const int np = (gridDim.x & 7) == 0 ? (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) : (int)blockIdx.x;
    const uint64_t z = blockIdx.z;
    const int m0 = (int)blockIdx.y * (16 * MB), M = p.M - m0;  // rows of this workgroup: up to 16 MB from m0 on (MB = 4 beyond 64 rows)
    const int KT = p.K >> 8;
    const int per = (KT + NW - 1) / NW;
    const int s_begin = wave * per;
    const int s_end = (s_begin + per) < KT ? (s_begin + per) : KT;
    const uint32_t b_row_bytes = BF == MXF_FP4 ? (uint32_t)p.K >> 1 : (uint32_t)p.K;
    const uint32_t a_row_bytes = AF == MXF_FP4 ? (uint32_t)p.K >> 1 : (uint32_t)p.K;
    const uint32_t a_rs = (uint32_t)p.a_row_stride, sa_cs = (uint32_t)p.sa_chunk_stride, chunk_bytes = (uint32_t)KT * 256u;

    __amdgpu_buffer_rsrc_t ra = make_rsrc_uniform(p.a + z * (uint64_t)p.a_batch + (uint64_t)m0 * a_rs, (uint64_t)(M - 1) * a_rs + a_row_bytes);  // rows >= M read as zero
    __amdgpu_buffer_rsrc_t rb = make_rsrc(p.b + z * (uint64_t)p.b_batch + (uint64_t)np * 32ull * b_row_bytes, 32ull * b_row_bytes);
    __amdgpu_buffer_rsrc_t rsa = make_rsrc(p.sa + z * (uint64_t)p.sa_batch + (uint64_t)(m0 >> 5) * sa_cs, (uint64_t)(((M + 31) >> 5) - 1) * sa_cs + chunk_bytes);
    __amdgpu_buffer_rsrc_t rsb = make_rsrc(p.sb + z * (uint64_t)p.sb_batch + (uint64_t)np * chunk_bytes, chunk_bytes);
    // the lane's 16-byte pieces of a 128-element step of its A row: fp4 g; fp6 2g, 2g + 1; fp8 g, 4 + g
    const uint32_t a_voff = (uint32_t)li * a_rs + (uint32_t)lg * 16u;

    v4f acc[MB][2];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) acc[mb][0] = acc[mb][1] = (v4f){0.f, 0.f, 0.f, 0.f};

    auto widen = [](const v4i* x, auto L) {
        if constexpr (decltype(L)::value == 1) return __builtin_shufflevector(x[0], x[0], 0, 1, 2, 3, -1, -1, -1, -1);
        else return __builtin_shufflevector(x[0], x[1], 0, 1, 2, 3, 4, 5, 6, 7);
    };
    uint8_t* const patch = lds + wave * PW;
    const uint32_t patch_lds = (uint32_t)(uintptr_t)patch;
    // DMA instruction ps fills rows 4 ps .. + 3: lane l writes physical chunk l % 16 of row 4 ps + l / 16 and therefore fetches that row's
    // logical chunk (l % 16) ^ (row % 16); the term repeats every four instructions
    uint32_t dma_voff[PATCH ? 4 : 1];
    if constexpr (PATCH) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int row = v * 4 + (lane >> 4);
            dma_voff[v] = (uint32_t)row * a_rs + (uint32_t)((lane & 15) ^ row) * 16u;
        }
    }
    v4i bq[2][2][2][BL], aq[2][PATCH ? 1 : MB][2][AL];
    int sav[2][MC], sbv[2];
    constexpr int BEHIND = 4 * BL + MC + 1;  // loads requested behind the DMAs of a step: W and scales of the next one
    // requests of step s: W, scales and fragment-order A into register set SET.  A step past the slice reads zeros.
    auto load_regs = [&](int s, auto SETP) __attribute__((always_inline)) {
        constexpr int u = decltype(SETP)::value;
        const bool ok = s < s_end;  // wave-uniform
        const uint32_t so = ok ? (uint32_t)s : 0u;
        if constexpr (!PATCH) {
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
#pragma unroll
                for (int kh = 0; kh < 2; kh++)
#pragma unroll
                    for (int l = 0; l < AL; l++)
                        aq[u][mb][kh][l] = buf_load16(ra, ok ? a_voff + (uint32_t)mb * 16u * a_rs : OOB, (so * 2u + (uint32_t)kh) * (uint32_t)AB);
        }
#pragma unroll
        for (int mc = 0; mc < MC; mc++) sav[u][mc] = buf_load4(rsa, ok ? (uint32_t)mc * sa_cs + (uint32_t)lane * 4u : OOB, so * 256u);
        sbv[u] = buf_load4(rsb, ok ? (uint32_t)lane * 4u : OOB, so * 256u);
#pragma unroll
        for (int nb = 0; nb < 2; nb++)
#pragma unroll
            for (int kh = 0; kh < 2; kh++)
#pragma unroll
                for (int l = 0; l < BL; l++)
                    bq[u][nb][kh][l] = buf_load16_nt(rb, ok ? (uint32_t)lane * 16u + (uint32_t)nb * 16u * b_row_bytes + (uint32_t)l * 1024u : OOB, (so * 2u + (uint32_t)kh) * (16u * BB));
        // keep the machine scheduler from sinking these loads below later code to save registers
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_patch = [&](int s) __attribute__((always_inline)) {
        if constexpr (PATCH) {
#pragma unroll
            for (int ps = 0; ps < PASSES; ps++) dma16(ra, patch_lds + (uint32_t)ps * 1024u, dma_voff[ps % 4] + (uint32_t)(ps / 4 * 16) * a_rs, (uint32_t)s * 256u);
        }
    };
    auto compute = [&](auto SETP) __attribute__((always_inline)) {
        constexpr int u = decltype(SETP)::value;
        if constexpr (PATCH) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(BEHIND) : "memory");
        static_for<2>([&](auto KH) {
            constexpr int kh = decltype(KH)::value;
            static_for<MB>([&](auto MBI) {
                constexpr int mb = decltype(MBI)::value;
                v8i af;
                if constexpr (PATCH) {
                    const uint8_t* row = patch + (mb * 16 + li) * 256;
                    const int c0 = kh * 8 + (AF == MXF_FP6 ? 2 * lg : lg), c1 = kh * 8 + (AF == MXF_FP6 ? 2 * lg + 1 : 4 + lg);
                    const v4i x[2] = {*reinterpret_cast<const v4i*>(row + ((c0 ^ li) << 4)), *reinterpret_cast<const v4i*>(row + ((c1 ^ li) << 4))};
                    af = widen(x, std::integral_constant<int, AL>{});
                } else {
                    af = widen(aq[u][mb][kh], std::integral_constant<int, AL>{});
                }
                static_for<2>([&](auto NB) {
                    constexpr int nb = decltype(NB)::value;
                    acc[mb][nb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(widen(bq[u][nb][kh], std::integral_constant<int, BL>{}), af, acc[mb][nb], MxCode<BF>::value,
                                                                                  MxCode<AF>::value, kh * 2 + nb, sbv[u], kh * 2 + (mb & 1), sav[u][mb / 2]);
                });
            });
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    load_regs(s_begin, I0{});
    for (int s = s_begin; s < s_end; s += 2) {
        load_patch(s);
        load_regs(s + 1, I1{});
        compute(I0{});
        if (s + 1 < s_end) {
            load_patch(s + 1);
            load_regs(s + 2, I0{});
            compute(I1{});
        }
    }

    auto red = [&](int w) { return reinterpret_cast<v4f*>(lds + w * PW); };  // (the wavefront is done with its patch)
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        red(wave)[(mb * 2 + 0) * 64 + lane] = acc[mb][0];
        red(wave)[(mb * 2 + 1) * 64 + lane] = acc[mb][1];
    }
    __syncthreads();
    uint16_t* c = reinterpret_cast<uint16_t*>(static_cast<uint8_t*>(p.c) + z * (uint64_t)p.c_batch);
    for (int t = tid; t < MB * 2 * 64; t += NW * 64) {
        const int f = t >> 6, mb = f >> 1, nb = f & 1;
        // all partial sums are read in one batch (no wait between them), then added in slice order
        v4f part[NW];
#pragma unroll
        for (int j = 0; j < NW; j++) part[j] = red(j)[f * 64 + lane];
        v4f sum = part[0];
#pragma unroll
        for (int j = 1; j < NW; j++) sum += part[j];
        const int m = mb * 16 + li, n = np * 32 + nb * 16 + lg * 4;
        if (m < M) *reinterpret_cast<v2i*>(c + (int64_t)(m0 + m) * p.c_row_stride + n) = p.out == OUT_BF16 ? pack4_out16<OUT_BF16>(sum[0], sum[1], sum[2], sum[3]) : pack4_out16<OUT_FP16>(sum[0], sum[1], sum[2], sum[3]);
    }
}

template <int AF, int BF>
hipError_t launch_fmt(const MxGenParams& p, int batch, hipStream_t stream) {
    const int groups = (p.M + 63) / 64;  // of 64 rows
    const bool wide = p.K >= 2048;  // eight wavefronts once each has a whole step
#define PSG_GO(MB_)                                                                                                                     \
    if (wide) hipLaunchKernelGGL((k_mx_smallm<AF, BF, MB_, 8>), dim3(p.N / 32, groups, batch), dim3(512), 0, stream, p);                      \
    else hipLaunchKernelGGL((k_mx_smallm<AF, BF, MB_, 4>), dim3(p.N / 32, groups, batch), dim3(256), 0, stream, p);
    if (p.M <= 16) { PSG_GO(1) } else if (p.M <= 32) { PSG_GO(2) } else { PSG_GO(4) }
#undef PSG_GO
    return hipGetLastError();
}

}  // namespace

// 16-bit output, M >= 1 (meant for up to a few hundred rows, 64 a workgroup); af: MXF_FP4 / MXF_FP6 / MXF_FP8; bf: MXF_FP4 / MXF_FP8; batch >= 1 (grid.z <= 65535)
hipError_t psg_launch_mx_smallm(const MxGenParams& p, int af, int bf, int batch, hipStream_t stream) {
    if (bf == MXF_FP4) {
        if (af == MXF_FP4) return launch_fmt<MXF_FP4, MXF_FP4>(p, batch, stream);
        if (af == MXF_FP6) return launch_fmt<MXF_FP6, MXF_FP4>(p, batch, stream);
        return launch_fmt<MXF_FP8, MXF_FP4>(p, batch, stream);
    }
    if (af == MXF_FP4) return launch_fmt<MXF_FP4, MXF_FP8>(p, batch, stream);
    if (af == MXF_FP6) return launch_fmt<MXF_FP6, MXF_FP8>(p, batch, stream);
    return launch_fmt<MXF_FP8, MXF_FP8>(p, batch, stream);
}
