// Accumulation of the down stage by way of one row per sorted position (gfx950): the stage stores its weighted 16-bit rows to
// a scratch buffer, and every token then sums its rows in fp32 and adds the sum into `out` once.
//
// Bound: the additions.  Packed 16-bit atomics run at about 0.65 TB/s whatever multiplies in front of them (4096 tokens x top-8,
// model 4096, i.e. 268 MB of additions: fp8 stage 2 434 us, MX-FP4 436), a store and a read of the same rows at 5.  So `topk`
// additions per output element become one; that one stays atomic, because launches on other streams may be adding into `out` too.
//
// The rows are written once and read once, non-temporally on both sides (stages on 128-row tiles), so that they don't push the operands out of the caches: MX stage 2 and the sum, us before / now,
// 4096 tokens x top-8 on 32 experts, 4096 x 1536 236 / 213 (weights in the last-level cache 236 / 175), inter 512 on 64 experts 177 / 159, 1024 tokens 73.3 / 72.0; with one side alone 218 and 223.
//
// Which sorted rows belong to a token is found on the device, by workgroups beside the stage's tiles (moe_rows_index_share) or in launches in front, so any sorted
// list the atomic epilogue accepts works here: rows are entered into a list of `topk` places per token, and rows that do not fit (a
// list that names a token more often than topk times) are chained behind its last entry.
#include "psg_common.h"
#include "moe_rows.h"

namespace {

typedef __fp16 v2h_t __attribute__((ext_vector_type(2)));
typedef __bf16 v2b_t __attribute__((ext_vector_type(2)));

constexpr int DWORDS = 4;       // dword columns per thread: 256 threads cover 2048 16-bit columns

__device__ __forceinline__ void add_packed(uint32_t* o, int bits, int out_dtype) {
    if (out_dtype == OUT_BF16) __builtin_amdgcn_global_atomic_fadd_v2bf16((__attribute__((address_space(1))) v2b_t*)o, __builtin_bit_cast(v2b_t, bits));
    else __builtin_amdgcn_global_atomic_fadd_v2f16((__attribute__((address_space(1))) v2h_t*)o, __builtin_bit_cast(v2h_t, bits));
}

// The same lists by all CUs, from counts and heads in memory (a list's last place is the head of its chain).
__global__ void __launch_bounds__(256) k_moe_rows_clear(MoeRowsParams p) {
    const int t = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (t >= p.tokens) return;
    p.count[t] = 0;
    p.list[(size_t)t * p.topk + p.topk - 1] = -1;
}
__global__ void __launch_bounds__(256) k_moe_rows_enter(MoeRowsParams p) {
    const int i = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (i >= moe_rows_limit(p) || (unsigned)p.expert_ids[i / p.block_m] >= (unsigned)p.experts) return;
    const uint32_t id = (uint32_t)p.sorted_ids[i];
    const int t = (int)(id & 0xFFFFFFu);
    if (t >= p.tokens || (int)(id >> 24) >= p.slots) return;
    const int k = atomicAdd(&p.count[t], 1);
    int* list = p.list + (size_t)t * p.topk;
    if (k < p.topk - 1) list[k] = i;
    else p.next[i] = atomicExch(&list[p.topk - 1], i);
}

template <int OUT>
__global__ void __launch_bounds__(256) k_moe_rows_add(MoeRowsParams p, int chunks) {
    const int dws = p.dim >> 1;
    const int unit = (int)blockIdx.x / chunks;
    const int c0 = ((int)blockIdx.x % chunks) * (256 * DWORDS) + (int)threadIdx.x;
    const uint32_t* rows = reinterpret_cast<const uint32_t*>(p.rows);
    uint32_t* out = reinterpret_cast<uint32_t*>(p.out);
    const int count = p.count[unit], n = count < p.topk ? count : p.topk;
    if (n <= 0) return;
    const int* list = p.list + (size_t)unit * p.topk;
    float lo[DWORDS] = {}, hi[DWORDS] = {};
    auto add4 = [&](const int* list, auto CNT) {
        constexpr int N = decltype(CNT)::value;
        uint32_t v[N][DWORDS];
#pragma unroll
        for (int k = 0; k < N; k++) {
            const size_t base = (size_t)__builtin_amdgcn_readfirstlane(list[k]) * dws;
#pragma unroll
            for (int j = 0; j < DWORDS; j++) {
                const int c = c0 + j * 256;
                v[k][j] = __builtin_nontemporal_load(&rows[base + (c < dws ? c : 0)]);
            }
        }
#pragma unroll
        for (int k = 0; k < N; k++)
#pragma unroll
            for (int j = 0; j < DWORDS; j++) {
                lo[j] += from_out16<OUT>((uint16_t)(v[k][j] & 0xFFFF));
                hi[j] += from_out16<OUT>((uint16_t)(v[k][j] >> 16));
            }
    };
    int k = 0;
    for (; k + 8 <= n; k += 8) add4(list + k, std::integral_constant<int, 8>{});
    for (; k + 2 <= n; k += 2) add4(list + k, std::integral_constant<int, 2>{});
    if (k < n) add4(list + k, std::integral_constant<int, 1>{});
    if (count > p.topk)  // uniform
        for (int pos = p.next[list[p.topk - 1]], left = count - p.topk; left > 0; pos = p.next[pos], left--) add4(&pos, std::integral_constant<int, 1>{});
#pragma unroll
    for (int j = 0; j < DWORDS; j++) {
        const int c = c0 + j * 256;
        if (c < dws) add_packed(out + (size_t)unit * dws + c, pack2_out16<OUT>(lo[j], hi[j]), OUT);
    }
}

uint64_t up16(uint64_t v) { return (v + 15) & ~15ull; }

}  // namespace

uint64_t psg_moe_rows_bytes(int64_t tokens, int64_t topk, int64_t sorted_size, int64_t dim) {
    return up16((uint64_t)sorted_size * dim * 2) + up16((uint64_t)(tokens + 1) * 4) + up16((uint64_t)tokens * topk * 4) + (uint64_t)sorted_size * 4;
}

void psg_moe_rows_carve(MoeRowsParams& p, void* workspace) {
    uint8_t* w = static_cast<uint8_t*>(workspace);
    p.rows = reinterpret_cast<uint16_t*>(w);
    w += up16((uint64_t)p.sorted_size * p.dim * 2);
    p.count = reinterpret_cast<int*>(w);
    w += up16((uint64_t)(p.tokens + 1) * 4);
    p.list = reinterpret_cast<int*>(w);
    w += up16((uint64_t)p.tokens * p.topk * 4);
    p.next = reinterpret_cast<int*>(w);
}

// the lists in launches of their own, where the stage does not make them beside its tiles
hipError_t psg_launch_moe_rows_index(const MoeRowsParams& p, hipStream_t stream) {
    hipLaunchKernelGGL(k_moe_rows_clear, dim3((p.tokens + 255) / 256), dim3(256), 0, stream, p);
    hipLaunchKernelGGL(k_moe_rows_enter, dim3((p.sorted_size + 255) / 256), dim3(256), 0, stream, p);
    return hipGetLastError();
}

hipError_t psg_launch_moe_rows_add(const MoeRowsParams& p, hipStream_t stream) {
    const int chunks = (p.dim / 2 + 256 * DWORDS - 1) / (256 * DWORDS);
    const dim3 grid((unsigned)p.tokens * (unsigned)chunks);
    if (p.out_dtype == OUT_BF16) hipLaunchKernelGGL((k_moe_rows_add<OUT_BF16>), grid, dim3(256), 0, stream, p, chunks);
    else hipLaunchKernelGGL((k_moe_rows_add<OUT_FP16>), grid, dim3(256), 0, stream, p, chunks);
    return hipGetLastError();
}
