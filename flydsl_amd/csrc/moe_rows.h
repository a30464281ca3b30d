// Accumulation of the MoE down stage through one row per sorted position (moe_rows.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct MoeRowsParams {
    uint16_t* out;              // [tokens, dim] 16-bit, added into
    uint16_t* rows;             // [sorted_size, dim] weighted rows of the stage
    int* count;                 // [tokens] rows of each token
    int* list;                  // [tokens, topk] sorted positions of a token's rows
    int* next;                  // [sorted_size] behind the last entry of a full list: the token's rows past topk, chained, -1 at the end
    const int32_t* sorted_ids;
    const int32_t* expert_ids;
    const int32_t* num_valid;
    int tokens, topk, experts, dim, sorted_size, blocks;
    int block_m;                // a power of two
    int slots;                  // ids with a slot number from here on are padding
    int granule;                // rows of the tiles the stage computes up to num_valid in
    int out_dtype;
    int wgs;                    // workgroups (k_moe_gemm: rows of the grid) in front of a stage's tiles that make the lists; 0 = none
};

// Workgroups that make the lists above.  The stages have them in front of their own tiles, where they work beside
// these and cost no time of their own (behind the tiles their own 15 us are the end of the launch: MX stage 2, 4096 tokens x top-8, 242 us against
// 231).  (One launch that cleared the counts and another that entered the rows took 9.5 us, 1024 or 4096 tokens x top-8.  Whole layers, us before / now: int4 1052
// tokens x top-8, 1536 x 1024, 128 / 124; int8 813 x top-4, 4096 x 512, 140 / 135; MX 410 x top-8, 4096 x 1536, 140.6 / 134.6; 1500 x top-6, 2048 x 768, 99 /
// 93; 4096 x top-8 602 / 596.)  A multiple of 8 leaves every tile on its XCD.
constexpr int ROWS_INDEX_WGS = 32;

// Every one of those workgroups looks through the whole list, so their work grows with its square; longer lists are made by two launches over
// all CUs.  Beside the tiles of k_moe_gemm that is better from about 50,000 sorted rows on with blocks of 16 and 32 rows, 120,000 with 64 and 128 (us
// beside the tiles / two launches, top-8 on 32 experts, 2048 x 512, fp8: blocks of 16 6000 tokens 249 / 247, 8192 356 / 350, 30000 1329 / 1293; of 32 8192 283 /
// 282, 16384 582 / 574; of 64 8192 250 / 251, 12000 372 / 371, 16384 515 / 508, 30000 935 / 917; int4, 1024 x 256, 14000 tokens, blocks of 16, 64 and 128 268 / 263, 177 /
// 179, 184 / 189); beside the MX pair's and the 128x256 tiles, with their 16 ids a thread, it never is (MX 16384 tokens 394 / 402, 65536 1490 / 1492).
inline int moe_rows_share_max(int block_m) { return block_m <= 32 ? 50000 : 120000; }

uint64_t psg_moe_rows_bytes(int64_t tokens, int64_t topk, int64_t sorted_size, int64_t dim);
void psg_moe_rows_carve(MoeRowsParams& p, void* workspace);
hipError_t psg_launch_moe_rows_index(const MoeRowsParams& p, hipStream_t stream);
hipError_t psg_launch_moe_rows_add(const MoeRowsParams& p, hipStream_t stream);

// the rows the stage computes: whole tiles up to num_valid, in blocks that are in the list
__device__ __forceinline__ int moe_rows_limit(const MoeRowsParams& p) {
    const int nv = p.num_valid[0];
    int limit = nv >= p.sorted_size ? p.sorted_size : nv <= 0 ? 0 : (nv + p.granule - 1) / p.granule * p.granule;
    if (limit > p.sorted_size) limit = p.sorted_size;
    return (int64_t)p.blocks * p.block_m < limit ? p.blocks * p.block_m : limit;
}

// Share `wg` of `wgs` of the lists: a range of tokens, for which it looks through the whole sorted list (16 to 600 KB out of L2).  The counts stay in
// LDS (`lds`, two ints a token, `lds_ints` in all), so nothing has to be cleared before.
// B = ids, and experts of their blocks, that a thread asks for at a time (few enough that the stage keeps its registers: 16 of them in the 16-row down
// stage, 64 registers without, cost it two wavefronts a SIMD and the decode layer of 64 tokens 3 us)
template <int B>
__device__ __forceinline__ void moe_rows_index_share(const MoeRowsParams& p, int wg, int wgs, int* lds, int lds_ints) {
    const int tid = (int)threadIdx.x, nt = (int)blockDim.x;
    const int per = (p.tokens + wgs - 1) / wgs, first = wg * per, last = first + per < p.tokens ? first + per : p.tokens;
    const int cap = lds_ints / 2;
    int* cnt = lds;
    int* head = lds + cap;
    const int limit = moe_rows_limit(p);
    const int sh = __builtin_ctz(p.block_m);
    for (int t0 = first; t0 < last; t0 += cap) {
        const int n = last - t0 < cap ? last - t0 : cap;
        for (int i = tid; i < n; i += nt) {
            cnt[i] = 0;
            head[i] = -1;
        }
        __syncthreads();
        for (int i0 = 0; i0 < limit; i0 += nt * B) {
            uint32_t id[B];
            int e[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int i = i0 + j * nt + tid, at = i < limit ? i : 0;
                id[j] = (uint32_t)p.sorted_ids[at];
                e[j] = p.expert_ids[at >> sh];
            }
#pragma unroll
            for (int j = 0; j < B; j++) {
                const int i = i0 + j * nt + tid, t = (int)(id[j] & 0xFFFFFFu), at = t - t0;
                if (i >= limit || (unsigned)at >= (unsigned)n || (int)(id[j] >> 24) >= p.slots) continue;
                if ((unsigned)e[j] >= (unsigned)p.experts) continue;  // a block without an expert
                const int k = atomicAdd(&cnt[at], 1);
                if (k < p.topk - 1) p.list[(size_t)t * p.topk + k] = i;
                else p.next[i] = atomicExch(&head[at], i);
            }
        }
        __syncthreads();
        for (int i = tid; i < n; i += nt) {
            p.count[t0 + i] = cnt[i];
            if (cnt[i] >= p.topk) p.list[(size_t)(t0 + i) * p.topk + p.topk - 1] = head[i];
        }
        __syncthreads();
    }
}
