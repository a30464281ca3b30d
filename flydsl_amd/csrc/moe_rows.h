// Accumulation of the MoE down stage through one row per sorted position (moe_rows.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct MoeRowsParams {
    uint16_t* out;              // [tokens, dim] 16-bit, added into
    uint16_t* rows;             // [sorted_size, dim] weighted rows of the stage
    int* count;                 // [tokens] rows of each token, then the number of entries of `extra`
    int* list;                  // [tokens, topk] sorted positions of a token's rows
    int* extra;                 // sorted positions of rows past topk
    const int32_t* sorted_ids;
    const int32_t* expert_ids;
    const int32_t* num_valid;
    int tokens, topk, experts, dim, sorted_size, blocks, block_m;
    int slots;                  // ids with a slot number from here on are padding
    int granule;                // rows of the tiles the stage computes up to num_valid in
    int out_dtype;
};

uint64_t psg_moe_rows_bytes(int64_t tokens, int64_t topk, int64_t sorted_size, int64_t dim);
void psg_moe_rows_carve(MoeRowsParams& p, void* workspace);
hipError_t psg_launch_moe_rows_index(const MoeRowsParams& p, hipStream_t stream);
hipError_t psg_launch_moe_rows_add(const MoeRowsParams& p, hipStream_t stream);
