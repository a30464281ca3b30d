// The sorted blocks of a MoE routing as a workgroup of the stages sees them.
#pragma once
#include "psg_common.h"

namespace {

// What a workgroup looks at to decide how it reads W (moe_reads_once): asked for in one go with the block's own expert, so that it costs no latency of its own.
struct MoeNeighbours {
    int before, after;  // experts of the blocks in front of the tile and behind it
    int first[2];       // experts of the blocks `lane` and 64 + lane
};
__device__ __forceinline__ MoeNeighbours moe_neighbours(const int32_t* expert_ids, int blocks, int blk, int per_tile, int lane) {
    const int last = blocks - 1;
    return {expert_ids[blk > 0 ? blk - 1 : 0], expert_ids[blk + per_tile < last ? blk + per_tile : last], {expert_ids[lane < last ? lane : last], expert_ids[64 + lane < last ? 64 + lane : last]}};
}

// Whether the W that the tile of `per_tile` blocks from `blk` on reads is read this once until it is gone from the last-level cache anyway: no other tile of its expert, and
// more than `cached` experts with rows among the `n` blocks in use (of a list grouped by expert; whatever the list, the results are the same).  Uniform over the workgroup.
__device__ __forceinline__ bool moe_reads_once(const MoeNeighbours& b, const int32_t* expert_ids, int n, int blk, int per_tile, int e, int experts, int cached, int lane) {
    if ((blk > 0 && b.before == e) || (blk + per_tile < n && b.after == e)) return false;
    int seen = 0, last = -1;
    auto count = [&](int v) {  // of 64 blocks
        int prev = __shfl_up(v, 1);
        if (lane == 0) prev = last;
        seen += __builtin_popcountll(__ballot((unsigned)v < (unsigned)experts && v != prev));
        last = __builtin_amdgcn_readlane(v, 63);
    };
    count(lane < n ? b.first[0] : -1);
    count(64 + lane < n ? b.first[1] : -1);
    for (int base = 128; base < n && seen <= cached; base += 64) count(base + lane < n ? expert_ids[base + lane] : -1);
    return seen > cached;
}

// Experts whose weights, both stages together, the last-level cache (256 MB) holds; bytes: of one expert's weights in `stage`
inline int moe_experts_cached(int stage, int64_t bytes) { return (int)(((2ll * (256 << 20)) - 1) / (bytes * (stage == 1 ? 3 : 6))); }

}  // namespace
