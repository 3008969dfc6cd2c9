// Gather/scatter description shared by the mixture-of-experts forms of the few-row GEMM kernels.
#pragma once

#include <cmath>

#include "fnn_common.h"

namespace fnn {

// Mixture-of-experts form of the few-row kernels: the activation rows of a pass are gathered through a
// sorted token list, every block of block_m sorted rows multiplies one expert's weight matrix, and
// the output rows are scattered back by token id (flashnn/triton_kernels/fused_moe_a8w8.py:37-173, fused_moe_a16w4.py:50-206).
struct MoeArgs {
    const int32_t* sorted_ids;   // [EM] token ids (index into the M*top_k routed rows); >= num_valid: padding
    const int32_t* expert_ids;   // [EM / block_m]
    const int32_t* ntpp;         // [1] number of sorted rows in use (a multiple of block_m)
    const void* topk_w;          // [M*top_k] routing weights, or unused
    int topk_w_dtype, mul_w, top_k, block_m, num_valid, EM;
    int64_t stride_be;           // bytes (= elements) between the weight matrices of two experts
    int64_t stride_scale_be;     // elements between the column scales of two experts
    int64_t stride_zp_be;        // ... and between their zero points (weight-only form)
    // weight-only form: element strides of scale[e, n, kblock] and zero_point[e, n, kblock]
    int64_t stride_scale_n, stride_scale_k, stride_zp_n, stride_zp_k;
};

// The tiles of BM sorted rows that a tiled kernel cuts the routed rows into.  Blocks of BM rows and more are cut into
// whole tiles.  Smaller blocks are put together: a tile is up to BM / block_m consecutive blocks of one expert, so the
// height of the tile - what decides how often an expert's weights are read, and how many operand bytes a CU takes in per
// output - does not hang on the block size that the caller sorted for.  Where an expert's blocks end, and so how many tiles
// there are, is read from expert_ids by every wave for itself: 64 blocks per step, four steps' loads in flight (256
// blocks: one L2 latency, about 1 us before a tile of 40 to 60 us, and as much again to find the tile).  Long lists of small
// blocks pay for it: 64 experts of N=2816 K=2048, 6 per token, 4096 tokens (1600 blocks of 16, 448 of 64), A8W8 270 us in blocks of
// 16 and 220 in blocks of 64.
// WHOLE: the caller knows that blocks are of BM rows and more; the search is not compiled in then.
template <int BM, bool WHOLE = false>
struct MoeTiles {
    const MoeArgs& q;
    const int lane;
    int blocks, tiles;       // blocks in use and tiles that they make

    __device__ __forceinline__ MoeTiles(const MoeArgs& args, int lane_) : q(args), lane(lane_) {
        const int used = min(q.ntpp[0], q.EM);
        blocks = __builtin_amdgcn_readfirstlane((used + q.block_m - 1) / q.block_m);
        tiles = WHOLE || q.block_m >= BM ? blocks * (q.block_m / BM) : scan(-1);
    }

    // the number of tiles (want < 0), or the first block of tile `want`
    __device__ __forceinline__ int scan(int want) const {
        const int r = BM / q.block_m;
        int count = 0, last_expert = 0, run = 0;        // run: first block of the expert's blocks that are being walked
        for (int base = 0; base < blocks; base += 256) {
            int e[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) e[c] = q.expert_ids[min(base + 64 * c + lane, blocks - 1)];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int first = base + 64 * c, blk = first + lane;
                if (first >= blocks) break;
                // the lane before's value (wave_shr:1 - a shuffle keeps the lane's byte address in a register over the tile)
                const int before = __builtin_amdgcn_update_dpp(0, e[c], 0x138, 0xF, 0xF, false);
                const bool starts = blk < blocks && (blk == 0 || e[c] != (lane == 0 ? last_expert : before));
                const uint64_t runs = __ballot(starts);
                const uint64_t here = runs & (~0ull >> (63 - lane));
                const int mine = here ? first + 63 - __clzll(here) : run;
                const uint64_t heads = __ballot(blk < blocks && (blk - mine) % r == 0);
                const int n = __popcll(heads);
                if (want >= 0 && want < count + n) {
                    const bool hit = (heads >> lane & 1) && __popcll(heads & ((1ull << lane) - 1)) == want - count;
                    return __builtin_amdgcn_readfirstlane(first + __ffsll((unsigned long long)__ballot(hit)) - 1);
                }
                count += n;
                last_expert = __builtin_amdgcn_readlane(e[c], 63);
                if (runs) run = first + 63 - __clzll(runs);
            }
        }
        return count;
    }

    // first sorted row of a tile, how many of its rows belong to it, and their expert
    __device__ __forceinline__ void find(int tile, int& m0, int& rows, int& expert) const {
        if (WHOLE || q.block_m >= BM) {
            m0 = tile * BM;
            rows = BM;
            expert = q.expert_ids[m0 / q.block_m];
        } else {
            const int r = BM / q.block_m, b = scan(tile);
            const int e = q.expert_ids[min(b + lane, blocks - 1)];
            expert = __builtin_amdgcn_readfirstlane(e);
            const uint64_t same = __ballot(lane < r && b + lane < blocks && e == expert);
            m0 = b * q.block_m;
            rows = (__ffsll((unsigned long long)~same) - 1) * q.block_m;
        }
    }
};

// What the host can say about the routing without reading it.  A sorted list as callers allocate it holds every routed row
// and block_m - 1 padding rows per expert, rounded up to whole blocks, which gives the number of experts.  A list cut to the
// rows in use has less padding: with less than one expert's worth it says nothing, and every block is then taken for an expert
// of its own, so that tiles stay within what the caller sorted for.  An estimate: used for grid sizes and prices only.
inline int64_t moe_experts_estimate(const MoeArgs& q) {
    const int64_t blocks = q.EM / q.block_m, pad = (int64_t)q.EM - q.num_valid;
    const int64_t e = q.block_m > 1 ? pad / (q.block_m - 1) : 0;
    return e >= 1 && e < blocks ? e : (blocks > 0 ? blocks : 1);
}
// ... and so the number of tiles of bm rows
inline int64_t moe_tiles_estimate(const MoeArgs& q, int bm) {
    const int64_t blocks = q.EM / q.block_m;
    if (q.block_m >= bm) return blocks * (q.block_m / bm);
    const int64_t t = (q.num_valid + bm - 1) / bm + moe_experts_estimate(q);
    return t < blocks ? t : blocks;
}
// ... and the rounds of tiles of bm rows x bn of n channels that a call makes with per_round of them at a time, the rows of an
// expert taken as spread round their mean the way an even random routing spreads them
inline double moe_rounds(const MoeArgs& q, int n, int bm, int bn, int per_round) {
    const double experts = (double)moe_experts_estimate(q), mean = (double)q.num_valid / experts, off = 1.2 * sqrt(mean);
    const double tall = (ceil((mean - off) / bm) + ceil(mean / bm) + ceil((mean + off) / bm)) / 3.0;
    return experts * tall * ((n + bn - 1) / bn) / per_round;
}

}  // namespace fnn
