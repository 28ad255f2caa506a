// Interface between the MoE entry points and the many-token (grouped,
// matrix-core) expert path.
#pragma once

#include "lev_common.hpp"

struct lev_moe_grouped_args {
    const uint8_t *base;
    uint64_t gate_off, up_off, down_off;
    uint64_t gate_stride, up_stride, down_stride;
    uint32_t hidden, inter, experts, top_k, tokens;
};

// A work item of the integer matrix-core kernels: `count` (1..8) pairs of one expert, the pairs
// `first ..` of the expert-ordered list.  pair[k] is the (token * top_k + slot) index of column k,
// src[k] its token; columns past `count` repeat the last.
struct alignas(16) lev_grp_item {
    int32_t expert, count, first, pad;
    int32_t pair[8], src[8];
};

// Where a workgroup of the integer matrix-core kernels starts: its stretch of the line of rounds
// and the header of the first item it touches (one load in front of the first weight request
// instead of three that depend on each other).
struct alignas(32) lev_grp_start {
    uint32_t first_round, end_round, item;
    int32_t expert, count;
    uint32_t pad[3];
};

// Whether the many-token path takes the call (the caller also checks 4-byte aligned pools and x).
bool lev_moe_grouped_usable(const lev_ctx *ctx, const lev_moe_grouped_args &a, bool selects);
size_t lev_moe_grouped_scratch_bytes(const lev_ctx *ctx, const lev_moe_grouped_args &a);
// act: f32 [tokens*top_k][inter] (written here, read by the down stage).
hipError_t lev_moe_grouped_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const float *x,
                                  const int32_t *ids, const float *weights, float *y, float *act,
                                  void *scratch);
// y[t] = sum over slots, in slot order, of weights * dn (f32 [pair][hidden]); pairs that are not valid add zero.
hipError_t lev_moe_merge_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const float *dn, const float *weights,
                                const uint8_t *valid, float *y);

// Exclusive scan over a workgroup of 1024 threads, of sums that do not meet beyond 64 bits (fields of counts): what the threads
// in front of this one hold, and what all hold.  s_wave: 16 entries in LDS.  One barrier, between their stores and their reads: the
// caller needs another one before it writes s_wave again.  The steps within a wave are DPP
// moves: with lane permutations through the LDS they were most of what the grouping kernels' scan took.
__device__ __forceinline__ void lev_scan_1024(uint64_t own, uint64_t *s_wave, uint64_t &before, uint64_t &all) {
    uint32_t lo = (uint32_t)own, hi = (uint32_t)(own >> 32);
#define LEV_SCAN_STEP(CTRL, ROWS)                                                                                         \
    {                                                                                                                     \
        const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo, CTRL, ROWS, 0xF, false);                     \
        const uint32_t h = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, CTRL, ROWS, 0xF, false);                     \
        const uint64_t v = ((uint64_t)hi << 32 | lo) + ((uint64_t)h << 32 | l);                                           \
        lo = (uint32_t)v, hi = (uint32_t)(v >> 32);                                                                       \
    }
    LEV_SCAN_STEP(0x111, 0xF)   // row_shr:1, 2, 4, 8
    LEV_SCAN_STEP(0x112, 0xF)
    LEV_SCAN_STEP(0x114, 0xF)
    LEV_SCAN_STEP(0x118, 0xF)
    LEV_SCAN_STEP(0x142, 0xA)   // row_bcast:15 into rows 1 and 3
    LEV_SCAN_STEP(0x143, 0xC)   // row_bcast:31 into rows 2 and 3
#undef LEV_SCAN_STEP
    const uint64_t incl = (uint64_t)hi << 32 | lo;
    const uint32_t wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 63u) s_wave[wave] = incl;
    lev_barrier_lds();
    before = incl - own;
    all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16u; ++w) {
        const uint64_t v = s_wave[w];
        before += w < wave ? v : 0u;
        all += v;
    }
}
