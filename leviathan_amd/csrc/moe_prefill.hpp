// Interface between the MoE entry points and the grouped matrix product for prompts and large batches.
#pragma once

#include "moe_grouped.hpp"

// A work item: `count` (1..64) pairs of one expert, entries first .. of the expert-ordered pair list.
struct alignas(16) lev_pf_item {
    int32_t expert, first, count, pad;
};

size_t lev_moe_prefill_scratch_bytes(const lev_moe_grouped_args &a);
// Geometry it serves (the caller also checks 4-byte aligned pools and 16-byte aligned x).
bool lev_moe_prefill_usable(const lev_moe_grouped_args &a);
// act: f32 [tokens*top_k][inter] (written here, read by the down stage).
hipError_t lev_moe_prefill_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const float *x, const int32_t *ids,
                                  const float *weights, float *y, float *act, void *scratch);
