// What the fusions of recorded programs (lev_api.hip) know of the kernels of other files: which function of a kernel node is
// which, the memory that it touches, and the launches that stand for two of them.
#pragma once

#include "lev_common.hpp"

struct lev_span {
    uintptr_t at = 0;
    size_t bytes = 0;
    lev_span() = default;
    template <typename T>
    lev_span(const T *p, size_t n) : at(reinterpret_cast<uintptr_t>(p)), bytes(p ? n : 0u) {}
    bool meets(const lev_span &o) const { return at < o.at + o.bytes && o.at < at + bytes; }
};

// The memory of one kernel.
struct lev_footprint {
    lev_span reads[8], writes[4];
    // neither writes what the other touches: they may change places or run side by side
    bool apart(const lev_footprint &o) const {
        for (const lev_span &w : writes) {
            for (const lev_span &r : o.reads)
                if (w.meets(r)) return false;
            for (const lev_span &v : o.writes)
                if (w.meets(v)) return false;
        }
        for (const lev_span &w : o.writes)
            for (const lev_span &r : reads)
                if (w.meets(r)) return false;
        return true;
    }
};

struct lev_gemv_args {
    const uint8_t *w;
    const float *x;
    float *y;
    uint32_t in_dim, rows, wpr, slots;
    uint64_t slot_of_wave, pos_of_wave;
};
struct lev_scores_args {
    const float *wr, *x;
    float *scores;
    uint32_t hidden, experts;
};
struct lev_fused_launch {
    void *func;
    uint32_t blocks, threads, lds;
};

const void *lev_q4_0_gemv_one_round();     // q4_0_mfma_gemv<1, true, false>: the arguments of lev_gemv_args in order
const void *lev_moe_scores_few();          // moe_scores_few_kernel: those of lev_scores_args
lev_fused_launch lev_q4_0_gemv_and_scores(uint32_t gemv_blocks, uint32_t gemv_threads, uint32_t experts);
// Whether `func` is one of the MoE layer's kernels at one token (gate/up, down), and what it touches.
bool lev_moe_expert_node(const lev_ctx *ctx, const void *func, void **args, lev_footprint *touches);

// What follows an RMSNorm in a recorded program: y += c[k] * x[k], in order.
struct lev_norm_adds {
    static constexpr int kMost = 4;
    const float *x[kMost];
    float c[kMost];
    int count;
};
// The norm and adds (two at most) that make the input of an FFN: out = rmsnorm(y) * wy + adds, where adds number `own` is
// rmsnorm(s) * ws unless s is null.
struct lev_norm_front {
    static constexpr int kMost = 2;
    const float *y, *wy, *s, *ws;
    float *out;
    lev_norm_adds adds;
    float eps, eps_s;
    int own;
};
// s = rmsnorm(s) * ws, of n values
struct lev_norm_tail {
    float *s;
    const float *ws;
    uint32_t n;
    float eps;
};

struct lev_ffn_args {
    const uint8_t *gate, *up;
    const float *x, *gain;
    float *h, *gu, *act;
    uint32_t hidden, inter, rows_per_block;
    float eps;
};
// The first kernel of the shared expert's FFN: its arguments, what it touches, and the launches (without their number of
// workgroups) that compute the router's scores of h as well: arguments lev_ffn_args, lev_scores_args, its own workgroups;
// with_front: lev_norm_front behind them, in whose place x is.
struct lev_ffn_node {
    lev_ffn_args args;
    lev_footprint touches;
    lev_fused_launch with_scores, with_front;
};
bool lev_ffn_gate_up_node(const void *func, void **args, lev_ffn_node *out);

// The launch of the MoE layer's gate/up kernel of one token with a GEMV of one round beside it: `args` of the former with
// rows_per_block, then *g (its slots are those of the launch), extra, gemv_blocks, a lev_norm_tail; grid (launch.blocks, top_k).
struct lev_gate_up_gemv {
    lev_fused_launch launch;
    uint32_t rows_per_block, extra, gemv_blocks, top_k;
};
bool lev_moe_gate_up_and_gemv(const lev_ctx *ctx, const void *func, void **args, lev_gemv_args *g, lev_gate_up_gemv *out);
bool lev_moe_gate_up_and_gemv_is(const void *func);
// Gives such a launch its tail, which one more workgroup (of a slot) does.
hipError_t lev_moe_gate_up_and_gemv_tail(hipGraphNode_t node, const lev_norm_tail &tail);
