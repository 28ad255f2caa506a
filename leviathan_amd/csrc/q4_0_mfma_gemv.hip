// Q4_0 decode GEMV  y = W x  on the integer matrix cores (gfx950).
//
// Stands in for g4_q4_matvec and its tiled / generated variants
// (Sources/LeviathanCore/Gemma4.swift:3931, 4031; Q4Lowering.swift:541-664) for the rows that
// lev_q4_0_mfma_in_dim names; q4_0_gemv.hip keeps the vector-ALU kernels for every other shape and as forge candidates.  The last 256-value task of a row may be a part of one: 2112 columns, 20000 rows 6.8 us a call
// against 8.0 with the vector-ALU kernel, 8000 x 9000 9.9 against 12.9.
//
// Workgroup = 16 waves.  A row group is 16 rows; its in_dim / 256 column tasks are split over
// WPR waves, TPW adjacent tasks each (WPR * TPW >= tasks).  Rows narrower than 16 tasks leave
// room for 16 / WPR row groups per round of the workgroup.  A wave stages the activations of its
// own tasks once, keeps the operands in registers and walks the row groups of its slot with the
// next group's weights in flight; the WPR partial sums of a row meet in LDS behind ONE barrier a
// round, and the wave of the slot adds them in a fixed order.
//
// Rows of an odd number of blocks (ODD).  Every other row starts 18 bytes, half a pair, off the 36-byte grid on which
// pairs are dword aligned.  The kernel keeps to that grid: the matrix is taken as two, its even rows and its odd ones,
// half of the workgroups on each.  An even row's last pair is half its own, an odd row's first pair is, and the
// activations of the odd rows are one block late, so that within a row group everything is where it is for whole pairs;
// the scale of the block that belongs to a neighbour is taken as zero.  2400 x 17715 26.7 us with 2-byte loads, 7 here.
#include "moe_scores_few.hpp"
#include "program_nodes.hpp"
#include "q4_0_mfma_gemv.hpp"

namespace {

template <int TPW, bool SINGLE, bool ODD>
__global__ void __launch_bounds__(kQ4mThreads)
q4_0_mfma_gemv(const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ y,
               uint32_t in_dim, uint32_t rows, uint32_t wpr, uint32_t slots, uint64_t slot_of_wave,
               uint64_t pos_of_wave) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    q4m_gemv<TPW, SINGLE, ODD>(w, x, y, in_dim, rows, wpr, slots, slot_of_wave, pos_of_wave, blockIdx.x, gridDim.x, smem);
}

// A GEMV of one round and the router scores of one token, which do not depend on each other (recorded programs): the first
// `gemv_blocks` workgroups are those of q4_0_mfma_gemv<1, true, false>, the others take blockDim.x / 256 experts each.
// The down projection of a shared expert and the scores behind it, 2112 x 2816 and 128 x 2816: 3.0 and 2.8 us as two
// launches in a row.
__global__ void __launch_bounds__(kQ4mThreads)
q4_0_gemv_and_scores(lev_gemv_args g, lev_scores_args r, uint32_t gemv_blocks) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    if (blockIdx.x < gemv_blocks) {
        q4m_gemv<1, true, false>(g.w, g.x, g.y, g.in_dim, g.rows, g.wpr, g.slots, g.slot_of_wave, g.pos_of_wave, blockIdx.x, gemv_blocks, smem);
        return;
    }
    const uint32_t each = blockDim.x >> 8, part = threadIdx.x >> 8, e = (blockIdx.x - gemv_blocks) * each + part;
    moe_score_few(r.wr, r.x, r.scores, r.hidden, r.experts, part < each ? e : r.experts, 0u, threadIdx.x & 255u,
                  reinterpret_cast<double *>(smem) + 4u * part);
}

template <int TPW, bool SINGLE, bool ODD>
hipError_t launch_grid(lev_ctx *ctx, const uint8_t *w, const float *x, float *y, uint32_t in_dim, uint32_t rows,
                       uint32_t wpr, uint32_t slots, uint32_t blocks) {
    constexpr size_t lds = q4m_gemv_lds(TPW);
    uint64_t slot_of_wave, pos_of_wave;
    lev_wave_tables(wpr, &slot_of_wave, &pos_of_wave);
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&q4_0_mfma_gemv<TPW, SINGLE, ODD>), lds); e != hipSuccess) return e;
    hipLaunchKernelGGL((q4_0_mfma_gemv<TPW, SINGLE, ODD>), dim3(blocks), dim3(slots * wpr * LEV_WAVE), lds, ctx->stream, w, x, y,
                       in_dim, rows, wpr, slots, slot_of_wave, pos_of_wave);
    return hipGetLastError();
}

// How the shape is split: tasks a wave (TPW), waves a row, row groups (slots) a round, rounds of each part of the
// matrix (two parts where rows alternate) and the workgroups of a part that stay resident.  A workgroup has no more waves
// than have work: rows of 17 to 20 tasks, two a wave, leave room for a second workgroup on the CU (20000 x 5120 14 us
// with sixteen waves, 10.8 with ten).
struct split {
    uint32_t tpw, wpr, slots, parts, nrounds, resident;
    bool single;
};
split split_of(const lev_ctx *ctx, uint32_t in_dim, uint32_t rows) {
    split s;
    const uint32_t ntask = (in_dim + 255u) >> 8, cus = (uint32_t)ctx->num_cus;
    s.tpw = (ntask + (uint32_t)kQ4mWaves - 1u) / (uint32_t)kQ4mWaves;
    s.wpr = (ntask + s.tpw - 1u) / s.tpw;
    s.slots = (uint32_t)kQ4mWaves / s.wpr;
    s.parts = in_dim % 64u != 0u ? 2u : 1u;
    const uint32_t ngroups = ((rows + s.parts - 1u) / s.parts + 15u) / 16u;
    s.nrounds = (ngroups + s.slots - 1u) / s.slots;
    // One workgroup a round while all of them are on the chip at once (two a CU where ten waves are all they have);
    // and always with more than two tasks a wave, whose registers have no room for the next group's weights.
    const uint32_t per_cu = s.slots * s.wpr <= 10u ? 2u : 1u;
    s.single = s.tpw > 2u || s.nrounds * s.parts <= cus * per_cu;
    s.resident = cus * (s.tpw == 1u ? per_cu : 1u) / s.parts;
    if (s.resident == 0u) s.resident = 1u;
    return s;
}

template <int TPW, bool ODD>
hipError_t launch(lev_ctx *ctx, const uint8_t *w, const float *x, float *y, uint32_t in_dim, uint32_t rows,
                  const split &s, int persistent) {
    if constexpr (TPW <= 2)
        if (persistent < 0 ? !s.single : persistent != 0)
            return launch_grid<TPW, false, ODD>(ctx, w, x, y, in_dim, rows, s.wpr, s.slots,
                                                (s.nrounds < s.resident ? s.nrounds : s.resident) * s.parts);
    return launch_grid<TPW, true, ODD>(ctx, w, x, y, in_dim, rows, s.wpr, s.slots, s.nrounds * s.parts);
}

}  // namespace

bool lev_q4_0_mfma_gemv_usable(const uint8_t *w, const float *x, uint32_t in_dim, bool narrow) {
    return (lev_q4_0_mfma_in_dim(in_dim) || (narrow && in_dim != 0u && in_dim % 64u == 0u && in_dim <= 1280u)) && (reinterpret_cast<uintptr_t>(w) & 3u) == 0u &&
           (reinterpret_cast<uintptr_t>(x) & 15u) == 0u;
}

// persistent: 0 = one workgroup per round of row groups, 1 = resident grid, < 0 = built-in choice.
hipError_t lev_q4_0_mfma_gemv_launch(lev_ctx *ctx, const uint8_t *w, const float *x, float *y, uint32_t in_dim,
                                     uint32_t rows, int persistent) {
    const split s = split_of(ctx, in_dim, rows);
    if (in_dim % 64u != 0u) {
        switch (s.tpw) {
            case 1: return launch<1, true>(ctx, w, x, y, in_dim, rows, s, persistent);
            case 2: return launch<2, true>(ctx, w, x, y, in_dim, rows, s, persistent);
            case 3: return launch<3, true>(ctx, w, x, y, in_dim, rows, s, persistent);
            default: return launch<4, true>(ctx, w, x, y, in_dim, rows, s, persistent);
        }
    }
    if (s.tpw == 1u) return launch<1, false>(ctx, w, x, y, in_dim, rows, s, persistent);
    return launch<2, false>(ctx, w, x, y, in_dim, rows, s, persistent);
}

// The built-in choice as `persistent` (0 or 1), and whether there is another one to choose.
void lev_q4_0_mfma_gemv_choice(const lev_ctx *ctx, uint32_t in_dim, uint32_t rows, uint32_t *persistent, bool *other) {
    const split s = split_of(ctx, in_dim, rows);
    *persistent = s.single ? 0u : 1u;
    *other = s.tpw <= 2u;
}

const void *lev_q4_0_gemv_one_round() { return reinterpret_cast<const void *>(&q4_0_mfma_gemv<1, true, false>); }

lev_fused_launch lev_q4_0_gemv_and_scores(uint32_t gemv_blocks, uint32_t gemv_threads, uint32_t experts) {
    const uint32_t threads = gemv_threads < 256u ? 256u : gemv_threads, each = threads / 256u;
    return lev_fused_launch{reinterpret_cast<void *>(&q4_0_gemv_and_scores), gemv_blocks + (experts + each - 1u) / each, threads,
                            (uint32_t)q4m_gemv_lds(1u)};
}
