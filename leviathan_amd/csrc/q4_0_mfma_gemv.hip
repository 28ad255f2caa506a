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
#include "q4_0_mfma.hpp"

namespace {

constexpr int kQ4mWaves = 16;
constexpr int kQ4mThreads = kQ4mWaves * LEV_WAVE;

// LDS: part [2][16 waves][16 rows] f32 (2 KB, so that the round's half is one XOR away) | per
// wave TPW task areas and a zero strip
__host__ __device__ constexpr size_t q4m_gemv_lds(uint32_t tpw) {
    return 2u * kQ4mWaves * 16u * 4u + (size_t)kQ4mWaves * (tpw * kQ4mTaskArea + kQ4mZeroBytes);
}

// wave -> (slot, position in the slot): 4-bit entries of two 64-bit kernel arguments (lev_wave_tables).
// SINGLE: the grid covers every round once: straight-line code, nothing to prefetch.
template <int TPW, bool SINGLE, bool ODD>
__global__ void __launch_bounds__(kQ4mThreads)
q4_0_mfma_gemv(const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ y,
               uint32_t in_dim, uint32_t rows, uint32_t wpr, uint32_t slots, uint64_t slot_of_wave,
               uint64_t pos_of_wave) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    // wave-uniform by construction: in a scalar register, so that everything derived from it is
    // scalar arithmetic
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t slot = (uint32_t)(slot_of_wave >> (4u * wave)) & 15u;   // idle waves: slot >= slots
    const uint32_t tw = (uint32_t)(pos_of_wave >> (4u * wave)) & 15u;
    const uint32_t npairs = (in_dim + 63u) >> 6, ntask = (npairs + 3u) >> 2;   // the last task may be a part of one
    const uint32_t t_first = tw * TPW;
    // ODD: the workgroup's half of the matrix, rows parity, parity + 2, ...
    const uint32_t parity = ODD ? blockIdx.x & 1u : 0u;
    const uint32_t block = ODD ? blockIdx.x >> 1 : blockIdx.x, nblocks = ODD ? gridDim.x >> 1 : gridDim.x;
    const uint32_t nrows = ODD ? (rows + 1u - parity) >> 1 : rows;
    if (ODD && nrows == 0u) return;                              // a one-row matrix has no odd rows

    // the activations of the wave's tasks first (short, mostly L2 hits) ...
    lev_f32x4 v[TPW];
    bool v_live[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const uint32_t T = t_first + t < ntask ? t_first + t : ntask - 1u;
        v[t] = q4m_load_activations(x, T, in_dim >> 2, v_live[t], 8u * parity);
    }
    // ... the first row group's weights right behind them
    const bool active = slot < slots;
    const uint64_t row_bytes = (uint64_t)(in_dim >> 5) * 18u;
    const uint64_t row_step = ODD ? 2u * row_bytes : row_bytes;
    const uint8_t *const w0 = parity ? w + row_bytes - 18u : w;
    const uint8_t *const w_end = w + rows * row_bytes;
    const uint32_t ngroups = (nrows + 15u) >> 4;
    const uint32_t lrow = lane >> 2;                             // fetch order: lane = 4 * row + pair
    // bytes of a row in front of the lane's pair, past the row's end its last one, once for all rounds (8192 x 8192 10.53
    // us with the clamp in every round, 10.45 without; 20000 x 5120 12.99 and 12.84)
    uint32_t at[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const uint32_t T = t_first + t < ntask ? t_first + t : ntask - 1u, pair = 4u * T + (lane & 3u);
        at[t] = (pair < npairs ? pair : npairs - 1u) * 36u;
        if (!SINGLE) lev_pin(at[t]);
    }
    auto issue = [&](uint32_t round_block, uint32_t (&D)[TPW][9]) {
        uint32_t rg = round_block * slots + (active ? slot : 0u);
        rg = rg < ngroups ? rg : ngroups - 1u;
        uint32_t row = rg * 16u + lrow;
        row = row < nrows ? row : nrows - 1u;
        const uint8_t *rowp = w0 + (uint64_t)row * row_step;
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            const uint32_t T = t_first + t < ntask ? t_first + t : ntask - 1u;
            if (ODD)
                q4m_load_task_odd(rowp, 4u * T, npairs, w_end, D[t]);
            else
                lev_q4_load_pair(rowp + at[t], D[t]);
        }
    };
    uint32_t Da[TPW][9];
    uint32_t rb = block;
    issue(rb, Da);

    // ---- everything the tail of a round needs, while the loads are on their way ----
    uint8_t *area = smem + 2u * kQ4mWaves * 16u * 4u + (size_t)wave * (TPW * kQ4mTaskArea + kQ4mZeroBytes);
    uint8_t *zero = area + TPW * kQ4mTaskArea;                  // the wave's own: no barrier before the staging
    const uint32_t r = lane & 15u, q = lane >> 4;
    // the wave's partial sums: lanes 0..15 write row `lane`
    // (byte offsets into the workgroup's LDS, not pointers: an address that has been through an
    // integer register is no longer known to be LDS)
    uint32_t pw = (wave * 16u + lane) * 4u;
    // wave s < slots adds the wpr partial sums of slot s: lane (r, q) reads waves q, q + 4, q + 8, q + 12
    // of the slot (those past the slot's waves are masked after the read)
    uint32_t pr = (((wave < slots ? wave : 0u) * wpr + q) * 16u + r) * 4u;
    uint32_t k0 = q < wpr ? ~0u : 0u, k1 = q + 4u < wpr ? ~0u : 0u, k2 = q + 8u < wpr ? ~0u : 0u,
             k3 = q + 12u < wpr ? ~0u : 0u;
    uint32_t orow = (rb * slots + wave) * 16u + r;
    const uint32_t orow_step = nblocks * slots * 16u;
    const bool writer = wave < slots && q == 0u;
    uint32_t stores = writer && orow < nrows ? 1u : 0u;
    uint64_t yp = reinterpret_cast<uint64_t>(ODD ? y + 2u * (uint64_t)orow + parity : y + orow);   // (the pointer argument is read here, not behind the barrier)
    lev_pin(pw);
    lev_pin(pr);
    lev_pin(k0);
    lev_pin(k1);
    lev_pin(k2);
    lev_pin(k3);
    lev_pin(stores);
    lev_pin(yp);

    if (lane < kQ4mZeroBytes / 4u) reinterpret_cast<uint32_t *>(zero)[lane] = 0u;
    // more than two tasks' operands do not fit the registers: a product reads them again
    constexpr bool kKept = TPW <= 2;
    q4m_operand op[kKept ? TPW : 1];
    float unscale[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const bool live = active && t_first + t < ntask;
        unscale[t] = q4m_stage_planes(q4m_mask_activations(v[t], v_live[t]), area + t * kQ4mTaskArea, live);
        if (kKept) {
            q4m_read_operands(area + t * kQ4mTaskArea, zero, live, op[t]);
            op[t].unscale = unscale[t];
        }
    }
    // the operands are read back before the wait for the weights, not behind it
    __builtin_amdgcn_sched_barrier(0);

    const uint32_t nrounds = (ngroups + slots - 1u) / slots;     // rounds of `slots` row groups
    auto finish = [&](const uint32_t (&D)[TPW][9]) {
        float val = 0.f;
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            uint32_t W[9];
            q4m_turn_task(D[t], W);
            if (ODD) {
                // the scale of the neighbour's block: A of the first pair of an odd row, B of the last of an even one
                // (as requested: lanes and tasks past the row's end repeat its last pair)
                const uint32_t T = t_first + t < ntask ? t_first + t : ntask - 1u;
                const uint32_t pair = 4u * T + q < npairs ? 4u * T + q : npairs - 1u;
                W[0] &= parity && pair == 0u ? 0xFFFF0000u : ~0u;
                W[4] &= !parity && pair + 1u == npairs ? 0x0000FFFFu : ~0u;
            }
            if (!kKept) {
                q4m_read_operands(area + t * kQ4mTaskArea, zero, active && t_first + t < ntask, op[0]);
                op[0].unscale = unscale[t];
            }
            val += q4m_task_dot(W, op[kKept ? t : 0]);
        }
        val = lev_row_sum_f32(val);
        if (lane < 16u) *reinterpret_cast<float *>(smem + pw) = val;
        lev_barrier_lds();
        if (wave < slots) {
            const float *pp = reinterpret_cast<const float *>(smem + pr);
            const float p0 = pp[0], p1 = pp[64], p2 = pp[128], p3 = pp[192];   // four reads in flight together
            auto keep = [](float p, uint32_t k) { return __uint_as_float(__float_as_uint(p) & k); };
            float s = (keep(p0, k0) + keep(p1, k1)) + (keep(p2, k2) + keep(p3, k3));
            s = lev_row_sum_f32(s);
            if (stores) *reinterpret_cast<__attribute__((address_space(1))) float *>(yp) = s;   // a global store, not a flat one
        }
        if (!SINGLE) {
            pw ^= kQ4mWaves * 16u * 4u;                          // the other half of `part` next round
            pr ^= kQ4mWaves * 16u * 4u;
            orow += orow_step;
            yp += (uint64_t)orow_step * (ODD ? 8u : 4u);
            stores = writer && orow < nrows ? 1u : 0u;
        }
    };
    if (SINGLE) {
        finish(Da);
        return;
    }
    // Unconditional (clamped) prefetch: a branch around the loads would make the compiler wait
    // for them before the current group is multiplied.
    uint32_t Db[TPW][9];
    while (true) {
        uint32_t next = rb + nblocks;
        issue(next < nrounds ? next : rb, Db);
        finish(Da);
        if (next >= nrounds) break;
        rb = next;
        next = rb + nblocks;
        issue(next < nrounds ? next : rb, Da);
        finish(Db);
        if (next >= nrounds) break;
        rb = next;
    }
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

bool lev_q4_0_mfma_gemv_usable(const uint8_t *w, const float *x, uint32_t in_dim) {
    return lev_q4_0_mfma_in_dim(in_dim) && (reinterpret_cast<uintptr_t>(w) & 3u) == 0u &&
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
