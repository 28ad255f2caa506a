// The body of the Q4_0 decode GEMV on the integer matrix cores: of the kernel of its own (q4_0_mfma_gemv.hip) and of the
// part of a launch that it shares with an operator that does not depend on it.
#pragma once

#include "q4_0_mfma.hpp"

constexpr int kQ4mWaves = 16;
constexpr int kQ4mThreads = kQ4mWaves * LEV_WAVE;

// LDS: part [2][16 waves][16 rows] f32 (2 KB, so that the round's half is one XOR away) | per
// wave TPW task areas and a zero strip
__host__ __device__ constexpr size_t q4m_gemv_lds(uint32_t tpw) {
    return 2u * kQ4mWaves * 16u * 4u + (size_t)kQ4mWaves * (tpw * kQ4mTaskArea + kQ4mZeroBytes);
}

// wave -> (slot, position in the slot): 4-bit entries of two 64-bit kernel arguments (lev_wave_tables).
// SINGLE: the grid covers every round once: straight-line code, nothing to prefetch.
// block, nblocks: the workgroup's place among those of the product.  Waves beyond the slots' only meet the barrier.
// PIN: addresses and masks of the sums held in registers over the rounds (64 of which do not hold them as well).
template <int TPW, bool SINGLE, bool ODD, bool PIN = true>
__device__ __forceinline__ void q4m_gemv(const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ y,
                                         uint32_t in_dim, uint32_t rows, uint32_t wpr, uint32_t slots, uint64_t slot_of_wave,
                                         uint64_t pos_of_wave, uint32_t block_idx, uint32_t grid_dim, uint8_t *smem) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    // wave-uniform by construction: in a scalar register, so that everything derived from it is
    // scalar arithmetic
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t slot = (uint32_t)(slot_of_wave >> (4u * wave)) & 15u;   // idle waves: slot >= slots
    const uint32_t tw = (uint32_t)(pos_of_wave >> (4u * wave)) & 15u;
    const uint32_t npairs = (in_dim + 63u) >> 6, ntask = (npairs + 3u) >> 2;   // the last task may be a part of one
    const uint32_t t_first = tw * TPW;
    // ODD: the workgroup's half of the matrix, rows parity, parity + 2, ...
    const uint32_t parity = ODD ? block_idx & 1u : 0u;
    const uint32_t block = ODD ? block_idx >> 1 : block_idx, nblocks = ODD ? grid_dim >> 1 : grid_dim;
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
    if (PIN) {
        lev_pin(pw);
        lev_pin(pr);
        lev_pin(k0);
        lev_pin(k1);
        lev_pin(k2);
        lev_pin(k3);
        lev_pin(stores);
        lev_pin(yp);
    }

    if (lane < kQ4mZeroBytes / 4u) reinterpret_cast<uint32_t *>(zero)[lane] = 0u;
    // more than two tasks' operands do not fit the registers: a product reads them again
    constexpr bool kKept = TPW <= 2;
    q4m_operand op[kKept ? TPW : 1];
    q4m_unscale unscale[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const bool live = active && t_first + t < ntask;
        unscale[t] = q4m_stage_planes(q4m_mask_activations(v[t], v_live[t]), area + t * kQ4mTaskArea, live);
        if (kKept) {
            q4m_read_operands(area + t * kQ4mTaskArea, zero, live, op[t]);
            op[t].unscale = unscale[t];
        }
    }
    // ODD: without the scale of the neighbour's block, A of the first pair of an odd row, B of the last of an even one (as
    // requested: lanes and tasks past the row's end repeat its last pair).  Kept as masks over the rounds: seen through, they
    // become selects between the conversion of a scale and its product, which are one instruction otherwise (30092 x 3168
    // 11.00 us and 10.86; one round alone is 0.1 of 6.9 us faster without the registers).
    uint32_t own_a[TPW], own_b[TPW];
    if (ODD) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            const uint32_t T = t_first + t < ntask ? t_first + t : ntask - 1u;
            const uint32_t pair = 4u * T + q < npairs ? 4u * T + q : npairs - 1u;
            own_a[t] = parity && pair == 0u ? 0xFFFF0000u : ~0u;
            own_b[t] = !parity && pair + 1u == npairs ? 0x0000FFFFu : ~0u;
            if (!SINGLE) lev_pin(own_a[t]);
            if (!SINGLE) lev_pin(own_b[t]);
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
                W[0] &= own_a[t];
                W[4] &= own_b[t];
            }
            if (!kKept) {
                q4m_read_operands(area + t * kQ4mTaskArea, zero, active && t_first + t < ntask, op[0]);
                op[0].unscale = unscale[t];
            }
            const float dot = q4m_task_dot(W, op[kKept ? t : 0]);
            val = t ? val + dot : dot;
        }
        val = lev_row_sum_f32(val);
        if (lane < 16u) *reinterpret_cast<float *>(smem + pw) = val;
        lev_barrier_lds();
        if (wave < slots) {
            const float *pp = reinterpret_cast<const float *>(smem + pr);
            const float p0 = pp[0], p1 = pp[64], p2 = pp[128], p3 = pp[192];   // four reads in flight together
            auto keep = [](float p, uint32_t k) { return __uint_as_float(__float_as_uint(p) & k); };
            float s = (keep(p0, k0) + keep(p1, k1)) + (keep(p2, k2) + keep(p3, k3));
            s = 0.5f * lev_row_sum_f32(s);
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
