// Router scores of few tokens: the body of the kernel of its own (moe.hip) and of the part of a launch that it shares with an
// operator that does not depend on it.
#pragma once

#include "lev_common.hpp"

// DPP lane exchange of a 64-bit value; lanes the control word does not write
// keep their own value.
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ double dpp_move_f64(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xF, false);
    hi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xF, false);
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double lane63_f64(double v) {
    int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
    int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
    return __hiloint2double(hi, lo);
}

// Sum over the 64 lanes, returned in every lane (wave-uniform).
__device__ __forceinline__ double wave_sum_f64(double v) {
    v += dpp_move_f64<0xB1>(v);
    v += dpp_move_f64<0x4E>(v);
    v += dpp_move_f64<0x141>(v);
    v += dpp_move_f64<0x140>(v);
    {   // row_bcast steps: lanes outside the mask must add nothing
        int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x142, 0xA, 0xF, false);
        int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x142, 0xA, 0xF, false);
        v += __hiloint2double(hi, lo);
        lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x143, 0xC, 0xF, false);
        hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x143, 0xC, 0xF, false);
        v += __hiloint2double(hi, lo);
    }
    return lane63_f64(v);
}
// Router scores of few tokens, f64 accumulation rounded to f32 once: 256 threads per expert and token, whose waves
// share the row and meet in LDS (`partial`, four of them).  A launch is one trip to memory, so a thread's four pieces of both
// operands are requested together (rows of up to 4096 columns; longer ones repeat that).  The router comes from L2 for all
// tokens but the first: at 2816 columns and 128 experts five tokens take 20 us with a row read once for four tokens by one
// wave, 4.5 us this way.  e >= experts: only the barrier.
__device__ __forceinline__ void moe_score_few(const float *__restrict__ wr, const float *__restrict__ x, float *__restrict__ scores,
                                              uint32_t hidden, uint32_t experts, uint32_t e, uint32_t t, uint32_t tid,
                                              double *partial) {
    double acc = 0.0;
    if (e < experts) {
        const float *row = wr + (uint64_t)e * hidden, *xv = x + (uint64_t)t * hidden;
        if ((hidden & 3u) == 0u && ((reinterpret_cast<uintptr_t>(wr) | reinterpret_cast<uintptr_t>(x)) & 15u) == 0u) {
            const lev_f32x4 *r4 = reinterpret_cast<const lev_f32x4 *>(row), *x4 = reinterpret_cast<const lev_f32x4 *>(xv);
            const uint32_t n4 = hidden >> 2;
            double a0 = 0.0, a1 = 0.0;
            for (uint32_t i0 = tid; i0 < n4; i0 += 1024u) {
                lev_f32x4 a[4], b[4];
    #pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) {
                    const uint32_t i = i0 + 256u * k < n4 ? i0 + 256u * k : i0;
                    a[k] = r4[i];
                    b[k] = x4[i];
                }
    #pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) {
                    if (i0 + 256u * k >= n4) b[k] = lev_f32x4{0.f, 0.f, 0.f, 0.f}, a[k] = b[k];
                    a0 = fma((double)a[k].x, (double)b[k].x, a0);
                    a1 = fma((double)a[k].y, (double)b[k].y, a1);
                    a0 = fma((double)a[k].z, (double)b[k].z, a0);
                    a1 = fma((double)a[k].w, (double)b[k].w, a1);
                }
            }
            acc = a0 + a1;
        } else {
            acc = 0.0;
            for (uint32_t i = tid; i < hidden; i += 256u) acc = fma((double)row[i], (double)xv[i], acc);
        }
        acc = wave_sum_f64(acc);
        if ((tid & 63u) == 0u) partial[tid >> 6] = acc;
    }
    lev_barrier_lds();
    if (e < experts && tid == 0u)
        scores[(uint64_t)t * experts + e] = (float)(((partial[0] + partial[1]) + partial[2]) + partial[3]);
}
