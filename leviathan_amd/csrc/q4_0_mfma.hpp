// Q4_0 x f32 on the integer matrix cores: the building block of the decode GEMV and of the
// MoE expert kernels at few tokens.
//
// One TASK is 16 weight rows x 4 pairs of blocks (256 activations).  v_mfma_i32_16x16x64_i8
// multiplies 16 rows x 64 codes; lane (r, g) = (lane % 16, lane / 16) supplies, as B, 16 codes of
// row r: the low nibbles, then the high nibbles, of one block of ITS OWN pair (pair 4T + g of the
// task), as int8 bytes 16*(n - 8) -- one bit operation per four codes: masking a nibble into the
// high half of a byte and flipping its top bit IS the signed value, so the offset of the format
// never needs a correction term.  A row 4g + p holds digit plane p of the 16 activations lane
// group g multiplies and zeros elsewhere (the other lanes read a zeroed strip), so accumulator
// register p of lane (r, g) is the plane-p sum of that lane's own codes: nothing is exchanged
// between lanes until a row's four lane groups add their finished pair sums.
//
// Activations: per block (32 values) x becomes integers X = rint(x * 2^(156 - ex)),
// |X| <= 2^30, ex the biased exponent of the block's largest magnitude: every value within 2^-6 of
// that maximum is represented exactly.  X is cut into four balanced base-256 digits (the bytes of
// (X + 0x808080) ^ 0x808080 read as int8).  The integer sums are exact; a block's planes are
// recombined and scaled by d in f32, so what is rounded is one number per block of 32 weights.
//
// Against 64-bit sums, on normal activations: 6e-8 to 8e-8 (2-norm) over rows of 480 to 8000 values, where the f32
// chains of the vector-ALU kernels leave 2.0e-7 to 3.3e-7.  What the integers do not have is f32's range: a value far
// below the largest of its block keeps multiples of 2^-31 of that maximum.  Where the block has a scale the maximum costs the
// chains more, which add n * x and take 8 * x off in the end: an outlier of 2^13 in every other block that meets the code of
// zero leaves 3.2e-4 with them (1216 values) and 3e-6 here.  Where the scale is zero the block adds nothing in either, which
// is why the power of two is a block's and not a pair's: with one for 64 values the pair's other block was 5e-6 off beside
// 2^13 and lost beside 2^31.  Below a maximum of 2^-93 the unit stays 2^-123.
//
// A wave stages the 256 activations of its own task by itself (one float4 per lane, a 1 KB area
// of LDS nobody else touches): no workgroup barrier stands between the activations and the
// products, and the A operands (16 registers a task) serve every row group the wave visits.
//
// Weight bytes are fetched with the four pairs of a row in four ADJACENT lanes (lane = 4*row +
// pair: a quad reads 144 contiguous bytes; with lane = 16*pair + row every quad touches four
// rows and the same read of a cold 9 MB matrix takes 0.3 us longer) and handed to the lane the
// matrix core wants them in by one lane permutation per dword.
#pragma once

#include "q4_0_device.hpp"

typedef int lev_i32x4 __attribute__((ext_vector_type(4)));

// Rows the matrix-core GEMV takes, up to 8192 values: whole 256-value tasks, and from five tasks on rows that end
// inside one (narrower ones of those are the launch floor with either kernel, 3 us at 1088 x 5000, and stay with the
// vector-ALU kernels).  From a task on and up to 16384 values: rows of an odd number of blocks, which only a kernel of
// 2-byte loads takes beside it (narrower ones keep that: the experts' kernels form such rows' sums in its order).
__host__ inline bool lev_q4_0_mfma_in_dim(uint32_t in_dim) {
    if (in_dim == 0u || in_dim % 32u != 0u) return false;
    if (in_dim % 64u != 0u) return in_dim > 256u && in_dim <= 16384u;
    return in_dim <= 8192u && (in_dim % 256u == 0u || in_dim > 1280u);
}
constexpr uint32_t kQ4mTaskArea = 1024u;   // LDS bytes of one staged task: [pair 4][plane 4][half 4][16 B]
constexpr uint32_t kQ4mZeroBytes = 16u;    // what the lanes outside a row's own lane group read as their A operand

// Twice the powers of two that undo the scaling of the two blocks of the lane's own pair (and the 16 of the codes): times a
// scale d of the weights, subnormal ones included, they are exact.
struct q4m_unscale {
    float a, b;
};
// A operands of one task (four halves: block A low / high nibbles, block B low / high).
struct q4m_operand {
    lev_i32x4 a[4];
    q4m_unscale unscale;
};

// Stages the task whose activations are v (lane i holds elements 4i..4i+3 of the task's 256)
// into `area` (kQ4mTaskArea bytes, this wave's own); returns the lane's `unscale`.  live == false: the
// task lies beyond the row (it adds nothing).  A NaN or an infinity among the 32 activations of a block
// makes the block's factor NaN, and with it every row's sum.
__device__ __forceinline__ q4m_unscale q4m_stage_planes(const lev_f32x4 v, uint8_t *area, bool live) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t r = lane & 15u, g = lane >> 4;
    uint32_t mb = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t bits = __float_as_uint(v[k]) & 0x7FFFFFFFu;
        mb = bits > mb ? bits : mb;
    }
    mb = lev_row8_max_u32(mb);    // the 8 lanes of a block hold the block's maximum
    uint32_t ex = mb >> 23;                                    // |x| < 2^(ex - 126)
    const bool bad = ex == 255u;
    ex = ex < 34u ? 34u : (ex > 254u ? 254u : ex);             // keeps both powers of two normal numbers
    const float scale = __uint_as_float((283u - ex) << 23);    // 2^(156 - ex): |x * scale| < 2^30
    uint32_t Y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) Y[k] = (uint32_t)(int)rintf(v[k] * scale) + 0x00808080u;
    // 4x4 byte transpose: digit p of the lane's four values in one dword
    const uint32_t t0 = __builtin_amdgcn_perm(Y[1], Y[0], 0x05010400u);
    const uint32_t t1 = __builtin_amdgcn_perm(Y[1], Y[0], 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(Y[3], Y[2], 0x05010400u);
    const uint32_t t3 = __builtin_amdgcn_perm(Y[3], Y[2], 0x07030602u);
    uint32_t dw[4];
    dw[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
    dw[1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
    dw[2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
    dw[3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
    for (int p = 0; p < 3; ++p) dw[p] ^= 0x80808080u;
    // lane i: pair i / 16, half (i % 16) / 4, k-slots 4 * (i % 4) .. + 3
    uint8_t *at = area + g * 256u + (r >> 2) * 16u + (r & 3u) * 4u;
#pragma unroll
    for (int p = 0; p < 4; ++p) *reinterpret_cast<uint32_t *>(at + 64 * p) = dw[p];
    // the area belongs to this wave alone: LDS runs a wave's accesses in order, the fences only
    // keep the compiler from moving the reads above the writes
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // 2^(ex - 159) of the lane's block; the pair's two from lanes 0 and 8 of its 16
    const uint32_t own = !live ? 0u : bad ? 0x7FC00000u : (ex - 32u) << 23;
    return q4m_unscale{lev_row_bcast<0>(own), lev_row_bcast<8>(own)};
}

// The lane's A operands of a staged task.  `zero` points at kQ4mZeroBytes of zeros: what a lane outside the
// row's own lane group reads, and every lane of a task that is not live.
__device__ __forceinline__ void q4m_read_operands(const uint8_t *area, const uint8_t *zero, bool live, q4m_operand &op) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t r = lane & 15u, g = lane >> 4;
    const bool feeds = live && (r >> 2) == g;                  // A row r belongs to lane group r / 4
    const uint8_t *ab = feeds ? area + g * 256u + (r & 3u) * 64u : zero;
    const uint32_t hs = feeds ? 16u : 0u;
#pragma unroll
    for (int h = 0; h < 4; ++h) op.a[h] = *reinterpret_cast<const lev_i32x4 *>(ab + h * hs);
}

__device__ __forceinline__ void q4m_stage_task(const lev_f32x4 v, uint8_t *area, const uint8_t *zero,
                                               bool live, q4m_operand &op) {
    op.unscale = q4m_stage_planes(v, area, live);
    q4m_read_operands(area, zero, live, op);
}

// The weights of one task as they are fetched: lane 4*row + pair holds pair `pair` of row `row`.
// `rowp` = first byte of the lane's row (row lane / 4 of the group), task_pair0 = 4 * task.
__device__ __forceinline__ void q4m_load_task(const uint8_t *rowp, uint32_t task_pair0, uint32_t D[9]) {
    const uint32_t lane = threadIdx.x & 63u;
    lev_q4_load_pair(rowp + (uint64_t)(task_pair0 + (lane & 3u)) * 36u, D);
}

// The same where the row's last task may be a part of one (npairs pairs a row): lanes past the row's end
// repeat its last pair.  Their activations count as zero (q4m_load_activations).
__device__ __forceinline__ void q4m_load_task_part(const uint8_t *rowp, uint32_t task_pair0, uint32_t npairs, uint32_t D[9]) {
    const uint32_t pair = task_pair0 + (threadIdx.x & 3u);
    lev_q4_load_pair(rowp + (uint64_t)((pair < npairs ? pair : npairs - 1u) * 36u), D);
}

// The same for rows of an odd number of blocks, whose half of a pair may end the matrix, at w_end: nothing behind it is
// requested.  Of such a pair block A is right, its last two bytes moved to where they belong, and block B arbitrary.
__device__ __forceinline__ void q4m_load_task_odd(const uint8_t *rowp, uint32_t task_pair0, uint32_t npairs, const uint8_t *w_end, uint32_t D[9]) {
    struct __attribute__((packed, aligned(2))) u4 { uint32_t v[4]; };
    struct __attribute__((packed, aligned(2))) u1 { uint32_t v; };
    const uint32_t pair = task_pair0 + (threadIdx.x & 3u);
    const uint8_t *p = rowp + (uint64_t)((pair < npairs ? pair : npairs - 1u) * 36u);
    const bool half = w_end - p < 36;
    const u4 a = *reinterpret_cast<const u4 *>(p);
    const u1 m = *reinterpret_cast<const u1 *>(half ? p + 14 : p + 16);
    const u4 b = *reinterpret_cast<const u4 *>(half ? p : p + 20);
    D[0] = a.v[0], D[1] = a.v[1], D[2] = a.v[2], D[3] = a.v[3];
    D[4] = half ? m.v >> 16 : m.v;
    D[5] = b.v[0], D[6] = b.v[1], D[7] = b.v[2], D[8] = b.v[3];
}

// The 256 activations of task T of a vector of n4 float4: lane i requests elements 4i..4i+3 (`late` float4 earlier); past
// either end one of the vector's is requested, and `live` (what to pass to q4m_mask_activations behind the wait) is false.
__device__ __forceinline__ lev_f32x4 q4m_load_activations(const float *x, uint32_t T, uint32_t n4, bool &live, uint32_t late = 0u) {
    const uint32_t i = 64u * T + (threadIdx.x & 63u) - late;
    live = i < n4;                                             // (a lane before the first element wraps round)
    return reinterpret_cast<const lev_f32x4 *>(x)[live ? i : n4 - 1u];
}
__device__ __forceinline__ lev_f32x4 q4m_mask_activations(lev_f32x4 v, bool live) {
    return live ? v : lev_f32x4{0.f, 0.f, 0.f, 0.f};
}

// Lane (r, g) <- lane 4*r + g, for every dword of a fetched task.
__device__ __forceinline__ void q4m_turn_task(const uint32_t D[9], uint32_t W[9]) {
    const uint32_t lane = threadIdx.x & 63u;
    const int src = (int)((4u * (lane & 15u) + (lane >> 4)) * 4u);
#pragma unroll
    for (int k = 0; k < 9; ++k) W[k] = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)D[k]);
}

// Twice the contribution of the lane's pair (W: its 36 bytes, already turned) to its row's dot product, which is halved where
// the row's sum ends.
__device__ __forceinline__ float q4m_task_dot(const uint32_t W[9], const q4m_operand &op) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    const float da = fmaf(lev_f16_bits_to_f32(W[0] & 0xFFFFu), op.unscale.a, 0.f);   // (converts and multiplies in one)
    const float db = fmaf(lev_f16_bits_to_f32(W[4] >> 16), op.unscale.b, 0.f);
    u4 qa, qb;
    qa.x = __builtin_amdgcn_alignbit(W[1], W[0], 16);
    qa.y = __builtin_amdgcn_alignbit(W[2], W[1], 16);
    qa.z = __builtin_amdgcn_alignbit(W[3], W[2], 16);
    qa.w = __builtin_amdgcn_alignbit(W[4], W[3], 16);
    qb = u4{W[5], W[6], W[7], W[8]};
    // int8 bytes 16*(n - 8): the nibble in the high half of its byte, its top bit flipped
    const lev_i32x4 bal = __builtin_bit_cast(lev_i32x4, ((qa << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
    const lev_i32x4 bah = __builtin_bit_cast(lev_i32x4, (qa & 0xF0F0F0F0u) ^ 0x80808080u);
    const lev_i32x4 bbl = __builtin_bit_cast(lev_i32x4, ((qb << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
    const lev_i32x4 bbh = __builtin_bit_cast(lev_i32x4, (qb & 0xF0F0F0F0u) ^ 0x80808080u);
    lev_i32x4 sa = __builtin_amdgcn_mfma_i32_16x16x64_i8(op.a[0], bal, lev_i32x4{0, 0, 0, 0}, 0, 0, 0);
    lev_i32x4 sb = __builtin_amdgcn_mfma_i32_16x16x64_i8(op.a[2], bbl, lev_i32x4{0, 0, 0, 0}, 0, 0, 0);
    sa = __builtin_amdgcn_mfma_i32_16x16x64_i8(op.a[1], bah, sa, 0, 0, 0);
    sb = __builtin_amdgcn_mfma_i32_16x16x64_i8(op.a[3], bbh, sb, 0, 0, 0);
    // |plane sum| <= 32 * 128 * 128 = 2^19: two planes recombine in 32 bits, the halves in f32
    const float fa = fmaf((float)(sa[2] + (sa[3] << 8)), 65536.0f, (float)(sa[0] + (sa[1] << 8)));
    const float fb = fmaf((float)(sb[2] + (sb[3] << 8)), 65536.0f, (float)(sb[0] + (sb[1] << 8)));
    return fmaf(da, fa, db * fb);
}
