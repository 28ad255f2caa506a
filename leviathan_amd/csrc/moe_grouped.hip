// Routed Q4_0 experts for MANY tokens on gfx950: (token, slot) pairs are
// grouped by expert, and each expert's weights are streamed once and applied
// to all of its tokens on the matrix cores.
//
// Stands in for runMoeBatchedRouted applied token after token
// (Sources/LeviathanCore/Gemma4.swift:2073, per-slot loop :3856-3880;
// moegen_gu/act/dn, MoELowering.swift:749-835): same results per pair, same
// slot-ordered f32 merge; only the order in which pairs are visited changes.
// With one launch per (token, slot) every pair streams its expert's 2.65 MB
// again (64 tokens x top-8 = 512 x 2.65 MB against 126 distinct experts).
//
// Pipeline (all on the context's stream): group (histogram of expert ids -> pair lists, work items,
// where each workgroup starts), gate/up on the integer matrix cores -> act = gelu_tanh(g)*u (f32,
// [pair][inter]), down -> dn (f32, [pair][hidden]), merge: y[t] = sum over slots, IN SLOT ORDER,
// fmaf(w_slot, dn_slot, acc).
//
// Batches of at most eight pairs per expert on average, with rows of up to 4096
// activations, take these kernels (the digit planes of the few-token kernels, four tokens of an expert
// per product, operands in registers): they cost less per product than the grouped matrix product of
// moe_prefill.hip and more per token, and win while most experts hold no more than a handful of pairs.
#include "moe_prefill.hpp"

#include <array>
#include <cmath>
#include <cstdio>
#include "q4_0_mfma.hpp"

#include <cstdlib>

namespace {

constexpr int kFlagBadExpertId = 1;                       // same bit as the per-token kernels
constexpr int kG8NT = 8;                                  // tokens per item
static_assert(kG8NT == 4 || kG8NT == 8, "an item is one or two groups of four tokens");

// ---------------------------------------------------------------------------
// 1. group pairs by expert.  One workgroup.  A pair is dropped (and flagged)
// when its id is out of range or repeats an earlier slot of the same token,
// as MoEModelBinding.offsets requires (MoEModelBinding.swift:174-214).
// valid[p]: pair p takes part.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024)
moe_group_kernel(const int32_t *__restrict__ ids, uint32_t pairs, uint32_t experts, uint32_t top_k,
                 uint8_t *__restrict__ valid, int *__restrict__ flag, lev_grp_item *items,
                 lev_grp_start *__restrict__ starts, uint32_t grid, uint32_t rpi_gu, uint32_t rpi_dn, uint32_t w1_gu,
                 uint32_t w2_gu, uint32_t w1_dn, uint32_t w2_dn, uint32_t s0_gu, uint32_t s0_dn) {
    // [experts] counts | cursors | first pair | first item of more than four pairs | first other item; [items] expert * 16 + count
    extern __shared__ int32_t s_cnt[];
    int32_t *s_cur = s_cnt + experts, *s_first = s_cur + experts, *s_big = s_first + experts, *s_small = s_big + experts;
    int32_t *s_item = s_small + experts;
    const uint32_t tid = threadIdx.x;
    // (barriers that leave stores on their way: the workgroup exchanges nothing but LDS)
    for (uint32_t e = tid; e < experts; e += 1024u) s_cnt[e] = 0;
    lev_barrier_lds();
    bool bad_seen = false;
    int32_t e_own = -1;                          // the thread's first pair, kept for the placement: its expert, or -1
    for (uint32_t p = tid; p < pairs; p += 1024u) {
        const int32_t e = ids[p];
        bool ok = e >= 0 && (uint32_t)e < experts;
        const uint32_t slot = p % top_k, first = p - slot;
        // both copies of a duplicate are dropped; the token's ids are requested eight at a time (one
        // wait for eight, not one after the other)
        for (uint32_t k0 = 0; k0 < top_k; k0 += 8u) {
            int32_t other[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) other[u] = ids[first + (k0 + u < top_k ? k0 + u : slot)];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u)
                if (k0 + u < top_k && k0 + u != slot && other[u] == e) ok = false;
        }
        valid[p] = ok ? 1 : 0;
        if (ok) atomicAdd(&s_cnt[e], 1);
        if (p == tid && ok) e_own = e;
        bad_seen = bad_seen || !ok;
    }
    if (bad_seen) atomicOr(flag, kFlagBadExpertId);
    lev_barrier_lds();
    // exclusive scan of the counts (experts <= 4096: up to four a thread, side by side).  One scan carries three counts of at most
    // 2^20 each in 21-bit fields: pairs, items of more than four pairs, other items.
    __shared__ uint64_t s_wave[16];
    uint32_t n_big = 0u, n_all = 0u;            // items of more than four pairs, all items
    {
        const uint32_t per_thread = (experts + 1023u) >> 10;
        int32_t c4[4], big4[4], small4[4];
        constexpr int32_t ip = kG8NT, ish = ip == 8 ? 3 : 2;
        uint64_t local = 0;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            if (k >= per_thread) break;
            const uint32_t e = per_thread * tid + k;
            c4[k] = e < experts ? s_cnt[e] : 0;
            // work items of the integer matrix-core kernels: runs of at most kG8NT pairs of one expert
            const int32_t full = c4[k] >> ish, rem = c4[k] - (full << ish);
            big4[k] = (ip > 4 ? full : 0) + (rem > 4 ? 1 : 0);
            small4[k] = (ip > 4 ? 0 : full) + (rem > 0 && rem <= 4 ? 1 : 0);
            local += (uint64_t)c4[k] | (uint64_t)big4[k] << 21 | (uint64_t)small4[k] << 42;
        }
        uint64_t before, all;
        lev_scan_1024(local, s_wave, before, all);
        int32_t run = (int32_t)(before & 0x1FFFFFu);
        const int32_t first_pair = run;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            if (k >= per_thread) break;
            const uint32_t e = per_thread * tid + k;
            if (e < experts) s_cur[e] = run;
            run += c4[k];
        }
        // Items of more than four pairs (two products a block) come first, in expert order, the
        // others behind them: what a round costs then depends on its position in the line of
        // rounds alone.
        const int32_t nbig = (int32_t)(all >> 21 & 0x1FFFFFu), nsmall = (int32_t)(all >> 42);
        int32_t brun = (int32_t)(before >> 21 & 0x1FFFFFu), srun = nbig + (int32_t)(before >> 42);
        n_big = (uint32_t)nbig;
        n_all = (uint32_t)(nbig + nsmall);
        int32_t prun = first_pair;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            if (k >= per_thread) break;
            const uint32_t e = per_thread * tid + k;
            if (e < experts) {
                s_first[e] = prun;
                s_big[e] = brun;
                s_small[e] = srun;
            }
            const int32_t n = big4[k] + small4[k];
            for (int32_t j = 0; j < n; ++j) {
                const int32_t left = c4[k] - j * ip, count = left < ip ? left : ip;
                const int32_t at = count > 4 ? brun++ : srun++;
                s_item[at] = (int32_t)e * 16 + count;
                lev_grp_item *it = items + at;
                it->expert = (int32_t)e;
                it->count = count;
                it->first = prun + j * ip;
            }
            prun += c4[k];
        }
    }
    lev_barrier_lds();   // (the items' headers are still on their way to memory: what is read of them below is in LDS as well)
    const uint32_t sid = 1023u - tid;   // (the high threads: the low ones place the first 1024 pairs below)
    if (sid < 2u * grid) {
        // Where the workgroups of the two expert kernels start.  A round of an item of more than
        // four pairs costs w2, any other w1, and beginning an item (its header, its activations,
        // their staging) costs s0 wherever the item begins; the line of items is cut into
        // stretches of equal COST.  The items of more than four pairs come first, so a position in
        // cost is a position in rounds by a few divisions (32-bit arithmetic: cost < 2^29,
        // grid <= 2^9).
        const uint32_t down = sid >= grid ? 1u : 0u, L = sid - down * grid, rpi = down ? rpi_dn : rpi_gu;
        const uint32_t w1 = down ? w1_dn : w1_gu, w2 = down ? w2_dn : w2_gu, s0 = down ? s0_dn : s0_gu;
        const uint32_t I2 = s0 + rpi * w2, I1 = s0 + rpi * w1;       // cost of a whole item
        const uint32_t R2 = n_big * rpi, C2 = n_big * I2;
        const uint32_t total = C2 + (n_all - n_big) * I1, per = total / grid, rest = total - per * grid;
        // rounds that lie wholly or partly before cost position c
        auto rounds_before = [&](uint32_t c) {
            const bool big = c <= C2;
            const uint32_t cc = big ? c : c - C2, I = big ? I2 : I1, w = big ? w2 : w1;
            const uint32_t item = cc / I, in_item = cc - item * I;
            const uint32_t r = in_item <= s0 ? 0u : (in_item - s0 + w - 1u) / w;
            return (big ? 0u : R2) + item * rpi + r;
        };
        lev_grp_start st;
        st.first_round = rounds_before(per * L + rest * L / grid);
        st.end_round = rounds_before(per * (L + 1u) + rest * (L + 1u) / grid);
        st.item = st.first_round / rpi;
        const int32_t header = n_all ? s_item[st.item < n_all ? st.item : 0u] : 0;
        st.expert = header >> 4;
        st.count = header & 15;
        st.pad[0] = st.pad[1] = st.pad[2] = 0u;
        starts[sid] = st;
    }
    // The order of an expert's pairs in the list depends on the atomics; no
    // result does: every pair is computed independently and owns its outputs.
    for (uint32_t p = tid; p < pairs; p += 1024u)
        if (p == tid ? e_own >= 0 : valid[p] != 0) {
            const int32_t e = p == tid ? e_own : ids[p];
            const int32_t at = atomicAdd(&s_cur[e], 1);
            // the pair's column in its item: the expert's items of more than four pairs come
            // first in the expert's list (whole items, then a remainder of more than four)
            constexpr int32_t ip = kG8NT, ish = ip == 8 ? 3 : 2;
            const int32_t c = s_cnt[e], pos = at - s_first[e];
            const int32_t full = c >> ish, rem = c - (full << ish), nbig = (ip > 4 ? full : 0) + (rem > 4 ? 1 : 0);
            const int32_t j = pos >> ish;
            lev_grp_item *it = items + (j < nbig ? s_big[e] + j : s_small[e] + (j - nbig));
            const int32_t left = c - j * ip, count = left < ip ? left : ip, col = pos - j * ip;
            it->pair[col] = (int32_t)p;
            it->src[col] = (int32_t)(p / top_k);
            if (col == count - 1)   // the columns past the count repeat the last pair
                for (int32_t k = count; k < 8; ++k) {
                    it->pair[k] = (int32_t)p;
                    it->src[k] = (int32_t)(p / top_k);
                }
        }
}

// ---------------------------------------------------------------------------
// 2./3. on the integer matrix cores, four tokens of an expert per product.
//
// v_mfma_i32_16x16x32_i8 multiplies 16 A rows x 32 k x 16 weight rows: ONE Q4_0 block of 16 weight
// rows.  A row 4t + p is digit plane p of token t (x as integers X = rint(x * 2^(156 - ex)), ex
// the exponent of the largest magnitude among the task's 256 activations, cut into four balanced
// base-256 digits: the arithmetic of the few-token kernels), so the output lane (row, t) holds
// the four plane sums of token t against its row's block: they are recombined in 32-bit integers
// and f32 and scaled by the block's d there, with nothing exchanged between lanes.  B: lane
// (row, g) supplies code bytes 4g..4g+3 of the block, low nibbles then high nibbles, as int8
// 16 * (n - 8) (flip the top bit of every nibble, mask; the low nibbles shifted up first).
//
// A task is fetched as in the decode GEMV (a quad of lanes reads the 144 contiguous bytes of a
// row's four block pairs; one lane permutation per dword brings pair g of row r to lane (r, g));
// the dwords of a block are then spread over the four lanes of its row by a 4 x 4 transpose
// between the lane groups (four row swaps), and the scales of the row's eight blocks are
// gathered the same way.
//
// A work ITEM is up to kG8NT pairs of one expert (the grouping kernel cuts each expert's list into
// such runs).  Every item takes the same number of ROUNDS over its expert's rows, so the rounds of
// all items form one line that the grid's workgroups cut into equal stretches, whatever the
// routing: a workgroup works through `total * L / G .. total * (L + 1) / G` and stages the
// activations of each item its stretch touches.  Stretches that follow each other go to
// workgroups of one XCD (an expert with more than kG8NT pairs is streamed by neighbours, through
// one L2).
//
// Workgroup = wpr * slots waves (eight for gate/up, twelve for down), as in the decode GEMV: wave (slot, pos) owns
// column task `pos` (256 activations) of the row groups of its slot, stages the task's
// activations for all of the item's tokens by itself and keeps the operands in registers (16 per
// four tokens).  A round of a wave is NTILE tiles of 16 rows x 256 codes: gate and up rows of one
// row group (PAIRED), or NTILE consecutive row groups (down); the next round's bytes are
// requested as soon as this round's have been handed to the lanes that multiply them.  The wpr
// partial sums of a (row, token) meet in LDS behind one barrier a batch of rounds; wave u adds
// unit u of the batch (a slot's 16 rows x four tokens), applies the activation function (PAIRED)
// and stores.
// ---------------------------------------------------------------------------
constexpr uint32_t kG8MaxGrid = 512;                      // workgroups of an expert kernel (one per CU)
constexpr int kG8WavesGateUp = 8;                         // up to 2048 activations: eight column tasks, one slot
constexpr int kG8WavesDown = 12;                          // 768 activations: three column tasks, four slots (three
                                                          // waves a SIMD; eight waves leave two SIMDs with one)
constexpr int kG8WavesWide = 12, kG8WavesMax = 16;        // wider rows: one wave per column task still, up to 3072 and 4096
constexpr int kG8TilesDown = 1;                          // row groups a wave of the down kernel takes per round (2: rounds twice
                                                          // as long, the stretches a workgroup gets then differ by more: 106.8
                                                          // against 104.4 us a layer at 64 tokens)
constexpr uint32_t g8_batch(int nw) { return nw > 12 ? 2u : 4u; }   // rounds between two barriers of a workgroup (2: 55.4
                                                          // against 53.6 us for gate/up, 1: 64.9; the sums of four rounds of
                                                          // sixteen waves do not fit the LDS)
constexpr uint32_t kG8MaxInLen = 256u * kG8WavesMax;
constexpr uint32_t kG8Plane = 272u;                       // a digit plane of a staged task: 256 bytes + 16, so that
constexpr uint32_t kG8TokArea = 4u * kG8Plane;            // the 64 lanes of an operand read hit 64 different banks
constexpr uint32_t kG8WaveLds = 4u * kG8TokArea;           // four tokens are staged at a time

// LDS: part [parity 2][round of the batch][tile NTILE][token group of the item][wave][row 16][token % 4] f32 | per
// wave four staged tasks
template <int NTILE, int NW>
constexpr size_t g8_lds() {
    return (size_t)2 * g8_batch(NW) * NTILE * (kG8NT / 4) * (NW * 256u) + (size_t)NW * kG8WaveLds;
}

// Digit planes of one token's task into `tok` (kG8TokArea bytes, this wave's own): lane i holds
// elements 4i..4i+3 of the task's 256 activations; plane p, byte e = digit p of element e.
// Returns the power of two that undoes the scaling (and the 16 of the codes); NaN when the task
// holds a NaN or an infinity.
__device__ __forceinline__ float g8_stage_token(const lev_f32x4 v, uint8_t *tok) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t mb = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t bits = __float_as_uint(v[k]) & 0x7FFFFFFFu;
        mb = bits > mb ? bits : mb;
    }
    mb = lev_wave_max_u32(mb);   // every lane: the task's maximum
    uint32_t ex = mb >> 23;                                    // |x| < 2^(ex - 126)
    const bool bad = ex == 255u;
    ex = ex < 34u ? 34u : (ex > 254u ? 254u : ex);             // keeps both powers of two normal numbers
    const float scale = __uint_as_float((283u - ex) << 23);    // 2^(156 - ex): |x * scale| < 2^30
    uint32_t Y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) Y[k] = ((uint32_t)(int)rintf(v[k] * scale) + 0x00808080u) ^ 0x00808080u;
    // 4x4 byte transpose: digit p of the lane's four values in one dword
    const uint32_t t0 = __builtin_amdgcn_perm(Y[1], Y[0], 0x05010400u);
    const uint32_t t1 = __builtin_amdgcn_perm(Y[1], Y[0], 0x07030602u);
    const uint32_t t2 = __builtin_amdgcn_perm(Y[3], Y[2], 0x05010400u);
    const uint32_t t3 = __builtin_amdgcn_perm(Y[3], Y[2], 0x07030602u);
    uint32_t *at = reinterpret_cast<uint32_t *>(tok + 4u * lane);
    at[0u * (kG8Plane / 4u)] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
    at[1u * (kG8Plane / 4u)] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
    at[2u * (kG8Plane / 4u)] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
    at[3u * (kG8Plane / 4u)] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
    return bad ? __builtin_nanf("") : __uint_as_float((ex - 33u) << 23);   // 2^(ex - 160)
}

// A operands of four staged tokens (`toks`: their kG8TokArea areas, one behind the other): lane
// (a, g) = (lane % 16, lane / 16) supplies, for block b of the task, plane a % 4 of token a / 4
// at the block's elements 4g..4g+3 and 16+4g..16+4g+3 (the elements whose codes lie in bytes
// 4g..4g+3 of the block).
__device__ __forceinline__ void g8_read_operands(const uint8_t *toks, long (&A)[8]) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t a = lane & 15u, g = lane >> 4;
    const uint32_t *p = reinterpret_cast<const uint32_t *>(toks + (a >> 2) * kG8TokArea + (a & 3u) * kG8Plane + 4u * g);
#pragma unroll
    for (int b = 0; b < 8; ++b) A[b] = (long)(((uint64_t)p[8 * b + 4] << 32) | (uint64_t)p[8 * b]);
}

// In: lane (r, g) holds q[j] = dword j of a record of lane group g.  Out: q[P] = dword g of the
// record of lane group P (a 4 x 4 transpose between the four lanes of a row, by row swaps).
__device__ __forceinline__ void g8_transpose4(uint32_t (&q)[4]) {
    const auto a = __builtin_amdgcn_permlane16_swap(q[0], q[1], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(q[2], q[3], false, false);
    const auto c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
    q[0] = c[0]; q[1] = d[0]; q[2] = c[1]; q[3] = d[1];
}

// One tile (16 rows x 256 codes; W: the lane's pair, already turned) against NJ groups of four
// tokens, of which the first ng take part: val[j] = the task's sum for (row lane % 16, token
// 4j + lane / 16), blocks added in their order.
template <uint32_t NJ>
__device__ __forceinline__ void g8_tile_dot(const uint32_t W[9], const long (&A)[NJ][8], uint32_t ng,
                                            const float (&unscale)[NJ], float (&val)[NJ]) {
    uint32_t qa[4], qb[4];
    qa[0] = __builtin_amdgcn_alignbit(W[1], W[0], 16);
    qa[1] = __builtin_amdgcn_alignbit(W[2], W[1], 16);
    qa[2] = __builtin_amdgcn_alignbit(W[3], W[2], 16);
    qa[3] = __builtin_amdgcn_alignbit(W[4], W[3], 16);
    qb[0] = W[5]; qb[1] = W[6]; qb[2] = W[7]; qb[3] = W[8];
    g8_transpose4(qa);
    g8_transpose4(qb);
    // the pair's two scales in one dword, then every lane of a row gets the row's four dwords
    const uint32_t dd = __builtin_amdgcn_perm(W[4], W[0], 0x07060100u);
    const auto s = __builtin_amdgcn_permlane16_swap(dd, dd, false, false);      // pairs g & ~1, g | 1
    const auto e = __builtin_amdgcn_permlane32_swap(s[0], s[0], false, false);  // pairs 0, 2
    const auto o = __builtin_amdgcn_permlane32_swap(s[1], s[1], false, false);  // pairs 1, 3
    const uint32_t dp[4] = {e[0], o[0], e[1], o[1]};
    long B[8];
    float d[8];
    uint32_t flip = 0x88888888u, high = 0xF0F0F0F0u;
    asm("" : "+v"(flip), "+v"(high));   // in registers, and not one exclusive or for both halves: (q ^ flip) & high is one instruction
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const uint32_t q = (b & 1) ? qb[b >> 1] : qa[b >> 1];
        B[b] = (long)(((uint64_t)((q ^ flip) & high) << 32) | (uint64_t)(((q << 4) ^ flip) & high));
        d[b] = lev_f16_bits_to_f32((b & 1) ? dp[b >> 1] >> 16 : dp[b >> 1] & 0xFFFFu);
    }
    // a group's eight products are independent: they issue back to back, the sums follow
    auto group = [&](const long (&Aj)[8]) {
        lev_i32x4 acc[8];
#pragma unroll
        for (int b = 0; b < 8; ++b)
            acc[b] = __builtin_amdgcn_mfma_i32_16x16x32_i8(Aj[b], B[b], lev_i32x4{0, 0, 0, 0}, 0, 0, 0);
        float v = 0.f;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            // |plane sum| <= 32 * 128 * 128 = 2^19: two planes recombine in 32 bits, the halves in f32
            const float f = fmaf((float)(acc[b][2] + (acc[b][3] << 8)), 65536.0f, (float)(acc[b][0] + (acc[b][1] << 8)));
            v = fmaf(d[b], f, v);
        }
        return v;
    };
    val[0] = group(A[0]);
#pragma unroll
    for (uint32_t j = 1; j < NJ; ++j) {
        val[j] = 0.f;
        if (j < ng) val[j] = group(A[j]);
    }
#pragma unroll
    for (uint32_t j = 0; j < NJ; ++j) val[j] *= unscale[j];
}

template <int NTILE, bool PAIRED, int NW>
__global__ void __launch_bounds__(NW * LEV_WAVE)
moe_grouped_i8_kernel(lev_moe_grouped_args a, const float *__restrict__ src, const lev_grp_item *__restrict__ items,
                      const lev_grp_start *__restrict__ starts, float *__restrict__ out, uint32_t wpr, uint32_t slots,
                      uint32_t rpi, uint64_t slot_of_wave, uint64_t pos_of_wave) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    constexpr uint32_t NT = kG8NT, NJ = NT / 4u;
    constexpr uint32_t TO = PAIRED ? 1u : (uint32_t)NTILE;       // row groups a slot finishes per round
    constexpr uint32_t kG8Unit = NW * 256u;                       // bytes of part[wave][row][token % 4]: one tile's sums of four tokens
    constexpr uint32_t kG8Batch = g8_batch(NW);
    constexpr uint32_t kHalf = kG8Batch * NTILE * NJ * kG8Unit;   // one parity of `part`: a batch of rounds (with one
                                                                  // token group an item: twice as many rounds)
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t nwaves = blockDim.x >> 6;                      // wpr * slots: every wave has a task
    const uint32_t slot = (uint32_t)(slot_of_wave >> (4u * wave)) & 15u;
    const uint32_t tw = (uint32_t)(pos_of_wave >> (4u * wave)) & 15u;
    const uint32_t in_len = PAIRED ? a.hidden : a.inter, out_rows = PAIRED ? a.inter : a.hidden;
    const uint32_t ngroups = (out_rows + 15u) >> 4;
    const uint64_t row_bytes = (uint64_t)(in_len >> 6) * 36u;
    const uint32_t r = lane & 15u, g = lane >> 4, lrow = lane >> 2;
    // the last task of a row may be a part of one: the pairs and activations past the row's end repeat
    // the row's last ones, and the activations count as zero
    const uint32_t npairs = in_len >> 6, wpair = 4u * tw + (lane & 3u), wpoff = (wpair < npairs ? wpair : npairs - 1u) * 36u;
    const uint32_t a4 = 64u * tw + lane, a4c = a4 < (in_len >> 2) ? a4 : (in_len >> 2) - 1u;

    // this workgroup's stretch of the line of rounds
    const uint32_t G = gridDim.x;
    const uint32_t L = (G & 7u) == 0u ? (blockIdx.x & 7u) * (G >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    // (stretches of equal cost, laid out by the grouping kernel together with the first item's header)
    const lev_grp_start st = starts[L];
    uint32_t R = st.first_round, it = st.item;
    const uint32_t Rend = st.end_round;
    uint32_t e = (uint32_t)st.expert, cnt = (uint32_t)st.count;

    uint8_t *area = smem + 2u * kHalf + (size_t)wave * kG8WaveLds;
    // byte offsets into the workgroup's LDS, not pointers; lane (r, g) writes row r, token 4j + g
    uint32_t pw = ((wave * 16u + r) * 4u + g) * 4u;
    uint32_t half = 0u;                                           // byte offset of the round's parity

    while (R < Rend) {
        const uint32_t r0 = R - it * rpi;
        const uint32_t nr = rpi - r0 < Rend - R ? rpi - r0 : Rend - R;   // rounds r0 .. r0 + nr of item `it`
        // request order = return order: the item's columns (scalar loads), the activations of the
        // wave's task for every token, and the first round's weights behind them, so that the
        // staging does not wait for the weights.  The header of the NEXT item is requested here as
        // well (the list has one record past its end): its expert is known when its turn comes.
        const lev_grp_item *item = items + it;
        const uint32_t e_next = (uint32_t)item[1].expert, cnt_next = (uint32_t)item[1].count;
        const uint32_t ng = (cnt + 3u) >> 2;                      // groups of four tokens that take part
        int32_t pk[NT];
        lev_f32x4 v[NT];
#pragma unroll
        for (uint32_t k = 0; k < NT; ++k) {
            pk[k] = item->pair[k];
            const uint32_t srow = (uint32_t)(PAIRED ? item->src[k] : item->pair[k]);
            v[k] = reinterpret_cast<const lev_f32x4 *>(src + (uint64_t)srow * in_len)[a4c];
        }
        const uint8_t *m0 = a.base + (PAIRED ? a.gate_off + e * a.gate_stride : a.down_off + e * a.down_stride);
        const uint8_t *m1 = PAIRED ? a.base + a.up_off + e * a.up_stride : m0;
        auto issue = [&](uint32_t rho, uint32_t (&D)[NTILE][9]) {
#pragma unroll
            for (int t = 0; t < NTILE; ++t) {
                uint32_t rg = PAIRED ? rho * slots + slot : (rho * slots + slot) * (uint32_t)NTILE + (uint32_t)t;
                rg = rg < ngroups ? rg : ngroups - 1u;
                uint32_t row = rg * 16u + lrow;
                row = row < out_rows ? row : out_rows - 1u;
                lev_q4_load_pair((PAIRED && t == 1 ? m1 : m0) + ((uint64_t)row * row_bytes + wpoff), D[t]);
            }
        };
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t r_last = r0 + nr - 1u;
        uint32_t Da[NTILE][9];
        issue(r0, Da);
        __builtin_amdgcn_sched_barrier(0);
        // the activations are requested for every column, whatever the item's count (columns past
        // the count repeat the last pair), in front of the weights: a request inside the branch
        // below would queue behind them
#pragma unroll
        for (uint32_t k = 0; k < NT; ++k) {
            lev_pin(v[k]);
            if (a4 != a4c) v[k] = lev_f32x4{0.f, 0.f, 0.f, 0.f};
        }
        long A[NJ][8];
        float unscale[NJ];
#pragma unroll
        for (uint32_t j = 0; j < NJ; ++j) {
#pragma unroll
            for (int b = 0; b < 8; ++b) A[j][b] = 0;
            unscale[j] = 0.f;
            if (j < ng) {
                // the area belongs to this wave alone: LDS runs a wave's accesses in order, the fences
                // only keep the compiler from moving reads above writes (and the next group's writes
                // above these reads)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                float us[4];
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) us[k] = g8_stage_token(v[4u * j + k], area + k * kG8TokArea);
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                g8_read_operands(area, A[j]);
                unscale[j] = g == 0u ? us[0] : g == 1u ? us[1] : g == 2u ? us[2] : us[3];
            }
        }
        // the operands are read back before the wait for the weights, not behind it
        __builtin_amdgcn_sched_barrier(0);

        const uint32_t per_round = slots * TO * ng, per_round_inv = 65536u / per_round + 1u;   // (units: fewer than 256)
        int32_t pair_of[NJ];                                      // of token 4j + g
#pragma unroll
        for (uint32_t j = 0; j < NJ; ++j) {
            pair_of[j] = pk[4u * j];
#pragma unroll
            for (uint32_t q = 1; q < 4u; ++q) pair_of[j] = g == q ? pk[4u * j + q] : pair_of[j];
            lev_pin(pair_of[j]);
        }
        uint32_t batch0 = r0, nb = 0u;                            // the batch's first round, rounds in it so far
        const uint32_t round_bytes = NTILE * ng * kG8Unit;        // one round's sums in `part`: [tile][token group][wave][row][token % 4]
        const uint32_t batch_rounds = kG8Batch * NJ / ng;
        auto round = [&](uint32_t rho, uint32_t (&D)[NTILE][9]) {
            // lane (r, g) <- lane 4r + g; the registers the bytes came in take a later round's
            // request at once (unconditional, clamped: a branch around the loads would make the
            // compiler wait for them before this round is multiplied)
            uint32_t W[NTILE][9];
#pragma unroll
            for (int t = 0; t < NTILE; ++t) q4m_turn_task(D[t], W[t]);
            __builtin_amdgcn_sched_barrier(0);
            issue(rho + 1u < r_last ? rho + 1u : r_last, D);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < NTILE; ++t) {
                float val[NJ];
                g8_tile_dot<NJ>(W[t], A, ng, unscale, val);
#pragma unroll
                for (uint32_t j = 0; j < NJ; ++j)
                    if (j < ng)
                        *reinterpret_cast<float *>(smem + half + nb * round_bytes + pw + ((uint32_t)t * ng + j) * kG8Unit) = val[j];
            }
            // the waves meet once per batch of rounds (and at the item's end): between two barriers
            // they run at their own pace, and the batch's sums are finished by several waves at once
            if (++nb < batch_rounds && rho != r_last) return;
            lev_barrier_lds();
            // unit u = (round b of the batch, slot s, row group t of the slot's round, tokens 4j .. 4j + 3):
            // lane (r, g) adds the slot's waves' sums of row r and token 4j + g in a fixed order.  All waves are in this chain
            // at once, 5 of gate/up's 50 us and 4 of down's 30 (2048 / 768, 64 tokens): what an item knows is not computed
            // here (a quotient, the pairs of the lanes), and rows of up to four tasks read no more sums than they have.
            // With the decode of three instructions a block the layer 98.3 -> 96.8 us; two rounds' weights ahead: 107.
            static_assert(NJ <= 2u, "the unit index is split by a shift");
            for (uint32_t u = wave; u < nb * per_round; u += nwaves) {
                const uint32_t b = u * per_round_inv >> 16, ur = u - b * per_round;
                const uint32_t j = ur & (ng - 1u), us_ = ur >> (ng - 1u), s = us_ / TO, t = us_ % TO;
                const uint32_t k = 4u * j + g;
                const uint32_t rg = PAIRED ? (batch0 + b) * slots + s : ((batch0 + b) * slots + s) * (uint32_t)NTILE + t;
                const uint32_t row = rg * 16u + r;
                const float *pp = reinterpret_cast<const float *>(
                    smem + half + b * round_bytes + (t * ng + j) * kG8Unit + ((s * wpr * 16u + r) * 4u + g) * 4u);
                auto slot_sum = [&](const float *q) {
                    float p[8];
                    if (!PAIRED && wpr <= 4u) {
#pragma unroll
                        for (uint32_t w = 0; w < 4u; ++w) p[w] = q[(w < wpr ? w : 0u) * 64u];
#pragma unroll
                        for (uint32_t w = 0; w < 4u; ++w) p[w] = w < wpr ? p[w] : 0.f;
                        return (p[0] + p[2]) + (p[1] + p[3]);
                    }
#pragma unroll
                    for (uint32_t w = 0; w < 8u; ++w) p[w] = q[(w < wpr ? w : 0u) * 64u];   // eight reads in flight
#pragma unroll
                    for (uint32_t w = 0; w < 8u; ++w) p[w] = w < wpr ? p[w] : 0.f;
                    if (NW > 8 && wpr > 8u) {
                        float hi[8];
#pragma unroll
                        for (uint32_t w = 0; w < 8u; ++w) hi[w] = q[(w + 8u < wpr ? w + 8u : 0u) * 64u];
#pragma unroll
                        for (uint32_t w = 0; w < 8u; ++w) p[w] += w + 8u < wpr ? hi[w] : 0.f;
                    }
                    return ((p[0] + p[4]) + (p[2] + p[6])) + ((p[1] + p[5]) + (p[3] + p[7]));
                };
                float res = slot_sum(pp);
                if (PAIRED) res = lev_gelu_up_value(res, slot_sum(pp + ng * (kG8Unit / 4u)));
                const int32_t pair = j == 0u ? pair_of[0] : pair_of[NJ - 1u];
                if (k < cnt && row < out_rows) out[(uint64_t)(uint32_t)pair * out_rows + row] = res;
            }
            half ^= kHalf;
            batch0 = rho + 1u;
            nb = 0u;
        };
        for (uint32_t rho = r0; rho <= r_last; ++rho) round(rho, Da);
        R += nr;
        ++it;
        e = e_next;
        cnt = cnt_next;
    }
}

// 4. merge in slot order (g4_axpy chain, Gemma4.swift:2171-2175); dropped pairs add nothing.
// grid (ceil(hidden / 1024), tokens), 256 threads, four outputs a thread.  Eight slots' rows are
// requested together (a row of a dropped pair was never written: it is read all the same, so that
// no load waits behind a branch, and replaced by zeros), the multiply-adds follow in slot order.
__global__ void __launch_bounds__(256)
moe_merge_kernel(const float *__restrict__ dn, const float *__restrict__ weights,
                 const uint8_t *__restrict__ valid, float *__restrict__ y, uint32_t hidden,
                 uint32_t top_k) {
    const uint32_t t = blockIdx.y, h = (blockIdx.x * 256u + threadIdx.x) * 4u;
    if (h >= hidden) return;
    const bool whole = h + 4u <= hidden && (hidden & 3u) == 0u;   // (hidden is a multiple of 256 on this path)
    lev_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t k0 = 0; k0 < top_k; k0 += 8u) {
        lev_f32x4 v[8];
        float w[8];
        bool ok[8];
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) {
            const uint32_t p = t * top_k + (k0 + u < top_k ? k0 + u : top_k - 1u);
            const float *row = dn + (uint64_t)p * hidden + h;
            if (whole) {
                v[u] = *reinterpret_cast<const lev_f32x4 *>(row);
            } else {
#pragma unroll
                for (uint32_t c = 0; c < 4u; ++c) v[u][c] = h + c < hidden ? row[c] : 0.f;
            }
            w[u] = weights[p];
            ok[u] = valid[p] != 0 && k0 + u < top_k;
        }
#pragma unroll
        for (uint32_t u = 0; u < 8u; ++u) {
            if (k0 + u >= top_k) break;
            const lev_f32x4 vu = ok[u] ? v[u] : lev_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t c = 0; c < 4u; ++c) acc[c] = fmaf(w[u], vu[c], acc[c]);
        }
    }
    if (whole) {
        *reinterpret_cast<lev_f32x4 *>(y + (uint64_t)t * hidden + h) = acc;
    } else {
        for (uint32_t c = 0; c < 4u && h + c < hidden; ++c) y[(uint64_t)t * hidden + h + c] = acc[c];
    }
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct grouped_layout {
    size_t valid, dn, items, starts, total;
};

grouped_layout layout_of(const lev_moe_grouped_args &a) {
    const size_t pairs = (size_t)a.tokens * a.top_k;
    grouped_layout L;
    size_t o = 0;
    L.valid = o; o += align256(pairs);
    L.dn = o; o += align256(pairs * a.hidden * 4);
    L.items = o; o += align256((pairs / 8 + a.experts + 1) * sizeof(lev_grp_item));   // an expert with c pairs: ceil(c / 8) items; one past the end
    L.starts = o; o += 2 * kG8MaxGrid * sizeof(lev_grp_start);
    L.total = o;
    return L;
}

// LDS of the grouping kernel: what it keeps of every expert and of every item (see layout_of).
size_t group_lds(const lev_moe_grouped_args &a) {
    return (size_t)5 * a.experts * 4 + ((size_t)a.tokens * a.top_k / 8 + a.experts + 1) * 4;
}

// Where the integer matrix-core kernels serve: rows of up to 4096 values, one 256-value task per wave, and
// at most eight pairs per expert on average -- they multiply four tokens at a time and are
// the faster ones while most experts hold no more than four or eight pairs; the grouped matrix product
// (moe_prefill.hip) takes 32 at one price.  LEV_MOE_GROUPED_I8=0 never takes them, =1 for any token
// count (for comparison and for the tests).
bool g8_usable(const lev_ctx *ctx, const lev_moe_grouped_args &a) {
    static const int mode = [] {
        const char *v = getenv("LEV_MOE_GROUPED_I8");
        return v && v[0] == '0' ? 0 : v && v[0] == '1' ? 1 : 2;
    }();
    if (mode == 0) return false;
    const bool shape = a.hidden % 64u == 0u && a.hidden <= kG8MaxInLen && a.inter % 64u == 0u && a.inter <= kG8MaxInLen;
    const size_t limit = ctx->props.sharedMemPerBlockOptin > ctx->props.sharedMemPerBlock
                             ? ctx->props.sharedMemPerBlockOptin
                             : ctx->props.sharedMemPerBlock;
    const size_t lds_group = group_lds(a);
    const bool fits = g8_lds<2, kG8WavesWide>() <= limit && g8_lds<2, kG8WavesMax>() <= limit && g8_lds<kG8TilesDown, kG8WavesMax>() <= limit &&
                      lds_group <= limit;
    // (us a layer, these kernels against the grouped product: 2048 / 768, top-8 of 128: 64 tokens 101, 145; 128 tokens
    // 129, 150; 2816 / 704, top-8 of 128: 128 tokens 164, 200; 1408 / 320, top-4 of 64: 128 tokens 58, 58; 3072 / 1024,
    // top-6 of 60: 64 tokens 116, 145; 96 tokens 142, 145; 128 tokens 166, 148.  Measured with 32 experts and more: fewer
    // keep the earlier line of five and a half pairs)
    return shape && fits && (mode == 1 || 2u * (uint64_t)a.tokens * a.top_k <= (a.experts >= 32u ? 16u : 11u) * (uint64_t)a.experts);
}

struct g8_geometry {
    int nw;                     // waves of the kernel's instantiation
    uint32_t wpr, slots, rpi;   // waves a row, row-group slots a workgroup, rounds an item
};
g8_geometry g8_geometry_of(const lev_moe_grouped_args &a, bool paired) {
    const uint32_t in_len = paired ? a.hidden : a.inter, out_rows = paired ? a.inter : a.hidden;
    g8_geometry q;
    q.wpr = (in_len + 255u) >> 8;
    q.nw = paired && q.wpr <= (uint32_t)kG8WavesGateUp ? kG8WavesGateUp : q.wpr <= (uint32_t)kG8WavesWide ? kG8WavesWide : kG8WavesMax;
    q.slots = (uint32_t)q.nw / q.wpr;
    const uint32_t ngroups = (out_rows + 15u) / 16u;
    const uint32_t per_round = q.slots * (paired ? 1u : (uint32_t)kG8TilesDown);   // row groups a round finishes
    q.rpi = (ngroups + per_round - 1u) / per_round;
    return q;
}
static_assert(kG8WavesDown == kG8WavesWide, "one instantiation serves both");

template <int NTILE, bool PAIRED, int NW>
hipError_t g8_launch_as(lev_ctx *ctx, const lev_moe_grouped_args &a, const g8_geometry &q, const float *src,
                        const lev_grp_item *items, const lev_grp_start *starts, uint32_t grid, float *out) {
    uint64_t slot_of_wave, pos_of_wave;
    lev_wave_tables(q.wpr, &slot_of_wave, &pos_of_wave);
    constexpr size_t lds = g8_lds<NTILE, NW>();
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&moe_grouped_i8_kernel<NTILE, PAIRED, NW>), lds); e != hipSuccess) return e;
    hipLaunchKernelGGL((moe_grouped_i8_kernel<NTILE, PAIRED, NW>), dim3(grid), dim3(64u * q.wpr * q.slots), lds,
                       ctx->stream, a, src, items, starts, out, q.wpr, q.slots, q.rpi, slot_of_wave, pos_of_wave);
    return hipGetLastError();
}
template <int NTILE, bool PAIRED>
hipError_t g8_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const g8_geometry &q, const float *src,
                     const lev_grp_item *items, const lev_grp_start *starts, uint32_t grid, float *out) {
    if (PAIRED && q.nw == kG8WavesGateUp)
        return g8_launch_as<NTILE, PAIRED, PAIRED ? kG8WavesGateUp : kG8WavesDown>(ctx, a, q, src, items, starts, grid, out);
    if (q.nw == kG8WavesWide) return g8_launch_as<NTILE, PAIRED, kG8WavesWide>(ctx, a, q, src, items, starts, grid, out);
    return g8_launch_as<NTILE, PAIRED, kG8WavesMax>(ctx, a, q, src, items, starts, grid, out);
}

}  // namespace

hipError_t lev_moe_merge_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const float *dn, const float *weights,
                                const uint8_t *valid, float *y) {
    hipLaunchKernelGGL(moe_merge_kernel, dim3((a.hidden + 1023) / 1024, a.tokens), dim3(256), 0, ctx->stream, dn,
                       weights, valid, y, a.hidden, a.top_k);
    return hipGetLastError();
}

// Grouping costs some 13 us of launches over the kernels that stream an expert for every pair, and saves the
// bytes of the experts that several tokens share (top_k of `experts` each: expected number of distinct
// ones). Those kernels also stream large experts less well: ten experts' worth of bytes.  Where they select the
// experts themselves (`selects`) they save a launch more, and 125 MB is where the two meet (us a layer, grouped
// against per pair: 2816 / 704, top-8 of 128: 5 tokens 52, 40; 12 tokens 76, 71; 15 tokens 84, 85; 2176 / 768, top-4 of
// 60: 15 tokens 50, 45; 3072 / 1408, top-6 of 256: 8 tokens 97, 89; 12 tokens 128, 134); with a selection in front 65 MB
// (2816 / 704: 16 tokens 89, 109; 1408 / 320, top-4 of 64: 16 tokens 39, 31; 64 tokens 50, 57; 1024 / 576, top-2 of 32:
// 32 tokens 34, 31; 64 tokens 36, 45).
// Rows of whole 256-value tasks up to 2048 wide are grouped from five tokens on whatever that saves: from there up to
// eight pairs per expert a token's bits do not depend on how many travel with it (up to four tokens and beyond
// eight pairs other kernels run, and the last bits differ).  It is not for speed: the line above would choose better
// below twelve tokens (us a layer, grouped against pair by pair: 2048 / 768, top-8 of 128: 5 tokens 41, 26; 8 tokens 45,
// 33; 10 tokens 49, 39; 12 tokens 53, 52; 15 tokens 58, 58; 1536 / 768, top-4 of 60: 5 tokens 31, 16; 15 tokens 40, 28).
bool lev_moe_grouped_usable(const lev_ctx *ctx, const lev_moe_grouped_args &a, bool selects) {
    if (!lev_moe_prefill_usable(a)) return false;
    if (a.hidden % 256u == 0u && a.inter % 256u == 0u && a.hidden <= 2048u && a.inter <= 2048u) return true;
    const double expert_bytes = 3.0 * a.hidden * a.inter * 18.0 / 32.0;
    const double distinct = a.experts * (1.0 - std::pow(1.0 - (double)a.top_k / a.experts, (double)a.tokens));
    return ((double)a.tokens * a.top_k - distinct + 10.0) * expert_bytes >= (selects ? 125e6 : 65e6);
}

size_t lev_moe_grouped_scratch_bytes(const lev_ctx *ctx, const lev_moe_grouped_args &a) {
    return g8_usable(ctx, a) ? layout_of(a).total : lev_moe_prefill_scratch_bytes(a);
}

// act: f32 [tokens*top_k][inter] (written here, read by the down stage).
hipError_t lev_moe_grouped_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const float *x,
                                  const int32_t *ids, const float *weights, float *y, float *act,
                                  void *scratch) {
    if (!g8_usable(ctx, a)) return lev_moe_prefill_launch(ctx, a, x, ids, weights, y, act, scratch);
    const grouped_layout L = layout_of(a);
    char *s = static_cast<char *>(scratch);
    uint8_t *valid = reinterpret_cast<uint8_t *>(s + L.valid);
    float *dn = reinterpret_cast<float *>(s + L.dn);
    const uint32_t pairs = a.tokens * a.top_k;
    hipError_t e;

    lev_grp_item *items = reinterpret_cast<lev_grp_item *>(s + L.items);
    lev_grp_start *starts = reinterpret_cast<lev_grp_start *>(s + L.starts);
    const uint32_t grid = (uint32_t)ctx->num_cus < kG8MaxGrid ? (uint32_t)ctx->num_cus : kG8MaxGrid;
    const g8_geometry q_gu = g8_geometry_of(a, true), q_dn = g8_geometry_of(a, false);
    // what a round of an item of up to four pairs and of a larger one cost, relative to each other
    // (gate/up 52 against 62 us, down 33 against 38 with every item of the one or the other kind;
    // equal weights: 62 + 39 us at 64 tokens, these: 58 + 36.5)
    // cost of a round of an item of at most four pairs / of more, and of beginning an item, per kernel.
    // Measured at 64 tokens over 128 experts, us a layer in alternating runs on one box: no cost of
    // beginning 106.4, with it 104.5; down rounds 10:12 103.5, 10:14 101.6, 10:16 103.4 (the items of more
    // than four pairs come first in the line and go to the first XCDs, which finished 8 % after the others
    // at 5:6); gate/up rounds 10:13 and 10:14 no better than 5:6.  Thirteen settings around these, five
    // alternating runs each: medians 101.4 to 103.7, these 102.0
    // (LEV_MOE_CUT="w1,w2,s0,w1,w2,s0", gate/up then down, each 1..64 resp. 0..256: other weights, for measurement)
    static const std::array<uint32_t, 6> cut = [] {
        std::array<uint32_t, 6> c = {5u, 6u, 12u, 10u, 14u, 24u};
        unsigned v[6];
        const char *e = getenv("LEV_MOE_CUT");
        if (e && sscanf(e, "%u,%u,%u,%u,%u,%u", &v[0], &v[1], &v[2], &v[3], &v[4], &v[5]) == 6 && v[0] >= 1u &&
            v[0] <= 64u && v[1] >= 1u && v[1] <= 64u && v[2] <= 256u && v[3] >= 1u && v[3] <= 64u && v[4] >= 1u &&
            v[4] <= 64u && v[5] <= 256u)
            for (int i = 0; i < 6; ++i) c[i] = v[i];
        return c;
    }();
    const uint32_t w1 = cut[0], w2 = cut[1], s0_gu = cut[2], w1_dn = cut[3], w2_dn = cut[4], s0_dn = cut[5];
    const size_t lds_group = group_lds(a);
    if ((e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&moe_group_kernel), lds_group)) != hipSuccess) return e;
    hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(1024), lds_group, ctx->stream, ids, pairs,
                       a.experts, a.top_k, valid, ctx->d_flag, items, starts, grid, q_gu.rpi, q_dn.rpi, w1, w2, w1_dn, w2_dn,
                       s0_gu, s0_dn);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = g8_launch<2, true>(ctx, a, q_gu, x, items, starts, grid, act)) != hipSuccess) return e;
    // rows of act that belong to dropped pairs are never written and never read
    if ((e = g8_launch<kG8TilesDown, false>(ctx, a, q_dn, act, items, starts + grid, grid, dn)) != hipSuccess) return e;
    return lev_moe_merge_launch(ctx, a, dn, weights, valid, y);
}
