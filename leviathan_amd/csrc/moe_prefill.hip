// Routed Q4_0 experts for prompts and large batches on gfx950: a grouped matrix product.  The
// (token, slot) pairs are sorted by expert and cut into items of at most 64 pairs; a workgroup
// multiplies a tile of one expert's rows with all columns of one item.
//
// Stands in for runMoeBatchedRouted applied token after token
// (Sources/LeviathanCore/Gemma4.swift:2073, per-slot loop :3856-3880; moegen_gu/act/dn,
// MoELowering.swift:749-835): same results per pair, same slot-ordered f32 merge.
//
// Pipeline (all on the context's stream):
//   1. group:  expert ids -> list of pairs per expert, items; beside it x as two fp16 planes.
//   2. gate/up -> act = gelu_tanh(g)*u (f32, [pair][inter]).
//   3. planes of act.
//   4. down -> dn (f32, [pair][hidden]).
//   5. merge:  y[t] = sum over slots, IN SLOT ORDER, fmaf(w_slot, dn_slot, acc).
//
// Arithmetic.  Weights enter the matrix cores as the exact integers n - 8 in fp16, one Q4_0 block
// (32 weights) per product; its block scale d is applied to the f32 result, y += d * (A.B), in the
// lane that holds the weight row.  Activations are two fp16 planes, x = hi + lo to one f32 unit, after a
// power-of-two row scale: a finite row loses no more than that down to 2^-17 of its maximum.
// The sums of a row of more than 32 blocks are folded: parts of 16 blocks are added up on their own, then to
// each other.  As one chain of 88 blocks (hidden 2816) an f32 sum gathers 6.6 roundings of its size, folded
// 3.2; against 64-bit sums the layer's outputs are off by 2.2e-7 (2-norm) at 2816 / 704 and 2.3e-7 at
// 4096 / 448 where one chain left 3.0e-7 and 3.5e-7 and the kernels that these sizes took before 2.4e-7.
//
// Measured: hidden 2816, intermediate 704, top-8 of 128 experts, 1000 tokens: the layer 408 us (402 with one
// chain a row; 4420 with a workgroup per token and slot, which these sizes took before); 2048 / 768, 1000
// tokens: 324 us (317; 627 with twelve columns a pass over the weights); 4096 / 448, top-4 of 32, 300 tokens:
// 111 us (131).
//
// What bounds it: per 32 x 32 outputs and block, 4 v_mfma_f32_32x32x16_f16 (128 clocks of the matrix
// pipe) against 16 multiply-adds by d (some 70 clocks of vector issue) and, shared by a wave's two
// token tiles, 24 instructions of decode per row tile; the two kinds overlap between the two waves of a
// SIMD (eight 16x16x32 MFMAs and 32 multiply-adds of four waves: 900 clocks together, 600 and 640
// alone; four 32x32x16 and the same multiply-adds: 760; hence the larger instruction).
#include "moe_prefill.hpp"

#include <cmath>
#include <type_traits>

namespace {

typedef _Float16 p_h8 __attribute__((ext_vector_type(8)));
typedef float p_f16v __attribute__((ext_vector_type(16)));

constexpr int kFlagBadExpertId = 1;          // same bit as the other expert kernels
constexpr uint32_t kPfCols = 64;             // columns (pairs) of an item: two 32-column tiles
constexpr uint32_t kPfStep = 64;             // activations per K-step: two blocks, 128 bytes a row and plane
constexpr uint32_t kPfWRow = 80;             // a weight row's group of four blocks (72 bytes) in LDS: five pieces of 16 bytes
constexpr int kPfFetch = 3;                  // direct loads per group: 160 pieces, 64 a load (the third: half a wave)
constexpr uint32_t kPfWArea = 32 * kPfWRow;  // 32 rows a wave
constexpr uint32_t kPfFold = 8;              // steps (16 blocks) of a part of a folded sum
constexpr uint32_t kPfChain = 32;            // blocks of a row from which on its sums are folded: more

// ---------------------------------------------------------------------------
// Activation planes of one row, by one wave.  The row is scaled by the power of two that brings its
// maximum into [2^14, 2^15) (2^126 at most, which makes multiples of 2^-23 of the subnormal numbers; a row
// with a NaN or an infinity as it is: its results are not finite) and split into fp16 high and low halves;
// at the top of fp16's range the low half of every element down to 2^-17 of the maximum is still a normal
// number.  Run r (eight values) of block b holds elements 8r + 0, 2, 1, 3, 4,
// 6, 5, 7: the weights of code bytes 8(r & 1) .. +7 (r < 2: low nibbles, else high ones) in the order in
// which the masks of the matrix kernel deliver them.
// ---------------------------------------------------------------------------
struct pf_scale { float scale, unscale; };
__device__ __forceinline__ pf_scale pf_row_scale(uint32_t max_bits) {
    uint32_t ex = (max_bits >> 23) & 0xFFu;                    // maximum in [2^(ex - 127), 2^(ex - 126))
    if (ex == 255u) ex = 141u;                                 // (no scaling)
    ex = ex < 15u ? 15u : ex;                                  // keeps both powers of two normal numbers
    return pf_scale{__uint_as_float((268u - ex) << 23), __uint_as_float((ex - 14u) << 23)};   // 2^(141 - ex), 2^(ex - 141)
}

__device__ __forceinline__ void pf_planes_row(const float *__restrict__ row, uint32_t len, _Float16 *__restrict__ h,
                                              _Float16 *__restrict__ l, uint32_t *__restrict__ max_out) {
    const uint32_t lane = threadIdx.x & 63u, runs = len >> 3;
    const lev_f32x4 *s4 = reinterpret_cast<const lev_f32x4 *>(row);
    uint32_t mb = 0u;
    for (uint32_t q = lane; q < 2u * runs; q += 64u) {
        const lev_f32x4 v = s4[q];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t b = __float_as_uint(v[c]) & 0x7FFFFFFFu;
            mb = b > mb ? b : mb;
        }
    }
    mb = lev_wave_max_u32(mb);
    if (lane == 0u) *max_out = mb;
    const float scale = pf_row_scale(mb).scale;
    for (uint32_t q = lane; q < runs; q += 64u) {
        const lev_f32x4 a = s4[2u * q] * scale, b = s4[2u * q + 1u] * scale;
        const float m[8] = {a.x, a.z, a.y, a.w, b.x, b.z, b.y, b.w};
        p_h8 hv, lv;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            hv[k] = (_Float16)m[k];
            lv[k] = (_Float16)(m[k] - (float)hv[k]);
        }
        *reinterpret_cast<p_h8 *>(h + 8u * q) = hv;
        *reinterpret_cast<p_h8 *>(l + 8u * q) = lv;
    }
}

// rows of `src` as planes, a wave per row
__global__ void __launch_bounds__(256)
moe_pf_planes_kernel(const float *__restrict__ src, uint32_t rows, uint32_t len, _Float16 *__restrict__ h,
                     _Float16 *__restrict__ l, uint32_t *__restrict__ max_out) {
    const uint32_t r = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (r >= rows) return;
    pf_planes_row(src + (uint64_t)r * len, len, h + (uint64_t)r * len, l + (uint64_t)r * len, max_out + r);
}

// ---------------------------------------------------------------------------
// Workgroup 0: pairs by expert.  A pair is dropped (and flagged) when its id is out of range or
// repeats another slot's of the same token, as MoEModelBinding.offsets requires
// (MoEModelBinding.swift:174-214); valid[p]: pair p takes part.  glist: the pairs in expert order;
// items: runs of at most kPfCols of them, those of more than 32 pairs (two column tiles, twice the
// work) first.  Workgroups 1..: the planes of x, a wave per token.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024)
moe_pf_group_kernel(const int32_t *__restrict__ ids, uint32_t pairs, uint32_t experts, uint32_t top_k,
                    int32_t *__restrict__ glist, uint8_t *__restrict__ valid, int32_t *__restrict__ ranks,
                    lev_pf_item *__restrict__ items, uint32_t *__restrict__ nitems, int *__restrict__ flag, const float *__restrict__ x,
                    uint32_t tokens, uint32_t hidden, _Float16 *__restrict__ xh, _Float16 *__restrict__ xl,
                    uint32_t *__restrict__ xmax) {
    extern __shared__ int32_t s_cnt[];           // [experts] counts | cursors
    const uint32_t tid = threadIdx.x;
    if (blockIdx.x != 0u) {
        const uint32_t t = (blockIdx.x - 1u) * 16u + (tid >> 6);
        if (t < tokens)
            pf_planes_row(x + (uint64_t)t * hidden, hidden, xh + (uint64_t)t * hidden, xl + (uint64_t)t * hidden, xmax + t);
        return;
    }
    int32_t *s_cur = s_cnt + experts;
    __shared__ uint64_t s_wave[16];
    for (uint32_t e = tid; e < experts; e += 1024u) s_cnt[e] = 0;
    __syncthreads();
    bool bad_seen = false;
    // A thread takes a token, eight of its ids a wait.  The count's atomic gives the pair's place among its expert's: kept in
    // registers for a thread's first eight pairs, in `ranks` (-1: dropped) for others.  With the ids and `valid` read back and a
    // second round of atomics 1000 tokens, top-8 of 128, took 18.5 us here, now 14.4.
    const uint32_t tokens_all = pairs / top_k;
    int32_t first_id[8], first_rank[8];
#pragma unroll
    for (uint32_t u = 0; u < 8u; ++u) first_id[u] = first_rank[u] = -1;
    for (uint32_t t = tid; t < tokens_all; t += 1024u) {
        const int32_t *row = ids + (uint64_t)t * top_k;
        for (uint32_t k0 = 0; k0 < top_k; k0 += 8u) {
            int32_t own[8];
            bool ok[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) own[u] = row[k0 + u < top_k ? k0 + u : k0];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) ok[u] = own[u] >= 0 && (uint32_t)own[u] < experts;
            for (uint32_t j0 = 0; j0 < top_k; j0 += 8u) {
                int32_t other[8];
#pragma unroll
                for (uint32_t v = 0; v < 8u; ++v) other[v] = j0 == k0 ? own[v] : row[j0 + v < top_k ? j0 + v : j0];
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u)
#pragma unroll
                    for (uint32_t v = 0; v < 8u; ++v)
                        if (j0 + v < top_k && j0 + v != k0 + u && other[v] == own[u]) ok[u] = false;
            }
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) {
                if (k0 + u >= top_k) continue;
                valid[(uint64_t)t * top_k + k0 + u] = ok[u] ? 1 : 0;
                bad_seen = bad_seen || !ok[u];
            }
            int32_t rank[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) rank[u] = k0 + u < top_k && ok[u] ? atomicAdd(&s_cnt[own[u]], 1) : -1;
            if (t == tid && k0 == 0u) {
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u) first_id[u] = own[u], first_rank[u] = rank[u];
            } else {
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u)
                    if (k0 + u < top_k) ranks[(uint64_t)t * top_k + k0 + u] = rank[u];
            }
        }
    }
    if (bad_seen) atomicOr(flag, kFlagBadExpertId);
    __syncthreads();
    // exclusive scan over the experts (at most 4096: four a thread) of three counts in 21-bit fields:
    // pairs, items of more than 32 pairs, other items
    uint64_t local = 0;
    int32_t c4[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        const uint32_t e = 4u * tid + k;
        c4[k] = e < experts ? s_cnt[e] : 0;
        const uint32_t full = (uint32_t)c4[k] / kPfCols, rem = (uint32_t)c4[k] % kPfCols;
        local += (uint64_t)c4[k] | (uint64_t)(full + (rem > 32u)) << 21 | (uint64_t)(rem > 0u && rem <= 32u) << 42;
    }
    uint64_t incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t o = __shfl_up(incl, off);
        if ((int)(tid & 63u) >= off) incl += o;
    }
    if ((tid & 63u) == 63u) s_wave[tid >> 6] = incl;
    __syncthreads();
    uint64_t before = incl - local, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 16u; ++w) {
        before += w < (tid >> 6) ? s_wave[w] : 0u;
        all += s_wave[w];
    }
    const uint32_t nbig = (uint32_t)(all >> 21) & 0x1FFFFFu;
    if (tid == 0) *nitems = nbig + (uint32_t)(all >> 42);
    int32_t run = (int32_t)(before & 0x1FFFFFu);
    uint32_t big = (uint32_t)(before >> 21) & 0x1FFFFFu, small = nbig + (uint32_t)(before >> 42);
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        const uint32_t e = 4u * tid + k;
        if (e < experts) s_cur[e] = run;
        for (int32_t j = 0; j < c4[k]; j += (int32_t)kPfCols) {
            const int32_t left = c4[k] - j, count = left < (int32_t)kPfCols ? left : (int32_t)kPfCols;
            items[count > 32 ? big++ : small++] = lev_pf_item{(int32_t)e, run + j, count, 0};
        }
        run += c4[k];
    }
    __syncthreads();
    // The order of an expert's pairs depends on the atomics; no result does: every pair is computed
    // by itself and owns its outputs.
#pragma unroll
    for (uint32_t u = 0; u < 8u; ++u)
        if (first_rank[u] >= 0) glist[s_cur[first_id[u]] + first_rank[u]] = (int32_t)(tid * top_k + u);
    for (uint32_t t = tid; t < tokens_all; t += 1024u)
        for (uint32_t k0 = t == tid ? 8u : 0u; k0 < top_k; k0 += 8u) {
            int32_t own[8], rank[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) {
                const uint32_t p = t * top_k + (k0 + u < top_k ? k0 + u : k0);
                own[u] = ids[p];
                rank[u] = k0 + u < top_k ? ranks[p] : -1;   // (this thread's own)
            }
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u)
                if (rank[u] >= 0) glist[s_cur[own[u]] + rank[u]] = (int32_t)(t * top_k + k0 + u);
        }
}

// ---------------------------------------------------------------------------
// The grouped product.  A wave of a PAIRED (gate/up) workgroup owns 16 rows of the gate matrix and the
// same 16 rows of the up matrix, so that g and u of an output meet in one lane; down: 32 rows.  The
// activation step (64 values of every column, both planes) is shared by the workgroup in LDS, two
// buffers, brought by direct global -> LDS loads; the weights of a wave are its own: 72 bytes of each
// row fetched 16 bytes a lane with consecutive lanes on consecutive bytes, one group of four blocks
// ahead, parked as they lie in memory and decoded by the lane that multiplies them.
// One chain a row (FOLD false): eight waves, 71 KB of LDS and 128 registers, two workgroups per CU whose
// waits cover each other.  Folded, the parts already added take 32 registers more, three waves a SIMD:
// one workgroup of twelve waves a CU, or three of four (pf_waves).
// ---------------------------------------------------------------------------
template <uint32_t WAVES>
struct pf_lds_map {
    static constexpr uint32_t kABuf = 2u * 8u * 1024u;        // two planes x eight regions of eight columns
    static constexpr uint32_t kW = 2u * kABuf;
    static constexpr uint32_t kWBuf = WAVES * kPfWArea;
    static constexpr uint32_t kBytes = kW + 2u * kWBuf;
};

// the four code bytes of one dword -> half a B operand (fp16 integers n - 8): bytes (0, 2), (1, 3) of
// the nibble that `shift` (0 or 4) selects
__device__ __forceinline__ void pf_decode(uint32_t codes, uint32_t mask, uint32_t magic, uint32_t out[2]) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 bias = {(_Float16)1032.0f, (_Float16)1032.0f};
    // 0x6400 | n is the fp16 number 1024 + n
    out[0] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, (codes & mask) | magic) - bias));
    out[1] = __builtin_bit_cast(uint32_t, (f16x2)(__builtin_bit_cast(f16x2, ((codes >> 8) & mask) | magic) - bias));
}

template <bool PAIRED, uint32_t WAVES, bool FOLD, int T>
__device__ __forceinline__ void pf_tile(const lev_moe_grouped_args &a, const lev_pf_item it, uint32_t rt,
                                        const _Float16 *__restrict__ ph, const _Float16 *__restrict__ pl,
                                        const uint32_t *__restrict__ pmax, const int32_t *__restrict__ glist,
                                        float *__restrict__ out, uint8_t *lds, int32_t *s_pair, float *s_us) {
    typedef pf_lds_map<WAVES> L;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t lr = lane & 31u, g = lane >> 5;
    const uint32_t in_len = PAIRED ? a.hidden : a.inter, out_rows = PAIRED ? a.inter : a.hidden;
    const uint32_t nsteps = in_len / kPfStep, nblk = in_len >> 5, row_bytes = nblk * 18u;
    const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane(it.expert), count = (uint32_t)it.count;

    // ---- weights: rows 0..15 of a PAIRED wave's 32 are gate rows, 16..31 the same rows of the up matrix (rows come in
    // whole waves: both row counts are multiples of 64).  Piece q of a group is piece q % 5 of row q / 5: the row's
    // bytes 0, 16, 32, 48 and 56 .. + 15 at 16 bytes a piece, so the fourth block's codes lie at 64, not 56; the last
    // group of a row may hold two blocks (36 bytes): then its third piece is bytes 20 .. 35, the second block's codes ----
    const uint32_t row0 = (rt * WAVES + wave) * (PAIRED ? 16u : 32u);
    const bool live = row0 < out_rows;   // a wave past the last row only brings activations
    const uint32_t lds0 = lev_lds_offset(lds);
    const uint8_t *wsrc[kPfFetch];
    uint32_t wpos = 0u;                  // three bytes: the pieces' positions in a whole group
#pragma unroll
    for (int j = 0; j < kPfFetch; ++j) {
        const uint32_t q = lane + 64u * j < 159u ? lane + 64u * j : 159u, r = q / 5u, i = q - 5u * r;
        const uint32_t row = live ? row0 + (PAIRED ? r & 15u : r) : 0u;
        const uint64_t mat = PAIRED ? (r & 16u ? a.up_off + e * a.up_stride : a.gate_off + e * a.gate_stride)
                                    : a.down_off + e * a.down_stride;
        wpos |= (i < 4u ? 16u * i : 56u) << (8 * j);
        wsrc[j] = a.base + mat + (uint64_t)row * row_bytes;
    }
    const uint32_t ngrp = (nblk + 3u) >> 2;
    auto w_request = [&](uint32_t grp) {
        const uint32_t gc = grp < ngrp ? grp : ngrp - 1u, left = row_bytes - gc * 72u, last = (left < 72u ? left : 72u) - 16u;
        const uint32_t dst = lds0 + L::kW + (grp & 1u) * L::kWBuf + wave * kPfWArea;
#pragma unroll
        for (int j = 0; j < kPfFetch; ++j) {
            const uint32_t at = (wpos >> (8 * j)) & 0xFFu;
            if (j < 2 || lane < 32u) lev_load_lds16(wsrc[j] + (gc * 72u + (at < last ? at : last)), dst + j * 1024u);
        }
    };
    w_request(0);

    // ---- columns ----
    if (tid < kPfCols) {
        const int32_t p = glist[it.first + (int32_t)(tid < count ? tid : count - 1u)];
        s_pair[tid] = p;
        s_us[tid] = pf_row_scale(pmax[PAIRED ? (uint32_t)p / a.top_k : (uint32_t)p]).unscale;
    }
    __syncthreads();

    // ---- activations: load k of a step (T of them a wave) is plane k & 1 of region k / 2; a region is eight
    // columns x eight runs of eight values.  Slot 8 * (run ^ region parity) + ((column & 7) ^ run) of a
    // region: a load's 64 lanes fetch 8 rows x 128 contiguous bytes, and the lanes of a fragment read (32
    // columns, one run each half) hit every bank equally ----
    constexpr uint32_t kALoads = (8u * T + WAVES - 1u) / WAVES;
    const _Float16 *asrc[kALoads];
#pragma unroll
    for (uint32_t j = 0; j < kALoads; ++j) {
        const uint32_t k = wave * kALoads + j < 8u * T ? wave * kALoads + j : 8u * T - 1u, region = k >> 1, run = (lane >> 3) ^ (region & 1u);
        const uint32_t p = (uint32_t)s_pair[region * 8u + ((lane & 7u) ^ run)];
        asrc[j] = (k & 1u ? pl : ph) + (uint64_t)(PAIRED ? p / a.top_k : p) * in_len + run * 8u;
    }
    auto a_request = [&](uint32_t step) {
        const uint32_t s = step < nsteps ? step : nsteps - 1u;   // past the end: any valid step, never read
        const uint32_t dst = lds0 + (step & 1u) * L::kABuf;
#pragma unroll
        for (uint32_t j = 0; j < kALoads; ++j) {
            const uint32_t k = wave * kALoads + j;
            if (kALoads * WAVES == 8u * T || k < 8u * T) lev_load_lds16(asrc[j] + s * kPfStep, dst + (k & 1u) * 8192u + (k >> 1) * 1024u);
        }
    };
    a_request(0);

    float y[T][16], whole[T][16];   // FOLD: the part under way, and the parts before it
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[t][i] = whole[t][i] = 0.f;
    auto fold = [&]() {
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                whole[t][i] += y[t][i];
                y[t][i] = 0.f;
            }
    };
    uint32_t k_mask = 0x000F000Fu, k_magic = 0x64006400u;
    asm("" : "+v"(k_mask), "+v"(k_magic));   // in registers: (v & mask) | magic is one instruction
    const uint8_t *const wmine = lds + L::kW + wave * kPfWArea + lr * kPfWRow;
    const uint32_t areg = (lr >> 3) * 1024u, apar = (lr >> 3) & 1u, acol = lr & 7u;
    uint32_t aoff[4];   // this lane's fragment of half s of block b of a step: aoff[2b + s], + 4096 per column tile, + 8192 for the low plane
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        const uint32_t run = 2u * k + g;
        aoff[k] = areg + ((run ^ apar) * 8u + (acol ^ run)) * 16u;
    }

    auto step_of = [&](uint32_t step, auto odd) {
        constexpr uint32_t st = decltype(odd)::value;   // second step of a group
        // This step's activations have landed: they are the newest loads but for the next group's
        // weights, which are requested behind them in the first step of a group.
        if (st == 1u) LEV_WAIT_VMCNT(kPfFetch);
        else LEV_WAIT_VMCNT(0);
        lev_barrier_lds();   // everybody's have, and everybody is done with the other buffer
        a_request(step + 1u);
        if (st == 0u) w_request((step >> 1) + 1u);
        if (!live) return;
        const uint8_t *const ab = lds + (step & 1u) * L::kABuf;
        const uint8_t *const wb = wmine + ((step >> 1) & 1u) * L::kWBuf + st * 36u;
        // codes and scales of the step's two blocks: code bytes 8g .. 8g + 7 of the first start two bytes
        // behind a dword boundary, those of the second on one
        const uint32_t *const wq = reinterpret_cast<const uint32_t *>(wb + 8u * g);
        const uint32_t at = st == 1u ? 28u : step + 1u == nsteps ? 32u : 20u;   // (see the pieces above)
        const uint32_t *const wo = reinterpret_cast<const uint32_t *>(wb + at + 8u * g);
        const uint32_t q0 = wq[0], q1 = wq[1], q2 = wq[2], q5 = wo[0], q6 = wo[1];
        const _Float16 dh[2] = {*reinterpret_cast<const _Float16 *>(wb), *reinterpret_cast<const _Float16 *>(wb + 18)};
        p_h8 A[2][2][2];   // [unit parity][plane][half of the block]
        auto a_read = [&](uint32_t u) {
            const uint32_t b = u / T, t = u % T;
#pragma unroll
            for (uint32_t s = 0; s < 2u; ++s) {
                const uint8_t *q = ab + aoff[2u * b + s] + t * 4096u;
                A[u & 1u][0][s] = *reinterpret_cast<const p_h8 *>(q);
                A[u & 1u][1][s] = *reinterpret_cast<const p_h8 *>(q + 8192u);
            }
        };
        a_read(0);
        p_h8 B0, B1;
        float d = 0.f;
#pragma unroll
        for (uint32_t u = 0; u < 2u * T; ++u) {   // unit: one block x one column tile
            const uint32_t b = u / T, t = u % T;
            if (t == 0u) {
                const uint32_t c0 = b ? q5 : __builtin_amdgcn_alignbit(q1, q0, 16), c1 = b ? q6 : __builtin_amdgcn_alignbit(q2, q1, 16);
                d = (float)dh[b];
                asm("" : "+v"(d));   // converted once: the mixed-precision multiply-add takes longer than the f32 one
                uint32_t w[8];
                pf_decode(c0, k_mask, k_magic, w);
                pf_decode(c1, k_mask, k_magic, w + 2);
                pf_decode(c0 >> 4, k_mask, k_magic, w + 4);
                pf_decode(c1 >> 4, k_mask, k_magic, w + 6);
                B0 = __builtin_bit_cast(p_h8, lev_u32x4{w[0], w[1], w[2], w[3]});
                B1 = __builtin_bit_cast(p_h8, lev_u32x4{w[4], w[5], w[6], w[7]});
            }
            // the next unit's fragments are requested ahead of this unit's products
            if (u + 1u < 2u * T) a_read(u + 1u);
            __builtin_amdgcn_sched_barrier(0);
            const p_h8(&F)[2][2] = A[u & 1u];
            p_f16v acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(F[0][0], B0, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(F[0][1], B1, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(F[1][0], B0, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(F[1][1], B1, acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; ++i) y[t][i] = fmaf(d, acc[i], y[t][i]);
        }
    };
    for (uint32_t step = 0; step < nsteps; step += 2u) {
        step_of(step, std::integral_constant<uint32_t, 0>());
        if (step + 1u < nsteps) step_of(step + 1u, std::integral_constant<uint32_t, 1>());
        if (FOLD && (step & (kPfFold - 2u)) == kPfFold - 2u) fold();
    }
    if (FOLD) fold();
    float(&sum)[T][16] = FOLD ? whole : y;

    LEV_WAIT_VMCNT(0);   // the request past the end lands before the LDS is given back
    if (!live) return;
    // lane (lr, g), register i of a tile: weight row lr, column 8 (i / 4) + 4 g + i % 4
    const uint32_t row = row0 + (PAIRED ? lr & 15u : lr);
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 16; i += PAIRED ? 2 : 1) {
            uint32_t col = 32u * t + 8u * (i / 4) + 4u * g + (i % 4);
            float v = sum[t][i];
            if (PAIRED) {
                // lanes 0..15 of a half hold gate rows, 16..31 the same up rows: two columns trade halves, so
                // that every lane has a gate and its up value, of column i in lanes 0..15, of i + 1 in 16..31
                const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(sum[t][i + 1]), false, false);
                col += lr >> 4;
                const float us = s_us[col];
                v = lev_gelu_up_value(__uint_as_float(sw[0]) * us, __uint_as_float(sw[1]) * us);
            } else {
                v = v * s_us[col];
            }
            if (col < count) out[(uint64_t)(uint32_t)s_pair[col] * out_rows + row] = v;
        }
}

// grid: 8 * ceil(items / 8) * row tiles, in one line.  Workgroups go to the XCDs in turn, so item 8j + c
// sits on XCD c with all its row tiles, which read the same activations through one L2.
template <bool PAIRED, uint32_t WAVES, bool FOLD>
__global__ void __launch_bounds__(WAVES * 64, FOLD ? 3 : 4)
moe_pf_kernel(lev_moe_grouped_args a, uint32_t row_tiles, const _Float16 *__restrict__ ph,
              const _Float16 *__restrict__ pl, const uint32_t *__restrict__ pmax, const int32_t *__restrict__ glist,
              const lev_pf_item *__restrict__ items, const uint32_t *__restrict__ nitems, float *__restrict__ out) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    __shared__ int32_t s_pair[kPfCols];
    __shared__ float s_us[kPfCols];
    const uint32_t j = blockIdx.x >> 3, at = (j / row_tiles) * 8u + (blockIdx.x & 7u), rt = j % row_tiles;
    if (at >= *nitems) return;
    const lev_pf_item it = items[at];
    if (it.count > 32) pf_tile<PAIRED, WAVES, FOLD, 2>(a, it, rt, ph, pl, pmax, glist, out, smem, s_pair, s_us);
    else pf_tile<PAIRED, WAVES, FOLD, 1>(a, it, rt, ph, pl, pmax, glist, out, smem, s_pair, s_us);
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct pf_layout {
    size_t glist, valid, items, nitems, xh, xl, xmax, ah, al, amax, dn, total;
};
size_t pf_max_items(const lev_moe_grouped_args &a) {
    const size_t pairs = (size_t)a.tokens * a.top_k;
    return pairs / kPfCols + (a.experts < pairs ? a.experts : pairs);
}
pf_layout pf_layout_of(const lev_moe_grouped_args &a) {
    const size_t pairs = (size_t)a.tokens * a.top_k;
    pf_layout L;
    size_t o = 0;
    L.glist = o; o += align256(pairs * 4);
    L.valid = o; o += align256(pairs);
    L.items = o; o += align256(pf_max_items(a) * sizeof(lev_pf_item));
    L.nitems = o; o += 256;
    L.xh = o; o += align256((size_t)a.tokens * a.hidden * 2);
    L.xl = o; o += align256((size_t)a.tokens * a.hidden * 2);
    L.xmax = o; o += align256((size_t)a.tokens * 4);
    L.ah = o; o += align256(pairs * a.inter * 2);
    L.al = o; o += align256(pairs * a.inter * 2);
    L.amax = o; o += align256(pairs * 4);
    L.dn = o; o += align256(pairs * a.hidden * 4);
    L.total = o;
    return L;
}

template <bool PAIRED, uint32_t WAVES, bool FOLD>
hipError_t pf_launch_as(lev_ctx *ctx, const lev_moe_grouped_args &a, const _Float16 *ph, const _Float16 *pl, const uint32_t *pmax,
                        const int32_t *glist, const lev_pf_item *items, const uint32_t *nitems, float *out) {
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&moe_pf_kernel<PAIRED, WAVES, FOLD>), pf_lds_map<WAVES>::kBytes);
        e != hipSuccess)
        return e;
    const uint32_t slots = (uint32_t)((pf_max_items(a) + 7u) / 8u) * 8u;
    const uint32_t rows = PAIRED ? a.inter : a.hidden, per_wg = WAVES * (PAIRED ? 16u : 32u), tiles = (rows + per_wg - 1u) / per_wg;
    hipLaunchKernelGGL((moe_pf_kernel<PAIRED, WAVES, FOLD>), dim3(slots * tiles), dim3(WAVES * 64u), pf_lds_map<WAVES>::kBytes,
                       ctx->stream, a, tiles, ph, pl, pmax, glist, items, nitems, out);
    return hipGetLastError();
}

// Waves of a folded workgroup.  Three of four waves share a CU where one of twelve has it to itself: they read the
// activations three times, and their last round is finer.  So twelve where whole rounds of them come near the
// work there is (us a layer with twelve, with four: 2816 / 704, top-8 of 128: 1000 tokens, 2.9 rounds, 393, 409; 300
// tokens, 2 rounds, 209, 217; 2048 / 768, 1000 tokens, 310, 330; 1536 / 1088, top-4 of 60, 600 tokens, 1.5 rounds, 155,
// 147; 2304 / 1280, top-2 of 32, 1000 tokens, 1.3 rounds, 184, 167; 4096 / 448, top-4 of 32, 300 tokens, 0.4 rounds, 149,
// 105).  Items: one an expert that has pairs, and half an item more where they are many.
uint32_t pf_waves(const lev_ctx *ctx, const lev_moe_grouped_args &a, uint32_t out_rows, uint32_t rows_a_wave) {
    const double mean = (double)a.tokens * a.top_k / a.experts;
    const double items = a.experts * std::fmax(1.0 - std::exp(-mean), mean / kPfCols + 0.5);
    const double rounds = items * ((out_rows + 12u * rows_a_wave - 1u) / (12u * rows_a_wave)) / ctx->num_cus;
    return 0.95 * std::ceil(rounds) <= rounds + 0.25 ? 12u : 4u;
}

template <bool PAIRED>
hipError_t pf_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const _Float16 *ph, const _Float16 *pl, const uint32_t *pmax,
                     const int32_t *glist, const lev_pf_item *items, const uint32_t *nitems, float *out) {
    if ((PAIRED ? a.hidden : a.inter) <= 32u * kPfChain)
        return pf_launch_as<PAIRED, 8, false>(ctx, a, ph, pl, pmax, glist, items, nitems, out);
    if (pf_waves(ctx, a, PAIRED ? a.inter : a.hidden, PAIRED ? 16u : 32u) == 12u)
        return pf_launch_as<PAIRED, 12, true>(ctx, a, ph, pl, pmax, glist, items, nitems, out);
    return pf_launch_as<PAIRED, 4, true>(ctx, a, ph, pl, pmax, glist, items, nitems, out);
}

}  // namespace

size_t lev_moe_prefill_scratch_bytes(const lev_moe_grouped_args &a) { return pf_layout_of(a).total; }

// (the caller also checks 4-byte aligned pools and 16-byte aligned x)
bool lev_moe_prefill_usable(const lev_moe_grouped_args &a) {
    const uint64_t gu = (uint64_t)a.inter * (a.hidden / 32u) * 18u;
    return a.hidden % 64u == 0u && a.inter % 64u == 0u && a.experts <= 4096u &&
           (uint64_t)a.tokens * a.top_k <= (1u << 20) && gu < (1ull << 32);
}

// act: f32 [tokens*top_k][inter] (written here).
hipError_t lev_moe_prefill_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const float *x, const int32_t *ids,
                                  const float *weights, float *y, float *act, void *scratch) {
    const pf_layout L = pf_layout_of(a);
    char *s = static_cast<char *>(scratch);
    int32_t *glist = reinterpret_cast<int32_t *>(s + L.glist);
    uint8_t *valid = reinterpret_cast<uint8_t *>(s + L.valid);
    lev_pf_item *items = reinterpret_cast<lev_pf_item *>(s + L.items);
    uint32_t *nitems = reinterpret_cast<uint32_t *>(s + L.nitems);
    _Float16 *xh = reinterpret_cast<_Float16 *>(s + L.xh), *xl = reinterpret_cast<_Float16 *>(s + L.xl);
    _Float16 *ah = reinterpret_cast<_Float16 *>(s + L.ah), *al = reinterpret_cast<_Float16 *>(s + L.al);
    uint32_t *xmax = reinterpret_cast<uint32_t *>(s + L.xmax), *amax = reinterpret_cast<uint32_t *>(s + L.amax);
    float *dn = reinterpret_cast<float *>(s + L.dn);
    const uint32_t pairs = a.tokens * a.top_k;
    hipError_t e;
    hipLaunchKernelGGL(moe_pf_group_kernel, dim3(1u + (a.tokens + 15u) / 16u), dim3(1024), (size_t)2 * a.experts * 4,
                       ctx->stream, ids, pairs, a.experts, a.top_k, glist, valid, reinterpret_cast<int32_t *>(dn), items, nitems, ctx->d_flag, x,
                       a.tokens, a.hidden, xh, xl, xmax);   // (the ranks are in the place of dn, which comes much later)
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = pf_launch<true>(ctx, a, xh, xl, xmax, glist, items, nitems, act)) != hipSuccess) return e;
    // rows of act that belong to dropped pairs were never written: their planes are never read
    hipLaunchKernelGGL(moe_pf_planes_kernel, dim3((pairs + 3u) / 4u), dim3(256), 0, ctx->stream, act, pairs, a.inter, ah,
                       al, amax);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = pf_launch<false>(ctx, a, ah, al, amax, glist, items, nitems, dn)) != hipSuccess) return e;
    return lev_moe_merge_launch(ctx, a, dn, weights, valid, y);
}
