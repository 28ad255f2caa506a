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
// What bounds it: instructions.  A unit, 32 x 32 outputs and a block, is 4 v_mfma_f32_32x32x16_f16 (130 clocks of the matrix
// pipe), 16 multiply-adds by d, 4 fragment reads, and per row 18 instructions of decode shared by the item's column tiles: some
// 45 in all, and a SIMD's two to four waves issue one per 4.4 to 5 clocks, whatever its kind; over the whole chip the products
// alone run at 1.45 GHz (92 ns a unit and SIMD, 117 with the rest).  So the loop is written for their number (three buffers
// of activations, weights read 8 bytes a lane, two codes decoded by three instructions) and for what the others cover: fragments and
// weights of the next step are read and decoded behind this step's products, requests are issued one behind a product, and
// a workgroup's start is three dependent trips to memory (nine thousand clocks of a down product's 42 thousand before).
//
// Measured (us, the two products, before -> now; 2816 / 704, top-8 of 128 experts): 1000 tokens 231 + 117 -> 208 + 108; 300 tokens
// 114 + 62 -> 110 + 59; 2048 / 768, 1000 tokens 167 + 89 -> 156 + 82; 1024 / 256, top-4 of 32, 300 tokens 23 + 9.9 -> 18.6 + 8.7;
// 4096 / 1536, top-6 of 64, 500 tokens 277 + 149 -> 224 + 133; 4096 / 832, top-4 of 128, 420 tokens 205 + 93 -> 186 + 89.
// Tried and not kept: 64 rows a wave (half the fragment reads: no faster, the registers of two folded tiles spill), items of 96
// (203 + 113), deeper requests, wave priorities.
#include "moe_prefill.hpp"
#include "moe_prefill_plan.hpp"

#include <type_traits>

namespace {

typedef _Float16 p_h8 __attribute__((ext_vector_type(8)));
typedef float p_f16v __attribute__((ext_vector_type(16)));

constexpr int kFlagBadExpertId = 1;          // same bit as the other expert kernels
constexpr uint32_t kPfListLds = 16384;       // pairs up to which, from a quarter on, the grouping kernel puts their list together in LDS
constexpr uint32_t kPfStep = 64;             // activations per K-step: two blocks, 128 bytes a row and plane
constexpr int kPfFetch = 3;                  // direct loads per group: 160 pieces, 64 a load (the third: half a wave)
constexpr uint32_t kPfWRow = 80;             // a weight row's group of four blocks (72 bytes) in LDS: five pieces of 16 bytes
constexpr uint32_t kPfFold = 8;              // steps (16 blocks) of a part of a folded sum

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

__host__ __device__ constexpr bool pf_list_in_lds(uint32_t pairs) { return pairs > kPfListLds / 4u && pairs <= kPfListLds; }

// ---------------------------------------------------------------------------
// Workgroup 0: pairs by expert.  A pair is dropped (and flagged) when its id is out of range or
// repeats another slot's of the same token, as MoEModelBinding.offsets requires
// (MoEModelBinding.swift:174-214); valid[p]: pair p takes part.  glist: the pairs in expert order;
// items: runs of at most `cols` of them (64 or 32), those of more than 32 pairs (two column tiles, twice the
// work) first.  Workgroups 1..: the planes of x, a wave per token.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024)
moe_pf_group_kernel(const int32_t *__restrict__ ids, uint32_t pairs, uint32_t experts, uint32_t top_k,
                    int32_t *__restrict__ glist, uint8_t *__restrict__ valid, int32_t *__restrict__ ranks,
                    lev_pf_item *__restrict__ items, uint32_t *__restrict__ nitems, int *__restrict__ flag, const float *__restrict__ x,
                    uint32_t tokens, uint32_t hidden, _Float16 *__restrict__ xh, _Float16 *__restrict__ xl,
                    uint32_t *__restrict__ xmax, uint32_t cols) {
    extern __shared__ int32_t s_cnt[];           // [experts] counts | cursors | a count of dropped pairs, never read | the list
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
    lev_barrier_lds();
    bool bad_seen = false;
    // A thread takes a token, eight of its ids a wait.  The count's atomic gives the pair's place among its expert's: kept in
    // registers for a thread's first eight pairs, in `ranks` (-1: dropped) for others.
    const uint32_t tokens_all = pairs / top_k;
    // (a token's eight ids by two loads: a dword a lane at a stride of 32 bytes keeps the address unit busy for 64 clocks a load)
    const bool wide = top_k == 8u && (reinterpret_cast<uintptr_t>(ids) & 15u) == 0u;
    int32_t first_id[8], first_rank[8];
#pragma unroll
    for (uint32_t u = 0; u < 8u; ++u) first_id[u] = first_rank[u] = -1;
    for (uint32_t t = tid; t < tokens_all; t += 1024u) {
        const int32_t *row = ids + (uint64_t)t * top_k;
        for (uint32_t k0 = 0; k0 < top_k; k0 += 8u) {
            int32_t own[8];
            bool ok[8];
            if (wide) {
                typedef int32_t i4 __attribute__((ext_vector_type(4)));
                const i4 a = reinterpret_cast<const i4 *>(row)[0], b = reinterpret_cast<const i4 *>(row)[1];
#pragma unroll
                for (uint32_t u = 0; u < 4u; ++u) own[u] = a[u], own[4u + u] = b[u];
            } else {
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u) own[u] = row[k0 + u < top_k ? k0 + u : k0];
            }
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) ok[u] = own[u] >= 0 && (uint32_t)own[u] < experts;
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u)
#pragma unroll
                for (uint32_t v = 0; v < u; ++v)
                    if (k0 + u < top_k && own[u] == own[v]) ok[u] = ok[v] = false;
            for (uint32_t j0 = 0; j0 < top_k; j0 += 8u) {
                if (j0 == k0) continue;
                int32_t other[8];
#pragma unroll
                for (uint32_t v = 0; v < 8u; ++v) other[v] = row[j0 + v < top_k ? j0 + v : j0];
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u)
#pragma unroll
                    for (uint32_t v = 0; v < 8u; ++v)
                        if (j0 + v < top_k && other[v] == own[u]) ok[u] = false;
            }
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) {
                ok[u] = ok[u] && k0 + u < top_k;
                bad_seen = bad_seen || (!ok[u] && k0 + u < top_k);
            }
            int32_t rank[8];
            pf_rank_pairs(own, ok, k0, top_k, experts, [&](uint32_t word) { return atomicAdd(&s_cnt[word], 1); }, rank);
            if (top_k == 8u) {
                uint64_t eight = 0;
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u) eight |= (uint64_t)(ok[u] ? 1 : 0) << (8u * u);
                reinterpret_cast<uint64_t *>(valid)[t] = eight;
            } else {
#pragma unroll
                for (uint32_t u = 0; u < 8u; ++u)
                    if (k0 + u < top_k) valid[(uint64_t)t * top_k + k0 + u] = ok[u] ? 1 : 0;
            }
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
    lev_barrier_lds();
    // exclusive scan over the experts (at most 4096: up to four a thread, side by side) of three counts in 21-bit fields:
    // pairs, items of more than 32 pairs, other items
    const uint32_t per_thread = (experts + 1023u) >> 10;
    uint64_t local = 0, before, all;
    int32_t c4[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        if (k >= per_thread) break;
        const uint32_t e = per_thread * tid + k;
        c4[k] = e < experts ? s_cnt[e] : 0;
        const uint32_t full = (uint32_t)c4[k] / cols, rem = (uint32_t)c4[k] % cols;
        local += (uint64_t)c4[k] | (uint64_t)((cols > 32u ? full : 0u) + (rem > 32u)) << 21 |
                 (uint64_t)((cols > 32u ? 0u : full) + (rem > 0u && rem <= 32u)) << 42;
    }
    lev_scan_1024(local, s_wave, before, all);
    const uint32_t nbig = (uint32_t)(all >> 21) & 0x1FFFFFu;
    if (tid == 0) *nitems = nbig + (uint32_t)(all >> 42);
    int32_t run = (int32_t)(before & 0x1FFFFFu);
    uint32_t big = (uint32_t)(before >> 21) & 0x1FFFFFu, small = nbig + (uint32_t)(before >> 42);
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        if (k >= per_thread) break;
        const uint32_t e = per_thread * tid + k;
        if (e < experts) s_cur[e] = run;
        for (int32_t j = 0; j < c4[k]; j += (int32_t)cols) {
            const int32_t left = c4[k] - j, count = left < (int32_t)cols ? left : (int32_t)cols;
            items[count > 32 ? big++ : small++] = lev_pf_item{(int32_t)e, run + j, count, 0};
        }
        run += c4[k];
    }
    lev_barrier_lds();
    // The order of an expert's pairs depends on the atomics; no result does: every pair is computed
    // by itself and owns its outputs.  A long list is put together in LDS where it fits (64 lanes that store to 64 places of memory
    // take the address unit 64 clocks) and stored as it lies there.  us stored in place and so, top-8 of 128 experts: 2000 pairs 5.1
    // and 5.2, 4160 7.2 and 6.4, 8000 9.5 and 7.4, 16000 24.2 and 19.0; top-2 of 32 4200 13.0 and 12.7, top-1 4200 19.6 and 20.0.
    // (Longer lists gain too, 28000 46.2 and 35.5: not taken, with 4096 experts' counts that is nine tenths of a CU's LDS.)
    const bool in_lds = pf_list_in_lds(pairs);
    int32_t *const s_list = s_cnt + 2u * experts + 1u;
    auto place = [&](int32_t e, int32_t rank, uint32_t pair) {
        if (rank < 0) return;
        const uint32_t at = (uint32_t)(s_cur[e] + rank);
        if (in_lds) s_list[at] = (int32_t)pair;
        else glist[at] = (int32_t)pair;
    };
#pragma unroll
    for (uint32_t u = 0; u < 8u; ++u) place(first_rank[u] >= 0 ? first_id[u] : 0, first_rank[u], tid * top_k + u);
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
            for (uint32_t u = 0; u < 8u; ++u) place(rank[u] >= 0 ? own[u] : 0, rank[u], t * top_k + k0 + u);
        }
    if (!in_lds) return;
    lev_barrier_lds();
    const uint32_t listed = (uint32_t)(all & 0x1FFFFFu);   // pairs that take part
    for (uint32_t i = tid; i < listed; i += 1024u) glist[i] = s_list[i];
}

// ---------------------------------------------------------------------------
// The grouped product.  A wave of a PAIRED (gate/up) workgroup owns 16 rows of the gate matrix and the
// same 16 rows of the up matrix, so that g and u of an output meet in one lane; down: 32 rows.  The
// activation step (64 values of every column, both planes) is shared by the workgroup in LDS, two
// or three buffers, brought by direct global -> LDS loads; the weights of a wave are its own: 72 bytes of each
// row fetched 16 bytes a lane with consecutive lanes on consecutive bytes, one group of four blocks
// ahead, parked as they lie in memory and decoded by the lane that multiplies them.
// One chain a row (FOLD false): eight waves, two buffers, 72 KB of LDS and 128 registers, two workgroups per CU whose
// waits cover each other.  Folded, the parts already added take up to 32 registers more: pf_estimate chooses among four forms.
// ---------------------------------------------------------------------------
template <uint32_t WAVES, uint32_t TMAX, uint32_t NBUF>
struct pf_lds_map {
    static constexpr uint32_t kPlane = TMAX * 4096u;          // four regions of eight columns a column tile
    static constexpr uint32_t kABuf = 2u * kPlane;
    static constexpr uint32_t kW = NBUF * kABuf;
    static constexpr uint32_t kWArea = 32u * kPfWRow;         // 32 rows a wave
    static constexpr uint32_t kWBuf = WAVES * kWArea;
    static constexpr uint32_t kBytes = kW + 2u * kWBuf;
};

// lev_load_lds16 for the lanes of a mask, of a wave that has all its lanes: without a branch, which would end the region in
// which products and requests are ordered.
__device__ __forceinline__ void pf_load_lds16_of(const void *src, uint32_t dst, uint32_t lanes_lo, uint32_t lanes_hi) {
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b32 exec_lo, %2\n\ts_mov_b32 exec_hi, %3\n\tglobal_load_lds_dwordx4 %0, off\n\ts_mov_b64 exec, -1"
                 ::"v"(src), "s"(dst), "s"(lanes_lo), "s"(lanes_hi) : "memory");
}
constexpr __host__ __device__ uint32_t pf_min(uint32_t a, uint32_t b) { return a < b ? a : b; }

// A block's 16 codes of a lane, two dwords (code bytes 8g .. 8g + 7) -> the operands of both halves, fp16 integers n - 8.
// 0x6400 | n is the fp16 number 1024 + n, 0x6400 | 16 n is 1024 + 16 n: a subtraction and a multiply-add, both exact.
template <bool SCALAR>
struct pf_consts {
    uint32_t low = 0x000F000Fu, high = 0x00F000F0u, magic = 0x64006400u;
    lev_f16x2 m1032 = {(_Float16)-1032.0f, (_Float16)-1032.0f}, sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f}, m72 = {(_Float16)-72.0f, (_Float16)-72.0f};
    // (in registers: (v & mask) | magic is one instruction, of which one operand may be a scalar register's)
    __device__ __forceinline__ pf_consts() {
        if constexpr (SCALAR) asm("" : "+s"(low), "+s"(high), "+v"(magic));
        else asm("" : "+v"(low), "+v"(high), "+v"(magic));
    }
};
template <bool SCALAR>
__device__ __forceinline__ void pf_decode(uint32_t c, const pf_consts<SCALAR> &k, uint32_t &low, uint32_t &high) {
    low = __builtin_bit_cast(uint32_t, (lev_f16x2)(__builtin_bit_cast(lev_f16x2, (c & k.low) | k.magic) + k.m1032));
    high = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(lev_f16x2, (c & k.high) | k.magic), k.sixteenth, k.m72));
}

template <bool PAIRED, uint32_t WAVES, uint32_t TMAX, uint32_t OCC, uint32_t NBUF, bool FOLD, uint32_t T>
__device__ __forceinline__ void pf_tile(const lev_moe_grouped_args &a, const lev_pf_item it, uint32_t rt,
                                        const _Float16 *__restrict__ ph, const _Float16 *__restrict__ pl,
                                        const uint32_t *__restrict__ pmax, const int32_t *__restrict__ glist,
                                        float *__restrict__ out, uint8_t *lds, int32_t *s_pair, float *s_us) {
    typedef pf_lds_map<WAVES, TMAX, NBUF> L;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t lr = lane & 31u, g = lane >> 5;
    const uint32_t in_len = PAIRED ? a.hidden : a.inter, out_rows = PAIRED ? a.inter : a.hidden;
    const uint32_t nsteps = in_len / kPfStep, nblk = in_len >> 5, row_bytes = nblk * 18u;
    const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane(it.expert), count = (uint32_t)it.count;

    // ---- weights: rows 0..15 of a PAIRED wave's 32 are gate rows, 16..31 the same rows of the up matrix (rows come in
    // whole waves: both row counts are multiples of 64).  Piece q of a group is piece q % 5 of row q / 5: the row's
    // bytes 0, 16, 32, 48 and 56 .. + 15 at 16 bytes a piece, so its last 8 bytes lie at 72, not 64; the last
    // group of a row may hold two blocks (36 bytes): then its third piece is bytes 20 .. 35 ----
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
    auto w_request = [&](uint32_t grp, uint32_t j) {
        const uint32_t gc = grp < ngrp ? grp : ngrp - 1u, left = row_bytes - gc * 72u, last = (left < 72u ? left : 72u) - 16u;
        const uint32_t dst = lds0 + L::kW + (grp & 1u) * L::kWBuf + wave * L::kWArea;
        const uint32_t at = (wpos >> (8 * j)) & 0xFFu;
        const uint8_t *const src = wsrc[j] + (gc * 72u + (at < last ? at : last));
        if (j == 2u) pf_load_lds16_of(src, dst + 2048u, ~0u, 0u);
        else lev_load_lds16(src, dst + j * 1024u);
    };

    // ---- activations: load k of a step is plane k & 1 of region k / 2; a region is eight
    // columns x eight runs of eight values.  Slot 8 * (run ^ region parity) + ((column & 7) ^ run) of a
    // region: a load's 64 lanes fetch 8 rows x 128 contiguous bytes, and the lanes of a fragment read (32
    // columns, one run each half) hit every bank equally ----
    // A wave that has fewer than the others brings one lane's piece of the last load once more (the same bytes to the same
    // place): every wave has as many requests in flight, which the waits count.
    constexpr uint32_t kALoads = (8u * T + WAVES - 1u) / WAVES;
    constexpr bool kAll = 8u * T == WAVES * kALoads;
    const _Float16 *asrc[kALoads];
#pragma unroll
    for (uint32_t j = 0; j < kALoads; ++j) {
        const uint32_t k = pf_min(wave * kALoads + j, 8u * T - 1u), region = k >> 1, run = (lane >> 3) ^ (region & 1u);
        const uint32_t col = region * 8u + ((lane & 7u) ^ run), p = (uint32_t)glist[it.first + (int32_t)(col < count ? col : count - 1u)];
        asrc[j] = (k & 1u ? pl : ph) + (uint64_t)(PAIRED ? p / a.top_k : p) * in_len + run * 8u;
    }
    int32_t own_pair = 0;     // a column's pair and scale, wanted at the end
    uint32_t own_max = 0u;
    if (tid < 32u * T) {
        own_pair = glist[it.first + (int32_t)(tid < count ? tid : count - 1u)];
        own_max = pmax[PAIRED ? (uint32_t)own_pair / a.top_k : (uint32_t)own_pair];
    }
    // (up to two steps past the end of a row, which lie in front of something else of the scratch: read, never used)
    auto a_request = [&](uint32_t buf, uint32_t j) {
        const uint32_t n = wave * kALoads + j, k = pf_min(n, 8u * T - 1u), dst = lds0 + buf + (k & 1u) * L::kPlane + (k >> 1) * 1024u;
        if (kAll) {
            lev_load_lds16(asrc[j], dst);
        } else {
            const uint32_t all = (uint32_t)__builtin_amdgcn_readfirstlane(n < 8u * T ? -1 : 0);
            pf_load_lds16_of(asrc[j], dst, all | 1u, all);
        }
        asrc[j] += kPfStep;
    };
#pragma unroll
    for (uint32_t j = 0; j < kALoads; ++j) a_request(0u, j);
#pragma unroll
    for (uint32_t j = 0; j < kPfFetch; ++j) w_request(0u, j);
    if (NBUF == 3u) {
#pragma unroll
        for (uint32_t j = 0; j < kALoads; ++j) a_request(L::kABuf, j);
    }

    // The buffers of this step's activations, of the next's and of the one's to be requested.  Three: at the start of a step
    // the next step's have landed, every wave's, and a wave reads its first fragments of a step behind the products of
    // the step before, not behind the barrier.  Two: this step's have landed, the next's are requested.
    uint32_t buf0 = 0u, buf1 = L::kABuf, buf2 = (NBUF - 1u) * L::kABuf;
    auto bring = [&](uint32_t step, auto kind) {
        // (newer than the activations waited for: the next group's weights, requested in the first step of a group)
        if (decltype(kind)::value == 1u) LEV_WAIT_VMCNT(kPfFetch);
        else LEV_WAIT_VMCNT(0);
        lev_barrier_lds();   // and everybody is done with the step before
    };
    // A step's requests, one behind a product each: issued together behind the barrier, by all waves, they waited in the issue
    // for 300 to 570 of a step's 2300 clocks.
    auto requests = [&](uint32_t step, auto kind, uint32_t b, uint32_t slot) {   // slot: of the 4 T products of a block
        if (b == 0u) {
#pragma unroll
            for (uint32_t j = 0; j < kALoads; ++j)
                if (slot == j * (4u * T / kALoads)) a_request(buf2, j);
        } else if (decltype(kind)::value != 1u) {
#pragma unroll
            for (uint32_t j = 0; j < kPfFetch; ++j)
                if (slot == j * (4u * T / 3u)) w_request((step >> 1) + 1u, j);
        }
    };
    auto turn = [&]() {
        const uint32_t b = buf0;
        if (NBUF == 3u) buf0 = buf1, buf1 = buf2, buf2 = b;
        else buf0 = buf2, buf2 = b;
    };
    const std::integral_constant<uint32_t, 0> first;    // of a group's steps
    const std::integral_constant<uint32_t, 1> second;
    const std::integral_constant<uint32_t, 2> only;     // of a group of two blocks
    LEV_WAIT_VMCNT(0);
    asm volatile("" : "+v"(own_pair), "+v"(own_max)::"memory");   // (not waited for in front of the requests)
    if (tid < 32u * T) {
        s_pair[tid] = own_pair;
        s_us[tid] = pf_row_scale(own_max).unscale;
    }
    lev_barrier_lds();
    if (!live) {
        auto pass = [&](uint32_t step, auto kind) {
            bring(step, kind);
#pragma unroll
            for (uint32_t i = 0; i < 8u * T; ++i) requests(step, kind, i / (4u * T), i % (4u * T));
            turn();
        };
        for (uint32_t step = 0; step + 1u < nsteps; step += 2u) pass(step, first), pass(step + 1u, second);
        if (nsteps & 1u) pass(nsteps - 1u, only);
        LEV_WAIT_VMCNT(0);
        return;
    }

    float y[T][16], whole[T][16];   // FOLD: the part under way, and the parts before it
#pragma unroll
    for (uint32_t t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) y[t][i] = whole[t][i] = 0.f;
    auto fold = [&]() {
#pragma unroll
        for (uint32_t t = 0; t < T; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                whole[t][i] += y[t][i];
                y[t][i] = 0.f;
            }
    };
    // Twelve waves have 168 registers each, which this and the lane's number made again at the end keep to: with five spilled, a
    // folded sum among them, the down product of 4096 / 1536 (500 tokens, top-6 of 64) took 149 us for 133.  Other forms have the masks
    // in vector registers (the down product of eight waves at 2304 / 1280 45.9 us, with scalar ones 46.7).
    const pf_consts<FOLD && OCC == 3u> kc;
    const uint8_t *const wmine = lds + L::kW + wave * L::kWArea + lr * kPfWRow;
    const uint32_t areg = (lr >> 3) * 1024u, apar = (lr >> 3) & 1u, acol = lr & 7u;
    uint32_t aoff[4];   // this lane's fragment of half s of block b of a step: aoff[2b + s], + 4096 per column tile, + kPlane for the low plane
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        const uint32_t run = 2u * k + g;
        aoff[k] = areg + ((run ^ apar) * 8u + (acol ^ run)) * 16u;
    }

    // Codes and scale of a block, 8 aligned bytes a read: at this row stride 4.2 clocks of the LDS, where one dword or half
    // word takes 8.1 and two dwords at once 16.  They are decoded behind the products of the block before.  Code bytes 8g .. 8g + 7 of a step's first block start two
    // bytes behind a dword boundary, those of its second on one.
    lev_u32x2 w[3];
    auto w_read = [&](const uint8_t *q, uint32_t st, uint32_t b, bool part) {
        auto at = [&](uint32_t byte) { return *reinterpret_cast<const lev_u32x2 *>(q + byte); };
        if (b == 0u) w[0] = at(32u * st + 8u * g), w[1] = at(32u * st + 8u * g + 8u), w[2] = at(32u * st);
        else if (st == 1u) w[0] = at(56u + 16u * g), w[2] = at(48u);   // (the last 8 bytes lie at 72)
        else if (part) w[0] = at(32u + 8u * g), w[2] = at(16u);
        else w[0] = at(16u + 8u * g), w[1] = at(24u + 8u * g), w[2] = at(16u);
    };
    uint32_t code[2];   // the next block's code dwords, its scale, its operands
    float dn;
    uint32_t bn[8];
    auto w_take = [&](uint32_t st, uint32_t b, bool part) {
        uint32_t dw;
        if (b == 0u) {
            code[0] = st ? __builtin_amdgcn_alignbit(w[1].x, w[0].y, 16) : __builtin_amdgcn_alignbit(w[0].y, w[0].x, 16);
            code[1] = st ? __builtin_amdgcn_alignbit(w[1].y, w[1].x, 16) : __builtin_amdgcn_alignbit(w[1].x, w[0].y, 16);
            dw = st ? w[2].y : w[2].x;
        } else {
            code[0] = st || part ? w[0].x : w[0].y;
            code[1] = st || part ? w[0].y : w[1].x;
            dw = (st ? w[2].y : w[2].x) >> 16;
        }
        dn = lev_f16_bits_to_f32(dw & 0xFFFFu);
        asm("" : "+v"(dn));   // converted once: the mixed-precision multiply-add takes longer than the f32 one
    };
    auto quarter = [&](uint32_t k) { pf_decode(k & 1u ? code[k >> 1] >> 8 : code[k >> 1], kc, bn[k], bn[4u + k]); };
    p_h8 A[4];   // high plane's halves of the block, low plane's
    auto a_read = [&](uint32_t buf, uint32_t u, uint32_t k) {
        A[k] = *reinterpret_cast<const p_h8 *>(lds + buf + aoff[2u * (u / T) + (k & 1u)] + (u % T) * 4096u + (k >> 1) * L::kPlane);
    };
    w_read(wmine, 0, 0, false);
    if (NBUF == 3u) {
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) a_read(0u, 0u, k);
    }
    w_take(0, 0, false);
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) quarter(k);

    // a unit's product is added behind the products of the next one (four waves a SIMD: at once, they have no registers for two)
    constexpr bool kLate = OCC < 4u;
    p_f16v pend = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float pend_d = 0.f;
    auto step_of = [&](uint32_t step, auto kind) {
        constexpr uint32_t st = decltype(kind)::value & 1u;
        constexpr bool part = decltype(kind)::value == 2u;
        bring(step, kind);
        if (NBUF == 2u) {
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) a_read(buf0, 0u, k);
        }
        const uint8_t *const wb = wmine + ((step >> 1) & 1u) * L::kWBuf, *const wnext = wmine + (((step + 1u) >> 1) & 1u) * L::kWBuf;
#pragma unroll
        for (uint32_t b = 0; b < 2u; ++b) {
            const float d = dn;
            const p_h8 B[2] = {__builtin_bit_cast(p_h8, lev_u32x4{bn[0], bn[1], bn[2], bn[3]}), __builtin_bit_cast(p_h8, lev_u32x4{bn[4], bn[5], bn[6], bn[7]})};
            if (b == 0u) {
                w_read(wb, st, 1u, part);
            } else {
                if (st == 1u) {
                    LEV_WAIT_VMCNT(kALoads);   // the next group's weights have landed
                    asm volatile("" ::: "memory");
                }
                w_read(wnext, st ^ 1u, 0u, false);
            }
#pragma unroll
            for (uint32_t t = 0; t < T; ++t) {   // unit: one block x one column tile
                const uint32_t u = b * T + t, pt = t ? t - 1u : T - 1u;
                p_f16v acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                if (t == T - 1u) w_take(b == 0u ? st : st ^ 1u, b ^ 1u, b == 0u && part);
#pragma unroll
                for (uint32_t k = 0; k < 4u; ++k) {
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[k], B[k & 1u], acc, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);   // (else it comes behind the additions, and they wait for the product before)
                    // the next unit's fragment takes the place of this one
                    if (u + 1u < 2u * T) a_read(buf0, u + 1u, k);
                    else if (NBUF == 3u) a_read(buf1, 0u, k);
                    // the product before this one, while the matrix cores have this one
#pragma unroll
                    for (uint32_t i = 4u * k; kLate && i < 4u * k + 4u; ++i) y[pt][i] = fmaf(pend_d, pend[i], y[pt][i]);
                    if (t == T - 1u) quarter(k);
                    requests(step, kind, b, 4u * t + k);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (kLate) {
                    pend = acc;
                    pend_d = d;
                    // the part before this step is whole only now, whatever T: the same bits wherever a pair lies in its item
                    if (FOLD && st == 0u && u == 0u && step != 0u && (step & (kPfFold - 1u)) == 0u) fold();
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) y[t][i] = fmaf(d, acc[i], y[t][i]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        turn();
    };
    for (uint32_t step = 0; step + 1u < nsteps; step += 2u) {
        step_of(step, first);
        step_of(step + 1u, second);
        if (FOLD && !kLate && (step & (kPfFold - 2u)) == kPfFold - 2u) fold();
    }
    if (nsteps & 1u) step_of(nsteps - 1u, only);
#pragma unroll
    for (int i = 0; kLate && i < 16; ++i) y[T - 1u][i] = fmaf(pend_d, pend[i], y[T - 1u][i]);
    if (FOLD) fold();
    float(&sum)[T][16] = FOLD ? whole : y;

    LEV_WAIT_VMCNT(0);   // the requests past the end land before the LDS is given back
    // lane (r, h), register i of a tile: weight row r, column 8 (i / 4) + 4 h + i % 4
    const uint32_t me = FOLD && OCC == 3u ? __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) : lane, r = me & 31u, h = me >> 5;
    const uint32_t row = row0 + (PAIRED ? r & 15u : r);
#pragma unroll
    for (uint32_t t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 16; i += PAIRED ? 2 : 1) {
            uint32_t col = 32u * t + 8u * (i / 4) + 4u * h + (i % 4);
            float v = sum[t][i];
            if (PAIRED) {
                // lanes 0..15 of a half hold gate rows, 16..31 the same up rows: two columns trade halves, so
                // that every lane has a gate and its up value, of column i in lanes 0..15, of i + 1 in 16..31
                const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(sum[t][i + 1]), false, false);
                col += r >> 4;
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
template <bool PAIRED, uint32_t WAVES, uint32_t TMAX, uint32_t OCC, uint32_t NBUF, bool FOLD>
__global__ void __launch_bounds__(WAVES * 64, OCC)
moe_pf_kernel(lev_moe_grouped_args a, uint32_t row_tiles, const _Float16 *__restrict__ ph,
              const _Float16 *__restrict__ pl, const uint32_t *__restrict__ pmax, const int32_t *__restrict__ glist,
              const lev_pf_item *__restrict__ items, const uint32_t *__restrict__ nitems, float *__restrict__ out) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    __shared__ int32_t s_pair[32u * TMAX];
    __shared__ float s_us[32u * TMAX];
    const uint32_t j = blockIdx.x >> 3, at = (j / row_tiles) * 8u + (blockIdx.x & 7u), rt = j % row_tiles;
    const lev_pf_item it = items[at];   // (there is room for the whole grid's)
    if (at >= *nitems) return;
    if constexpr (TMAX >= 2u)
        if (it.count > 32) return pf_tile<PAIRED, WAVES, TMAX, OCC, NBUF, FOLD, 2>(a, it, rt, ph, pl, pmax, glist, out, smem, s_pair, s_us);
    pf_tile<PAIRED, WAVES, TMAX, OCC, NBUF, FOLD, 1>(a, it, rt, ph, pl, pmax, glist, out, smem, s_pair, s_us);
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct pf_layout {
    size_t glist, valid, items, nitems, xh, xl, xmax, ah, al, amax, dn, total;
};
size_t pf_max_items(const lev_moe_grouped_args &a, uint32_t cols) {
    const size_t pairs = (size_t)a.tokens * a.top_k;
    return (pairs / cols + (a.experts < pairs ? a.experts : pairs) + 7u) & ~(size_t)7;   // whole turns of the XCDs
}
pf_layout pf_layout_of(const lev_moe_grouped_args &a) {
    const size_t pairs = (size_t)a.tokens * a.top_k;
    pf_layout L;
    size_t o = 0;
    L.glist = o; o += align256(pairs * 4);
    L.valid = o; o += align256(pairs);
    L.items = o; o += align256(pf_max_items(a, 32u) * sizeof(lev_pf_item));
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

template <bool PAIRED, uint32_t WAVES, uint32_t TMAX, uint32_t OCC, uint32_t NBUF, bool FOLD>
hipError_t pf_launch_as(lev_ctx *ctx, const lev_moe_grouped_args &a, uint32_t cols, const _Float16 *ph, const _Float16 *pl, const uint32_t *pmax,
                        const int32_t *glist, const lev_pf_item *items, const uint32_t *nitems, float *out) {
    constexpr size_t lds = pf_lds_map<WAVES, TMAX, NBUF>::kBytes;
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&moe_pf_kernel<PAIRED, WAVES, TMAX, OCC, NBUF, FOLD>), lds);
        e != hipSuccess)
        return e;
    const uint32_t slots = (uint32_t)pf_max_items(a, cols);
    const uint32_t rows = PAIRED ? a.inter : a.hidden, per_wg = WAVES * (PAIRED ? 16u : 32u), tiles = (rows + per_wg - 1u) / per_wg;
    hipLaunchKernelGGL((moe_pf_kernel<PAIRED, WAVES, TMAX, OCC, NBUF, FOLD>), dim3(slots * tiles), dim3(WAVES * 64u), lds,
                       ctx->stream, a, tiles, ph, pl, pmax, glist, items, nitems, out);
    return hipGetLastError();
}

template <bool PAIRED>
hipError_t pf_launch(lev_ctx *ctx, const lev_moe_grouped_args &a, const pf_plan &plan, const _Float16 *ph, const _Float16 *pl,
                     const uint32_t *pmax, const int32_t *glist, const lev_pf_item *items, const uint32_t *nitems, float *out) {
    switch (PAIRED ? plan.gate_up : plan.down) {
        case kChain: return pf_launch_as<PAIRED, 8, 2, 4, 2, false>(ctx, a, plan.cols, ph, pl, pmax, glist, items, nitems, out);
        case kTwelve: return pf_launch_as<PAIRED, 12, 2, 3, 3, true>(ctx, a, plan.cols, ph, pl, pmax, glist, items, nitems, out);
        case kEight: return pf_launch_as<PAIRED, 8, 2, 2, 3, true>(ctx, a, plan.cols, ph, pl, pmax, glist, items, nitems, out);
        case kFour: return pf_launch_as<PAIRED, 4, 2, 2, 3, true>(ctx, a, plan.cols, ph, pl, pmax, glist, items, nitems, out);
        default: return pf_launch_as<PAIRED, 8, 1, 4, 3, true>(ctx, a, plan.cols, ph, pl, pmax, glist, items, nitems, out);
    }
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
    const pf_plan plan = pf_plan_of(pf_shape{(uint32_t)ctx->num_cus, a.hidden, a.inter, a.experts, a.top_k, a.tokens});
    hipError_t e;
    const size_t lds = (size_t)2 * a.experts * 4 + 4 + (pf_list_in_lds(pairs) ? (size_t)pairs * 4 : 0);
    if ((e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&moe_pf_group_kernel), lds)) != hipSuccess) return e;
    hipLaunchKernelGGL(moe_pf_group_kernel, dim3(1u + (a.tokens + 15u) / 16u), dim3(1024), lds,
                       ctx->stream, ids, pairs, a.experts, a.top_k, glist, valid, reinterpret_cast<int32_t *>(dn), items, nitems, ctx->d_flag, x,
                       a.tokens, a.hidden, xh, xl, xmax, plan.cols);   // (the ranks are in the place of dn, which comes much later)
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = pf_launch<true>(ctx, a, plan, xh, xl, xmax, glist, items, nitems, act)) != hipSuccess) return e;
    // rows of act that belong to dropped pairs were never written: their planes are never read
    hipLaunchKernelGGL(moe_pf_planes_kernel, dim3((pairs + 3u) / 4u), dim3(256), 0, ctx->stream, act, pairs, a.inter, ah,
                       al, amax);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = pf_launch<false>(ctx, a, plan, ah, al, amax, glist, items, nitems, dn)) != hipSuccess) return e;
    return lev_moe_merge_launch(ctx, a, dn, weights, valid, y);
}
