// Q4_K and Q6_K prefill GEMM for short prompts and for matrices whose 256-token tiles leave the chip
// idle:  Y[t][r] = sum_k X[t][k] W[r][k], W rounded to fp16 as the other prefill GEMMs do
// (lev-forge/src/coopmat.rs:236-425), f32 accumulation.
//
// A wave owns 32 rows x 32 to 128 tokens of a slice of K.  It decodes its rows' weights straight into
// its own fp16 B fragments (lane = row l%32, half l/32; nothing of W goes through LDS) and multiplies
// each with T token tiles.  RW waves of a workgroup own different rows of one K slice and share its X
// steps (64 values of every token, direct global -> LDS loads, four buffers); KW groups of them take
// different slices (eight waves: four rows of tiles in two slices, or two in four), and S workgroups more: the partial
// tiles of a workgroup meet in LDS, those of
// the S workgroups in scratch, and a small kernel adds them in slice order.
//
// 4096 rows are 128 row tiles: one wave each would leave seven eighths of the chip idle, so K is cut until the
// CUs have work (lev_gemm_split_choose).  A wave that takes all of K adds the same products in the same
// order as the 256-token kernels: bit for bit their results.
//
// What bounds it: a step of a wave is some 80 (Q4_K) or 105 (Q6_K) vector instructions of decode and 4 T MFMAs, two waves a
// SIMD; and around the steps 2 to 5 us until the first weights are there, 1.5 for adding up the slices and storing, 5 for
// the kernel that adds the workgroups' (in-kernel time stamps).  With the products of a step right behind its barrier all
// waves waited for their first LDS reads together: 24 cases drawn over 1000 to 20000 rows and 19 to 740 tokens take 0.92 of
// that, 2048 columns x 3000 rows of Q4_K at 700 tokens 21.2 us and 18.2.
// 77 tokens, 4096 rows, 12288 columns of Q6_K: 23.8 us (24.4 with the sums of a row tile by one wave;
// 218 in 256-token tiles on 32 CUs); 123 tokens, 1617 rows, 4096 columns of Q4_K: 11.2 us (11.9; 17 in tiles of 128 tokens alone).
#include "prefill_decode.hpp"

#include <cmath>

namespace {

constexpr uint32_t kTile = 4096u;        // X step of 32 tokens: 32 rows of 128 bytes
// X steps in LDS: the one in use and three on their way, or one where 160 KB (for KW = 1, of which two workgroups share a
// CU, 80 KB) hold no more or more is no faster (32000 x 4096 of Q6_K at 90 tokens 51 us with one on its way, 47 with three)
template <typename W>
constexpr uint32_t x_bufs(int t, int rw, int kw) {
    return t >= (kw == 1 ? 4 : 3) || kw * (4u * t * kTile + rw * W::kArea) > 160u * 1024u ? 2u : 4u;
}

// grid: row tiles * token tiles * (zn slices from z0 on, of the `splits`) workgroups in one line, up to a multiple of
// eight.  All slices of a launch write partial tiles of their own to `out`, one behind the other; add: the one slice
// of the launch is added to what is there.  Workgroups go to the XCDs in
// turn: each takes an eighth of the tiles, whose order has the token tiles of a row tile together (they read the same
// weights).
template <typename W, int T, int RW, int KW>
__global__ void __launch_bounds__(RW *KW * 64, 2)
gemm_split_kernel(const uint8_t *__restrict__ w, const uint16_t *__restrict__ x, float *__restrict__ out, uint32_t in_dim,
                  uint32_t rows, uint32_t tokens, uint32_t row_tiles, uint32_t tok_tiles, uint32_t splits, uint32_t z0,
                  uint32_t zn, uint32_t add) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t lr = lane & 31u, lh = lane >> 5, rw = wave % RW, kw = wave / RW;
    const uint32_t tile = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3), zr = tile / tok_tiles;
    const uint32_t zl = zr / row_tiles, z = z0 + zl, rt = zr - zl * row_tiles, tok0 = (tile - zr * tok_tiles) * (32u * T);
    if (zl >= zn) return;
    const uint32_t row0 = (rt * RW + rw) * 32u, row = row0 + lr;
    const uint32_t nsb = in_dim >> 8, ns = KW * splits;
    const uint32_t sb0 = (z * KW + kw) * nsb / ns, sb1 = (z * KW + kw + 1u) * nsb / ns;
    uint32_t most = 0u;   // superblocks of the workgroup's longest slice: every wave meets that many barriers
#pragma unroll
    for (uint32_t k = 0; k < KW; ++k) {
        const uint32_t n = (z * KW + k + 1u) * nsb / ns - (z * KW + k) * nsb / ns;
        most = n > most ? n : most;
    }
    // X: load j brings the 128 bytes of eight tokens; 16-byte unit c of token t lies at c ^ (t / 2 & 7): the LDS serves sixteen
    // lanes of a fragment's read at once, 256 bytes, from sixteen different places (at c ^ (t & 7) tokens t and t + 8 met, and
    // a read took 8 clocks for 4: 390 of the 2500 of a step of T = 3)
    constexpr uint32_t kBufs = x_bufs<W>(T, RW, KW);
    constexpr int kXLoads = 4 * T / RW;
    const uint8_t *xsrc[kXLoads];
#pragma unroll
    for (int j = 0; j < kXLoads; ++j) {
        const uint32_t tl = 8u * (rw + RW * j) + (lane >> 3), t = tok0 + tl < tokens ? tok0 + tl : tokens - 1u;
        xsrc[j] = reinterpret_cast<const uint8_t *>(x) + ((uint64_t)t * in_dim * 2u + 16u * ((lane & 7u) ^ (tl >> 1 & 7u)));
    }
    const uint32_t xlds = lev_lds_offset(lds) + kw * (kBufs * T * kTile) + rw * 1024u, steps = (sb1 - sb0) * 4u;
    auto x_request = [&](uint32_t step, int from, int to) {   // loads from .. to - 1 of a step
        const uint32_t s = sb0 * 4u + (step < steps ? step : steps - 1u);   // past the end: any valid step, never read
#pragma unroll
        for (int j = from; j < to; ++j) lev_load_lds16(xsrc[j] + (uint64_t)s * 128u, xlds + (step % kBufs) * (T * kTile) + j * (RW * 1024u));
    };
    const uint8_t *const xmine = lds + kw * (kBufs * T * kTile) + lr * 128u;

#pragma unroll
    for (uint32_t s = 0; s + 1u < kBufs; ++s) x_request(s, 0, kXLoads);
    W wt;
    wt.init(w, row0, rows, nsb, lds + KW * (kBufs * T * kTile) + wave * W::kArea);
    wt.request(sb0);
    f32x16 acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;

    // The products run two groups (of the four of a step) behind the barriers: groups 2 and 3 of a step are multiplied
    // behind the next barrier, from fragments read in front of it, while the first fragments of the new step come in.
    // Otherwise all waves wait for their LDS reads at the same time, behind every barrier.  The first step's are zeros.
    const uint32_t mine = sb1 - sb0;
    f16x8 a[4][T], b;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        b[i] = (_Float16)0.f;
#pragma unroll
        for (int t = 0; t < T; ++t) a[2][t][i] = a[3][t][i] = (_Float16)0.f;
    }
    wt.clear();
    // products of a group and behind them, while they run, the X fragments of the group `read` (-1: none) and `next`,
    // which makes the following B: one MFMA, then what can issue while it runs (a wave issues in order, and a second
    // MFMA behind the first would hold it for 32 clocks)
    auto phase = [&](const uint8_t *xb, int q, int read, auto next) {
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[q][t], b, acc[t], 0, 0, 0);
        if (read >= 0) {
#pragma unroll
            for (int t = 0; t < T; ++t)
                a[read][t] = *reinterpret_cast<const f16x8 *>(xb + t * kTile + 16u * (wt.unit(read) ^ (lr >> 1 & 7u)));
        }
        next();
#pragma unroll
        for (int t = 0; t < T; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                    // MFMA
            if (read >= 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     // LDS read
            __builtin_amdgcn_sched_group_barrier(0x002, (28 + T - 1) / T, 0);     // VALU
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (uint32_t i = 0; i < mine; ++i) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t step = i * 4u + c;
            // This step's X has landed: newer are the X of the steps behind it and, behind a superblock's
            // first step, the next superblock's weights, which are wanted by the one after its fourth.
            static_assert(kBufs == 4u || kBufs == 2u, "the counts below");
            if (c == 1 || (c >= 2 && kBufs == 4u)) LEV_WAIT_VMCNT((kBufs - 2u) * kXLoads + W::kLoads);
            else LEV_WAIT_VMCNT((kBufs - 2u) * kXLoads);
            if (c == 0) wt.touch();   // the compiler's own wait for them goes here, behind ours for the X requested after them
            __builtin_amdgcn_sched_barrier(0);
            lev_barrier_lds();          // everybody's has, and everybody is done with the other buffer
            // Together, by all waves, right behind the barrier they wait in the issue for 400 to 800 clocks of a step's 3000. So
            // they go out behind the step's products (in front of the weights' request) where the data is not wanted for another two
            // steps and products are few (64 tokens x 12288 x 4096 of Q4_K 16.1 -> 15.4 us); else the data comes too
            // late for that (500 x 2500 x 5120 of Q4_K 24.4 -> 25.8, 350 x 9000 x 1280 of Q6_K 17.4 -> 18.0).
            constexpr bool kLater = kBufs == 4u && T <= 2;
            constexpr int kHalf = (kXLoads + 1) / 2, kOf4[5] = {0, (kXLoads + 3) / 4, kHalf, kHalf + (kXLoads - kHalf + 1) / 2, kXLoads};
            auto x_part = [&](int p) {
                if (!kLater) return;
                if (c != 0) x_request(step + kBufs - 1u, kOf4[p], kOf4[p + 1]);
                else if (p < 2) x_request(step + kBufs - 1u, p ? kHalf : 0, p ? kXLoads : kHalf);
                __builtin_amdgcn_sched_barrier(0);
            };
            if (!kLater) {
                x_request(step + kBufs - 1u, 0, kXLoads);
                __builtin_amdgcn_sched_barrier(0);
            }
            const uint8_t *const xb = xmine + (step % kBufs) * (T * kTile);
#pragma unroll
            for (int t = 0; t < T; ++t) a[0][t] = *reinterpret_cast<const f16x8 *>(xb + t * kTile + 16u * (wt.unit(0) ^ (lr >> 1 & 7u)));
            phase(xb, 2, -1, [&] { b = wt.frag((c + 3) & 3, 3); });
            x_part(0);
            phase(xb, 3, 1, [&] {
                // (Q4_K: a column's factors all at once.  Those of its second half in front of that: 6144 x 6144 at 260 tokens 39.0
                // us for 38.0, 4096 x 4096 at 200 17.1 for 16.8, 1536 x 16000 at 700 46.8 for 46.5.)
                if (c == 0) wt.take();
                if (c == (W::kQ6 ? 2 : 0)) wt.half(1);
                b = wt.frag(c, 0);
            });
            x_part(1);
            if (c == 0) {
                const uint32_t sb = sb0 + i + 1u;
                wt.request(sb < sb1 ? sb : sb1 - 1u);
                __builtin_amdgcn_sched_barrier(0);
            }
            phase(xb, 0, 2, [&] { b = wt.frag(c, 1); });
            x_part(2);
            phase(xb, 1, 3, [&] { b = wt.frag(c, 2); });
            x_part(3);
        }
    }
    phase(xmine, 2, -1, [&] { b = wt.frag(3, 3); });
    phase(xmine, 3, -1, [] {});
    // (the waves of a shorter slice: one superblock less)
    for (uint32_t i = 4u * mine; i < 4u * most; ++i) asm volatile("s_barrier" ::: "memory");
    LEV_WAIT_VMCNT(0);   // the request past the end lands before the LDS is used again

    // a tile's 32 tokens from `first` on; past the tokens' end and for rows past the last one nothing is stored
    float *const dst = out + (uint64_t)zl * tokens * rows;
    const uint32_t at = row < rows ? (4u * lh * rows + row) * 4u : lev_buffer::kNothing;
    auto store = [&](int t, int i, float v) {
        const uint32_t first = tok0 + 32u * t, here = first < tokens ? (tokens - first < 32u ? tokens - first : 32u) : 0u;
        const lev_buffer tile_out(dst + (uint64_t)(here ? first : 0u) * rows, here * rows * 4u);
        const uint32_t tok = (uint32_t)(8 * (i / 4) + (i % 4)) * rows * 4u;
        if (add) v += __uint_as_float(tile_out.load4(at, 0, tok));
        tile_out.store4(__float_as_uint(v), at, 0, tok);
    };
    // A wave adds up and stores one KW-th of its rows' outputs, registers i of part i / (16 / KW): it leaves the others'
    // parts in LDS and adds theirs to its own in slice order.  (By the waves of the first slice alone: 9 of 50 thousand
    // clocks at 77 tokens x 4096 x 12288.)
    constexpr int kPart = 16 / KW;
    float *const red = reinterpret_cast<float *>(lds);
    auto left = [&](uint32_t part, uint32_t from, int t, int i) -> float & {   // what slice `from` leaves for the wave of `part`
        return red[(((part * (KW - 1u) + (from < part ? from : from - 1u)) * RW + rw) * (T * kPart) + t * kPart + i % kPart) * 64 + lane];
    };
    if (KW > 1) {
        lev_barrier_lds();
#pragma unroll
        for (uint32_t p = 0; p < KW; ++p) {
            if (p == kw) continue;
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = p * kPart; i < (int)(p + 1u) * kPart; ++i) left(p, kw, t, i) = acc[t][i];
        }
        lev_barrier_lds();
    }
#pragma unroll
    for (uint32_t p = 0; p < KW; ++p) {
        if (p != kw) continue;
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int i = p * kPart; i < (int)(p + 1u) * kPart; ++i) {
                float v = p == 0u ? acc[t][i] : left(p, 0u, t, i);
#pragma unroll
                for (uint32_t k = 1; k < KW; ++k) v += k == p ? acc[t][i] : left(p, k, t, i);
                store(t, i, v);
            }
    }
}

// y[i] = sum over the splits, in order
template <int V>
__global__ void __launch_bounds__(256)
gemm_split_sum_kernel(const float *__restrict__ part, float *__restrict__ y, uint64_t n, uint32_t splits) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x, nv = n / V;
    if (i >= nv) return;
    const vec *p = reinterpret_cast<const vec *>(part);
    vec s = p[i];
    for (uint32_t k = 1; k < splits; ++k) s += p[(uint64_t)k * nv + i];
    reinterpret_cast<vec *>(y)[i] = s;
}

template <typename W, int T, int RW, int KW>
hipError_t launch_as(lev_ctx *ctx, const uint8_t *w, const uint16_t *x, float *out, uint32_t in_dim, uint32_t rows,
                     uint32_t tokens, uint32_t tok_tiles, uint32_t splits, uint32_t z0, uint32_t zn, bool add) {
    constexpr size_t lds = (size_t)KW * x_bufs<W>(T, RW, KW) * T * kTile + RW * KW * W::kArea;
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&gemm_split_kernel<W, T, RW, KW>), lds); e != hipSuccess) return e;
    const uint32_t row_tiles = (rows + RW * 32u - 1u) / (RW * 32u);
    hipLaunchKernelGGL((gemm_split_kernel<W, T, RW, KW>), dim3((row_tiles * tok_tiles * zn + 7u) / 8u * 8u), dim3(RW * KW * 64),
                       lds, ctx->stream, w, x, out, in_dim, rows, tokens, row_tiles, tok_tiles, splits, z0, zn, add ? 1u : 0u);
    return hipGetLastError();
}

template <typename W, int T>
hipError_t launch_tiles(lev_ctx *ctx, const uint8_t *w, const uint16_t *x, float *y, uint32_t in_dim, uint32_t rows,
                        uint32_t tokens, uint32_t tok_tiles, const lev_gemm_split_plan &plan) {
    if (plan.kw == 1u) return launch_as<W, T, 4, 1>(ctx, w, x, y, in_dim, rows, tokens, tok_tiles, 1u, 0u, 1u, false);
    const uint32_t splits = plan.splits;
    auto slices = [&](float *out, uint32_t z0, uint32_t zn, bool add) {
        if constexpr (4u * (x_bufs<W>(T, 2, 4) * T * kTile + 2u * W::kArea) <= 160u * 1024u)
            if (plan.kw == 4u) return launch_as<W, T, 2, 4>(ctx, w, x, out, in_dim, rows, tokens, tok_tiles, splits, z0, zn, add);
        return launch_as<W, T, 4, 2>(ctx, w, x, out, in_dim, rows, tokens, tok_tiles, splits, z0, zn, add);
    };
    if (splits == 1u) return slices(y, 0u, 1u, false);
    float *const part = static_cast<float *>(lev_scratch(ctx, (size_t)splits * tokens * rows * 4));
    if (!part) {
        // no memory, or a program is being recorded and the scratch is still too small: a launch for every slice, each added to y where
        // the others are, in the same order and so to the same bits
        for (uint32_t z = 0; z < splits; ++z)
            if (hipError_t e = slices(y, z, 1u, z != 0u); e != hipSuccess) return e;
        return hipSuccess;
    }
    if (hipError_t e = slices(part, 0u, splits, false); e != hipSuccess) return e;
    const uint64_t n = (uint64_t)tokens * rows;
    if (n % 4u == 0u && (reinterpret_cast<uintptr_t>(y) & 15u) == 0u)
        hipLaunchKernelGGL((gemm_split_sum_kernel<4>), dim3((uint32_t)((n / 4u + 255u) / 256u)), dim3(256), 0, ctx->stream,
                           part, y, n, splits);
    else
        hipLaunchKernelGGL((gemm_split_sum_kernel<1>), dim3((uint32_t)((n + 255u) / 256u)), dim3(256), 0, ctx->stream, part,
                           y, n, splits);
    return hipGetLastError();
}

template <typename W>
hipError_t launch(lev_ctx *ctx, const uint8_t *w, const uint16_t *x, float *y, uint32_t in_dim, uint32_t rows,
                  uint32_t tokens, const lev_gemm_split_plan &plan) {
    const uint32_t n = (tokens + 32u * plan.t - 1u) / (32u * plan.t);
    switch (plan.t) {
    case 1u: return launch_tiles<W, 1>(ctx, w, x, y, in_dim, rows, tokens, n, plan);
    case 2u: return launch_tiles<W, 2>(ctx, w, x, y, in_dim, rows, tokens, n, plan);
    case 3u: return launch_tiles<W, 3>(ctx, w, x, y, in_dim, rows, tokens, n, plan);
    default: return launch_tiles<W, 4>(ctx, w, x, y, in_dim, rows, tokens, n, plan);
    }
}

}  // namespace

// Which of the GEMMs takes a shape, in how many K slices and token tiles of which height: the least of what each would
// take, from times measured on every plan of 450 shapes a format drawn over 1000 to 32000 rows, 1024 to 12288 columns and
// 17 to 1024 tokens (us; a step is 64 values of K, t = 32-token tiles a wave; the choice is within 1.0 % of the best on
// average, 7 % in nineteen of twenty, and 0.7 % on 120 others a format).
//   256-token tiles:  a round of workgroups (one per CU), more as it fills the CUs, and X put into order in front;
//   KW = 1:           a round of up to two workgroups a CU; their steps take 1.8 times those of one alone, a tenth of the
//                     difference less where hardly any CU has two (3072 x 16536 of Q6_K at 330 tokens 57.7 us, with KW = 2 61.6);
//   KW = 2, KW = 4:   a round of one a CU, and with S > 1 splits the kernel that adds and its reads and writes; of estimates
//                     that are alike KW = 4 in splits is the better one in 56 of 71 shapes, by 3 %: 0.95 of its own.
// Lower token tiles are more workgroups that decode the same weights: what fills the chip where rows alone do not.
// Beyond 1024 tokens the times of these outgrow the estimates, by 1.1 in the middle and up to 1.4, those of the 256-token
// tiles hardly do: 1.15 is allowed for that (120 shapes a format of up to 8192 tokens).
// Tall matrices (768 row tiles and more) and rows of fewer than six superblocks are never cut along K, so that
// there every kernel adds in the same order.
lev_gemm_split_plan lev_gemm_split_choose(const lev_ctx *ctx, bool q6, uint32_t in_dim, uint32_t rows, uint32_t tokens) {
    const double cus = ctx->num_cus, long_prompt = tokens > 1024u ? 1.15 : 1.0;
    const uint32_t nsb = in_dim / 256u, tiles = (tokens + 31u) / 32u;
    lev_gemm_split_plan best{};
    double least = 1e300;
    auto offer = [&](double us, uint32_t kw, uint32_t splits, uint32_t t) {
        if (us < least) {
            least = us;
            best = lev_gemm_split_plan{kw, splits, t};
        }
    };
    struct wide_cost { double start, k, fill, once, order; };
    const wide_cost w3 = q6 ? wide_cost{5.3, 7.9, 4.25, 4.4, 1.15} : wide_cost{6.2, 5.15, 5.45, 3.75, 1.8};
    const wide_cost w4 = q6 ? wide_cost{6.9, 8.1, 7.0, 4.3, 1.05} : wide_cost{7.7, 6.1, 7.4, 3.0, 1.35};
    for (uint32_t rt = 3; rt <= 4u; ++rt) {
        const wide_cost &k = rt == 3u ? w3 : w4;
        const double n = (double)((rows + 32u * rt - 1u) / (32u * rt)) * ((tokens + 255u) / 256u), rounds = std::ceil(n / cus);
        offer(rounds * (k.start + in_dim / 1024.0 * (k.k + k.fill * n / (rounds * cus))) + k.once + k.order * 1e-6 * tokens * in_dim, 0u, rt, 0u);
    }
    struct cost { double start, step, per_tile, full, once, sum, sum_mb; };
    const cost k1 = q6 ? cost{0.66, 0.33, 0.089, 0.72, 2.9, 0, 0} : cost{0.0, 0.205, 0.085, 0.78, 3.0, 0, 0};
    const cost k2 = q6 ? cost{2.1, 0.457, 0.111, 0.27, 3.2, 1.6, 1.08} : cost{0.17, 0.224, 0.125, 0.42, 4.4, 2.1, 1.14};
    const cost k4 = q6 ? cost{2.56, 0.42, 0.165, 0.31, 2.06, 2.26, 0.93} : cost{0.83, 0.198, 0.193, 0.39, 3.6, 2.07, 1.47};
    for (uint32_t t = 1; t <= 4u && t <= tiles; ++t) {
        const double tok_tiles = (tiles + t - 1u) / t;
        // workgroups, whole eighths of them on an XCD each
        auto wgs_of = [&](uint32_t rows_wg, uint32_t splits) { return 8.0 * std::ceil((rows + rows_wg - 1u) / rows_wg * tok_tiles * splits / 8.0); };
        {
            const double n = wgs_of(128u, 1u), whole = std::floor(n / (2.0 * cus)), rest = n - whole * 2.0 * cus;
            const double rounds = whole + (rest > 0.0 ? 1.0 : 0.0), pairs = whole + (rest > cus ? 0.9 + 0.1 * (rest - cus) / cus : 0.0);
            offer(long_prompt * (rounds * k1.start + 4.0 * nsb * (k1.step + k1.per_tile * t) * (rounds + k1.full * pairs) + k1.once), 1u, 1u, t);
        }
        if ((rows + 31u) / 32u >= 768u || nsb < 6u) continue;
        for (uint32_t kw = 2; kw <= 4u; kw += 2u) {
            if (kw == 4u && q6 && t == 4u) continue;   // (more LDS than there is)
            const cost &k = kw == 2u ? k2 : k4;
            for (uint32_t s = 1; s <= 8u && s * kw <= nsb; ++s) {
                const double n = wgs_of(kw == 2u ? 128u : 64u, s), rounds = std::ceil(n / cus), full = n / (rounds * cus);
                const double steps = 4.0 * ((nsb + kw * s - 1u) / (kw * s));
                offer((kw == 4u && s > 1u ? 0.95 : 1.0) * long_prompt * (rounds * (k.start + steps * (k.step + k.per_tile * t) * (1.0 + k.full * full)) + k.once +
                                     (s > 1u ? k.sum + k.sum_mb * 1e-6 * (s + 1.0) * tokens * rows : 0.0)), kw, s, t);
            }
        }
    }
    return best;
}

hipError_t lev_gemm_split_launch(lev_ctx *ctx, bool q6, const uint8_t *w, const uint16_t *x, float *y, uint32_t in_dim,
                                 uint32_t rows, uint32_t tokens, const lev_gemm_split_plan &plan) {
    // every slice has a superblock at least: a wave without one would step below its first
    if (plan.kw == 0u || plan.splits == 0u || plan.kw * plan.splits > in_dim / 256u) return hipErrorInvalidValue;
    return q6 ? launch<weights_q6k>(ctx, w, x, y, in_dim, rows, tokens, plan)
              : launch<weights_q4k>(ctx, w, x, y, in_dim, rows, tokens, plan);
}
