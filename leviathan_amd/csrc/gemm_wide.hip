// Q4_K and Q6_K prefill GEMM for prompts whose 256-token tiles fill the chip:  Y[t][r] = sum_k X[t][k] W[r][k].
//
// Stands in for the cooperative-matrix "gemm blocked" kernels (lev-forge/src/coopmat.rs:236-425; caller
// lev-model/src/gpu.rs:345-355; gate lev-cli/src/main.rs:1187-1279).  As there, W is dequantised to fp16 (f32 arithmetic,
// then round-to-nearest-even) and X arrives as fp16; products accumulate in f32.  Both operands use the same 16-bit type
// because one MFMA takes one input type; fp16 keeps X exactly as given.
//
// A workgroup owns 256 tokens x 32 RT rows (RT = 3 or 4), one workgroup a CU, eight waves, two a SIMD:
//   * waves 0..3 multiply: 64 tokens x all rows each, 2 RT tiles of v_mfma_f32_32x32x16_f16, K step 64.  Their tokens are
//     nobody else's, so X never goes through LDS: a small kernel in front puts X into the order in which the lanes of a
//     fragment take it (1 KB of consecutive bytes a fragment), and a wave requests a fragment four or eight products ahead
//     of its use, straight into registers;
//   * waves 4..7 decode, one 32-row tile each (RT = 3: three of them): every weight is decoded once a workgroup, a span of two
//     steps (half a superblock) ahead, and handed over as B fragments in two LDS buffers of 8 RT KB, one barrier a span.
// The multiplying waves run two groups of products behind the barriers: the last two groups of a span are multiplied behind the
// next barrier, from fragments read in front of it, while the first fragments of the new span come in.
//
// Why this split.  A lone wave of a SIMD issues a vector instruction every six clocks, two waves one every three to five,
// and an MFMA leaves the vector pipe half of its 32 clocks, so decode and products on different waves of a SIMD cover each
// other.  What the LDS has to carry bounds the tile: with X in LDS as well it was
// 124 KB a step of 96 x 256 x 64, 990 clocks beside 770 of MFMAs; 60 KB here.  A span is two steps because a superblock's
// steps take the decoding waves unequal times (new weights and factors, then none): at a barrier a step both sides waited
// for 350 to 520 of a step's 1260 clocks.  And the compiler must not move a superblock's requests and factors in among
// its fragments: with the order kept a step takes 980 clocks where it took 1260.
// 512 tokens, 4096 columns, us under a sustained load: 12288 rows of Q4_K 57.2 before and 55.0, of Q6_K 61.2 and 58.4, 32000 rows of
// Q6_K 139 and 131; 9456 x 9472 of Q4_K 100.6 and 96.2.  Of the 22 % fewer clocks a step the first of these keeps 4: the
// clock under these products falls with them, from 1.73 to 1.5 GHz (a loop of MFMAs alone on random operands runs at 1.45 and
// takes 35 us for it; the library's fp16 product 51).
// What bounds it (time stamps; 256 workgroups, one round of 45 to 50 us, 71 to 76 thousand clocks of Q4_K at 1.55 GHz): the 64 steps, 1000
// clocks each for 770 of MFMAs, nine tenths of it; the first span is there after 4.0 to 4.8 thousand clocks (2.0 to 3.3 thousand until the first
// weights, one to decode them), the stores take 2.3 to 6.5 thousand, and nothing covers either.  Q6_K: 83 thousand clocks, steps
// of 1160, which wait for the decoding waves, the first span after 5.2 thousand.
//
// K order inside a 64-step is permuted consistently on both operands (unit_of of the formats' weights); the sums are formed
// in the order in which a wave of gemm_split.hip that takes all of K forms them: the same bits.
#include "prefill_decode.hpp"

namespace {

constexpr uint32_t kWideThreads = 512;      // four waves that multiply, four that decode
constexpr uint32_t kFrag = 1024u;           // a fragment: 16 bytes a lane
constexpr int kTM = 2;                      // 32-token tiles a wave

// X as fragments: [32-token tile][chunk of 64][group q][lane][16 bytes].  A wave a chunk of a tile; tokens past the end
// repeat the last.  512 x 4096: 2.6 us.
template <typename W>
__global__ void __launch_bounds__(256)
gemm_x_fragments(const uint16_t *__restrict__ x, lev_u32x4 *__restrict__ out, uint32_t in_dim, uint32_t tokens) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, lr = lane & 31u;
    const uint32_t chunk = blockIdx.x * 4u + wave, t = blockIdx.y * 32u + lr, nchunk = in_dim >> 6;
    if (chunk >= nchunk) return;
    const lev_u32x4 *src = reinterpret_cast<const lev_u32x4 *>(x + (uint64_t)(t < tokens ? t : tokens - 1u) * in_dim + 64u * chunk);
    lev_u32x4 v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = src[W::unit_of(lane >> 5, q)];
    lev_u32x4 *dst = out + ((uint64_t)blockIdx.y * nchunk + chunk) * 256u + lane;
#pragma unroll
    for (int q = 0; q < 4; ++q) dst[64 * q] = v[q];
}

// grid: row tiles * token tiles in one line, up to a multiple of eight; the workgroups of an XCD take an eighth of the tiles,
// in whose order the token tiles of a row tile are together (they read the same weights).
// LDS: two buffers of B fragments [group][row tile], and what the format's weights take a decoding wave.
template <typename W, int RT>
__global__ void __launch_bounds__(kWideThreads, 2)
gemm_wide_kernel(const uint8_t *__restrict__ w, const uint8_t *__restrict__ xf, float *__restrict__ y, uint32_t in_dim,
                 uint32_t rows, uint32_t tokens, uint32_t row_tiles, uint32_t tok_tiles) {
    constexpr int RING = RT == 4 ? 4 : 8;      // groups of X requested ahead, as many as the registers hold
    constexpr uint32_t kBuf = RT * 8u * kFrag;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lr = lane & 31u, lh = lane >> 5;
    const uint32_t tile = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3), rt = tile / tok_tiles;
    if (rt >= row_tiles) return;
    const uint32_t row0 = rt * (32u * RT), tt0 = (tile - rt * tok_tiles) * (4u * kTM);
    const uint32_t nsb = in_dim >> 8, nspans = nsb * 2u;
    if (wave >= 4u) {
        const uint32_t f = wave - 4u;
        if (f >= (uint32_t)RT) {
            for (uint32_t k = 0; k < nspans; ++k) asm volatile("s_barrier" ::: "memory");   // nothing to decode
            return;
        }
        W wt;
        wt.init(w, row0 + 32u * f, rows, nsb, lds + 2u * kBuf + f * W::kArea);
        uint8_t *const dst = lds + f * kFrag + lane * 16u;
        auto produce = [&](uint32_t hf) {   // the span of half a superblock
#pragma unroll
            for (uint32_t g = 0; g < 8u; ++g)
                *reinterpret_cast<f16x8 *>(dst + hf * kBuf + g * (RT * kFrag)) = wt.frag(2 * hf + (g >> 2), g & 3u);
        };
        auto next = [&](uint32_t sb) {   // the superblock whose bytes are here, and the request of the one behind it
            __builtin_amdgcn_sched_barrier(0);
            wt.touch();
            __builtin_amdgcn_sched_barrier(0);
            wt.take();
            __builtin_amdgcn_sched_barrier(0);
            wt.request(sb < nsb ? sb : nsb - 1u);
            __builtin_amdgcn_sched_barrier(0);
            produce(0u);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto meet = [&] {
            __builtin_amdgcn_s_waitcnt(0xC07F);
            asm volatile("s_barrier" ::: "memory");
        };
        wt.request(0);
        next(1u);
        for (uint32_t i = 0; i < nsb; ++i) {
            meet();
            __builtin_amdgcn_sched_barrier(0);
            wt.half(1);
            produce(1u);
            __builtin_amdgcn_sched_barrier(0);
            meet();
            if (i + 1u < nsb) next(i + 2u);
        }
        return;
    }
    const uint32_t ngroup = nsb * 16u;
    const uint32_t tile_bytes = ngroup * kFrag;
    const uint32_t tt = tt0 + wave * kTM, last_tt = (tokens + 31u) / 32u - 1u;
    const lev_buffer xb0(xf + (uint64_t)(tt < last_tt ? tt : last_tt) * tile_bytes, tile_bytes);
    const lev_buffer xb1(xf + (uint64_t)(tt + 1u < last_tt ? tt + 1u : last_tt) * tile_bytes, tile_bytes);
    lev_u32x4 xr[RING][kTM];
    auto x_request = [&](uint32_t n, int slot) {
        xr[slot][0] = xb0.load16(lane * 16u, 0, n * kFrag);
        xr[slot][1] = xb1.load16(lane * 16u, 0, n * kFrag);
    };
#pragma unroll
    for (int n = 0; n < RING; ++n) x_request(n, n);
    f32x16 acc[RT][kTM];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int m = 0; m < kTM; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[r][m][i] = 0.f;
    f16x8 b[4][RT];
    const uint8_t *const bb = lds + lane * 16u;
    auto b_read = [&](int g, int r, uint32_t buf) { b[g & 3][r] = *reinterpret_cast<const f16x8 *>(bb + buf * kBuf + (g * RT + r) * kFrag); };
    // products of group g of a span whose first group is n0, meanwhile group `rg` of buffer rbuf is read
    auto phase = [&](int g, uint32_t n0, int rg, uint32_t rbuf) {
        const int slot = g % RING;
#pragma unroll
        for (int i = 0; i < RT * kTM; ++i) {
            const int r = i % RT, m = i / RT;
            acc[r][m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, xr[slot][m]), b[g & 3][r], acc[r][m], 0, 0, 0);
            if (rg >= 0 && i < RT) b_read(rg, i, rbuf);
            if (i == RT * kTM - 1) x_request(n0 + g + RING, slot);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto meet = [&] {
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("s_barrier" ::: "memory");
    };
    meet();
#pragma unroll
    for (int r = 0; r < RT; ++r) b_read(0, r, 0u);
#pragma unroll
    for (int r = 0; r < RT; ++r) b_read(1, r, 0u);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 6; ++g) phase(g, 0u, g + 2, 0u);
    auto span = [&](auto parity, uint32_t k) {
        constexpr uint32_t p = decltype(parity)::value;
        meet();
#pragma unroll
        for (int r = 0; r < RT; ++r) b_read(0, r, p);
        __builtin_amdgcn_sched_barrier(0);
        phase(6, k * 8u - 8u, -1, 0u);
        phase(7, k * 8u - 8u, 1, p);
#pragma unroll
        for (int g = 0; g < 6; ++g) phase(g, k * 8u, g + 2, p);
    };
    uint32_t k = 1;
    for (; k + 1u < nspans; k += 2u) {
        span(std::integral_constant<uint32_t, 1>{}, k);
        span(std::integral_constant<uint32_t, 0>{}, k + 1u);
    }
    span(std::integral_constant<uint32_t, 1>{}, k);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    phase(6, k * 8u, -1, 0u);
    phase(7, k * 8u, -1, 0u);
    // past the tokens' end and for rows past the last one nothing is stored
#pragma unroll
    for (int m = 0; m < kTM; ++m) {
        const uint32_t first = (tt + m) * 32u, here = first < tokens ? (tokens - first < 32u ? tokens - first : 32u) : 0u;
        const lev_buffer out(y + (uint64_t)(here ? first : 0u) * rows, here * rows * 4u);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const uint32_t row = row0 + 32u * r + lr, at = row < rows ? (4u * lh * rows + row) * 4u : lev_buffer::kNothing;
#pragma unroll
            for (int i = 0; i < 16; ++i) out.store4(__float_as_uint(acc[r][m][i]), at, 0, (uint32_t)(8 * (i / 4) + (i % 4)) * rows * 4u);
        }
    }
}

template <typename W, int RT>
hipError_t launch_as(lev_ctx *ctx, const uint8_t *w, const uint8_t *xf, float *y, uint32_t in_dim, uint32_t rows, uint32_t tokens) {
    constexpr size_t lds = 2u * RT * 8u * kFrag + RT * W::kArea;
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&gemm_wide_kernel<W, RT>), lds); e != hipSuccess) return e;
    const uint32_t row_tiles = (rows + 32u * RT - 1u) / (32u * RT), tok_tiles = (tokens + 128u * kTM - 1u) / (128u * kTM);
    hipLaunchKernelGGL((gemm_wide_kernel<W, RT>), dim3((row_tiles * tok_tiles + 7u) / 8u * 8u), dim3(kWideThreads), lds, ctx->stream,
                       w, xf, y, in_dim, rows, tokens, row_tiles, tok_tiles);
    return hipGetLastError();
}

// plan.splits: row tiles a workgroup.  Without scratch for the fragments of X (no memory, or a program is being recorded and the
// context's is still too small) a wave of the kernel for short prompts takes all of K.
template <typename W>
hipError_t launch(lev_ctx *ctx, const uint8_t *w, const uint16_t *x, float *y, uint32_t in_dim, uint32_t rows, uint32_t tokens,
                  const lev_gemm_split_plan &plan) {
    const uint32_t tiles = (tokens + 31u) / 32u;
    uint8_t *const xf = static_cast<uint8_t *>(lev_scratch(ctx, (size_t)tiles * 32u * in_dim * 2u));
    if (!xf) return lev_gemm_split_launch(ctx, W::kQ6, w, x, y, in_dim, rows, tokens, lev_gemm_split_plan{1u, 1u, 4u});
    hipLaunchKernelGGL((gemm_x_fragments<W>), dim3((in_dim / 64u + 3u) / 4u, tiles), dim3(256), 0, ctx->stream, x,
                       reinterpret_cast<lev_u32x4 *>(xf), in_dim, tokens);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    return plan.splits == 4u ? launch_as<W, 4>(ctx, w, xf, y, in_dim, rows, tokens) : launch_as<W, 3>(ctx, w, xf, y, in_dim, rows, tokens);
}

template <typename W>
int prefill(lev_ctx *ctx, const char *op, uint32_t block_bytes, uintptr_t w_align, const void *d_w, size_t w_bytes, uint64_t w_off,
            const uint16_t *d_x_f16, size_t x_count, float *d_y, size_t y_capacity, uint32_t in_dim, uint32_t rows, uint32_t tokens) {
    if (tokens == 0 || tokens > (1u << 20)) return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "%s: %u tokens", op, tokens);
    if (in_dim > (1u << 22))
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "%s: in_dim %u above 4194304", op, in_dim);
    lev_geom g;
    int st = lev_check_matvec(ctx, op, 256, block_bytes, d_w, w_bytes, w_off, d_x_f16, x_count, (uint64_t)in_dim * tokens, d_y,
                              y_capacity, (uint64_t)rows * tokens, in_dim, rows, &g);
    if (st != LEV_OK) return st;
    const uint8_t *w = static_cast<const uint8_t *>(d_w) + w_off;
    if ((reinterpret_cast<uintptr_t>(w) & (w_align - 1u)) || (reinterpret_cast<uintptr_t>(d_x_f16) & 15u))
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "%s: weights must be %u-byte and x 16-byte aligned", op, (unsigned)w_align);
    const lev_gemm_split_plan plan = lev_gemm_split_choose(ctx, W::kQ6, in_dim, rows, tokens);
    const hipError_t e = plan.kw ? lev_gemm_split_launch(ctx, W::kQ6, w, d_x_f16, d_y, in_dim, rows, tokens, plan)
                                 : launch<W>(ctx, w, d_x_f16, d_y, in_dim, rows, tokens, plan);
    return e == hipSuccess ? LEV_OK : lev_hip_check(ctx, e, W::kQ6 ? "q6_k_gemm_prefill launch" : "q4_k_gemm_prefill launch");
}

}  // namespace

extern "C" int lev_hip_q4_k_gemm_prefill(lev_ctx *ctx, const void *d_w, size_t w_bytes, uint64_t w_off, const uint16_t *d_x_f16,
                                         size_t x_count, float *d_y, size_t y_capacity, uint32_t in_dim, uint32_t rows,
                                         uint32_t tokens) {
    LEV_REQUIRE_CTX(ctx);
    return prefill<weights_q4k>(ctx, "q4_k_gemm_prefill", 144, 16, d_w, w_bytes, w_off, d_x_f16, x_count, d_y, y_capacity, in_dim,
                                rows, tokens);
}

extern "C" int lev_hip_q6_k_gemm_prefill(lev_ctx *ctx, const void *d_w, size_t w_bytes, uint64_t w_off, const uint16_t *d_x_f16,
                                         size_t x_count, float *d_y, size_t y_capacity, uint32_t in_dim, uint32_t rows,
                                         uint32_t tokens) {
    LEV_REQUIRE_CTX(ctx);
    return prefill<weights_q6k>(ctx, "q6_k_gemm_prefill", 210, 2, d_w, w_bytes, w_off, d_x_f16, x_count, d_y, y_capacity, in_dim,
                                rows, tokens);
}
