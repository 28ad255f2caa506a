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
// What bounds it: a step of a wave is some 105 vector instructions of decode and 4 T MFMAs behind LDS reads and a
// barrier, about twice what the vector unit alone takes; 6 us of a launch are its first weights and its stores.
// 77 tokens, 4096 rows, 12288 columns of Q6_K: 27 us (218 in 256-token tiles on 32 CUs); 123 tokens, 1617 rows, 4096
// columns of Q4_K: 13.7 us (49; 17 in tiles of 128 tokens alone).
#include "prefill_decode.hpp"

#include <cmath>

namespace {

typedef lev_u32x4 u32x4_a4 __attribute__((aligned(4)));   // a vector on a dword boundary

constexpr uint32_t kTile = 4096u;        // X step of 32 tokens: 32 rows of 128 bytes
// X steps in LDS: the one in use and three on their way, or one where 160 KB hold no more
template <typename W>
constexpr uint32_t x_bufs(int t, int rw, int kw) {
    return t >= 3 || kw * (4u * t * kTile + rw * W::kArea) > 160u * 1024u ? 2u : 4u;
}

// The weights of a wave's 32 rows, a superblock column at a time: request() the column's bytes, touch() (the
// wait for them), take() them as the current column, frag() its fragments; unit(): the 16-byte unit of the
// step's X row that fragment q meets.  Rows past the end repeat the last row.
struct weights_q4k {
    static constexpr int kLoads = 5;
    static constexpr uint32_t kArea = 0u;    // LDS bytes a wave
    const uint8_t *row;
    uint32_t lh;
    lev_u32x4 nhdr, nqs[4], qs[4];
    float d1[8], mm[8];
    __device__ __forceinline__ void init(const uint8_t *w, uint32_t row0, uint32_t rows, uint32_t nsb, uint8_t *) {
        const uint32_t lane = threadIdx.x & 63u, r = row0 + (lane & 31u);
        lh = lane >> 5;
        row = w + (uint64_t)(r < rows ? r : rows - 1u) * nsb * 144u;
    }
    __device__ __forceinline__ void request(uint32_t sb) {
        const uint8_t *blk = row + (uint64_t)sb * 144u;
        nhdr = *reinterpret_cast<const lev_u32x4 *>(blk);
#pragma unroll
        for (int c = 0; c < 4; ++c) nqs[c] = *reinterpret_cast<const lev_u32x4 *>(blk + 16u + 32u * c + 16u * lh);
    }
    __device__ __forceinline__ void touch() {
        asm volatile("" : "+v"(nhdr.x), "+v"(nhdr.y), "+v"(nhdr.z), "+v"(nhdr.w));
#pragma unroll
        for (int c = 0; c < 4; ++c) asm volatile("" : "+v"(nqs[c].x), "+v"(nqs[c].y), "+v"(nqs[c].z), "+v"(nqs[c].w));
    }
    __device__ __forceinline__ void take() {
#pragma unroll
        for (int c = 0; c < 4; ++c) qs[c] = nqs[c];
        q4k_all_factors(nhdr, d1, mm);
    }
    __device__ __forceinline__ void half(int) {}
    __device__ __forceinline__ f16x8 frag(int c, int q) const {
        const bool hi = q >= 2;
        return q4k_frag(q & 1 ? qs[c].z : qs[c].x, q & 1 ? qs[c].w : qs[c].y, hi, d1[2 * c + hi], mm[2 * c + hi]);
    }
    __device__ __forceinline__ uint32_t unit(int q) const { return 2u * lh + (q < 2 ? q : 2u + q); }
};

// Q6_K blocks are 210 bytes on 2-byte boundaries.  A lane that fetches its own row's 37 dwords costs the
// address unit ten misaligned loads a column, 64 rows apart each: 84 us for 77 tokens x 4096 x 12288 on half of
// the chip, 45 without the loads.  So the wave fetches in the order of memory, from the dword that a block
// starts in: 14 pieces of 16 bytes a row (the last one ends with the block: bytes 196 .. 211), seven loads of
// 1 KB, parks them in an area of its own and reads every dword it needs back, shifted by the row's two bytes.
// (Of the dwords in which the matrix begins and ends two bytes may not be its own: read with the others, never used.)
struct weights_q6k {
    static constexpr int kLoads = 7;
    static constexpr uint32_t kRow = 240u;   // 224 bytes of pieces + 16: the 32 rows start in different banks
    static constexpr uint32_t kArea = 32u * kRow;
    const uint8_t *base;
    uint8_t *area;
    uint32_t lh, lr, row_off[kLoads], nshift, shift, stride;
    lev_u32x4 n[kLoads];
    uint32_t ql[8], qh[8], sc[4];
    float d;
    static __device__ __forceinline__ uint32_t piece(int j) {   // (recomputed: cheaper than registers)
        return (threadIdx.x & 63u) + 64u * j;
    }
    __device__ __forceinline__ void init(const uint8_t *w, uint32_t row0, uint32_t rows, uint32_t nsb, uint8_t *wave_area) {
        const uint32_t lane = threadIdx.x & 63u;
        lh = lane >> 5;
        lr = lane & 31u;
        area = wave_area;
        stride = nsb * 210u;
        base = w + (uint64_t)(row0 < rows ? row0 : rows - 1u) * stride;
        const uint32_t most = row0 < rows ? rows - 1u - row0 : 0u;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t r = piece(j) / 14u;
            row_off[j] = (r < most ? r : most) * stride;
        }
        lr_off = (lr < most ? lr : most) * stride;
    }
    uint32_t lr_off;
    __device__ __forceinline__ void request(uint32_t sb) {
        const uint8_t *const b = base + (uint64_t)sb * 210u;
        const uint32_t low = (uint32_t)(uintptr_t)b & 3u;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t i = piece(j) % 14u;
            n[j] = *reinterpret_cast<const u32x4_a4 *>((b - low) + (((low + row_off[j]) & ~3u) + (i < 13u ? 16u * i : 196u)));
        }
        nshift = ((low + lr_off) & 2u) * 8u;
    }
    __device__ __forceinline__ void touch() {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) asm volatile("" : "+v"(n[j].x), "+v"(n[j].y), "+v"(n[j].z), "+v"(n[j].w));
    }
    __device__ __forceinline__ void take() {
        // the area is this wave's own: LDS runs a wave's accesses in order
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t q = piece(j), r = q / 14u;
            *reinterpret_cast<lev_u32x4 *>(area + r * kRow + (q - 14u * r) * 16u) = n[j];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        shift = nshift;
        const uint8_t *const mine = area + lr * kRow;
        const lev_u32x4 s = *reinterpret_cast<const lev_u32x4 *>(mine + 192u);
        const uint32_t last = *reinterpret_cast<const uint32_t *>(mine + 220u);   // bytes 208 .. 211 from the first dword
        sc[0] = __builtin_amdgcn_alignbit(s.y, s.x, shift);
        sc[1] = __builtin_amdgcn_alignbit(s.z, s.y, shift);
        sc[2] = __builtin_amdgcn_alignbit(s.w, s.z, shift);
        sc[3] = __builtin_amdgcn_alignbit(last, s.w, shift);
        d = lev_f16_bits_to_f32((last >> shift) & 0xFFFFu);
        half(0);
    }
    // the codes of half a column: 32 bytes of ql (the lane's half of 64), 32 of qh
    __device__ __forceinline__ void half(int hf) {
        const uint8_t *const mine = area + lr * kRow;
        auto eight = [&](const uint8_t *p, uint32_t (&o)[8]) {
            const lev_u32x4 a = *reinterpret_cast<const lev_u32x4 *>(p), b = *reinterpret_cast<const lev_u32x4 *>(p + 16);
            const uint32_t c = *reinterpret_cast<const uint32_t *>(p + 32);
            o[0] = __builtin_amdgcn_alignbit(a.y, a.x, shift);
            o[1] = __builtin_amdgcn_alignbit(a.z, a.y, shift);
            o[2] = __builtin_amdgcn_alignbit(a.w, a.z, shift);
            o[3] = __builtin_amdgcn_alignbit(b.x, a.w, shift);
            o[4] = __builtin_amdgcn_alignbit(b.y, b.x, shift);
            o[5] = __builtin_amdgcn_alignbit(b.z, b.y, shift);
            o[6] = __builtin_amdgcn_alignbit(b.w, b.z, shift);
            o[7] = __builtin_amdgcn_alignbit(c, b.w, shift);
        };
        eight(mine + 64u * hf + 32u * lh, ql);
        eight(mine + 128u + 32u * hf, qh);
    }
    __device__ __forceinline__ f16x8 frag(int c, int q) const {
        const int hf = c >> 1, np = c & 1;
        const float ds = d * (float)(int)__builtin_amdgcn_sbfe((int)sc[2 * hf + np], 8u * (2u * lh + (uint32_t)(q >> 1)), 8u);
        const float nbm = -1056.0f * ds;
        f16x8 f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t a = ql[2 * q + i], h = qh[2 * q + i];
            const uint32_t code = np ? (((a >> 4) & 0x0F0F0F0Fu) | ((h >> (2u * lh)) & 0x30303030u))
                                     : ((a & 0x0F0F0F0Fu) | ((h << (4u - 2u * lh)) & 0x30303030u));
            q6g_put4_mix(code, ds, nbm, f, 4 * i);
        }
        return f;
    }
    __device__ __forceinline__ uint32_t unit(int q) const { return 4u * lh + (uint32_t)q; }
};

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
    // X: load j brings the 128 bytes of eight tokens; 16-byte unit c of token t lies at c ^ (t & 7)
    constexpr uint32_t kBufs = x_bufs<W>(T, RW, KW);
    constexpr int kXLoads = 4 * T / RW;
    const uint8_t *xsrc[kXLoads];
#pragma unroll
    for (int j = 0; j < kXLoads; ++j) {
        const uint32_t tl = 8u * (rw + RW * j) + (lane >> 3), t = tok0 + tl < tokens ? tok0 + tl : tokens - 1u;
        xsrc[j] = reinterpret_cast<const uint8_t *>(x) + ((uint64_t)t * in_dim * 2u + 16u * ((lane & 7u) ^ (tl & 7u)));
    }
    const uint32_t xlds = lev_lds_offset(lds) + kw * (kBufs * T * kTile) + rw * 1024u, steps = (sb1 - sb0) * 4u;
    auto x_request = [&](uint32_t step) {
        const uint32_t s = sb0 * 4u + (step < steps ? step : steps - 1u);   // past the end: any valid step, never read
#pragma unroll
        for (int j = 0; j < kXLoads; ++j) lev_load_lds16(xsrc[j] + (uint64_t)s * 128u, xlds + (step % kBufs) * (T * kTile) + j * (RW * 1024u));
    };
    const uint8_t *const xmine = lds + kw * (kBufs * T * kTile) + lr * 128u;

#pragma unroll
    for (uint32_t s = 0; s + 1u < kBufs; ++s) x_request(s);
    W wt;
    wt.init(w, row0, rows, nsb, lds + KW * (kBufs * T * kTile) + wave * W::kArea);
    wt.request(sb0);
    f32x16 acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;

    wt.touch();
    wt.take();
    f16x8 a[2][T], b = wt.frag(0, 0);
    for (uint32_t i = 0; i < most; ++i) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t step = i * 4u + c;
            // This step's X has landed: newer are the X of the steps behind it and, behind a superblock's
            // first step, the next superblock's weights, which are wanted by the fourth.
            static_assert(kBufs == 4u || kBufs == 2u, "the counts below");
            if (c == 1 || (c == 2 && kBufs == 4u)) LEV_WAIT_VMCNT((kBufs - 2u) * kXLoads + W::kLoads);
            else LEV_WAIT_VMCNT((kBufs - 2u) * kXLoads);
            if (c == 3) wt.touch();   // the compiler's own wait for them goes here, where it is free
            __builtin_amdgcn_sched_barrier(0);
            lev_barrier_lds();          // everybody's has, and everybody is done with the other buffer
            x_request(step + kBufs - 1u);
            if (c == 0) {
                __builtin_amdgcn_sched_barrier(0);
                const uint32_t sb = sb0 + i + 1u;
                wt.request(sb < sb1 ? sb : sb1 - 1u);
                __builtin_amdgcn_sched_barrier(0);
            }
            const uint8_t *const xb = xmine + (step % kBufs) * (T * kTile);
            auto a_read = [&](int q) {
#pragma unroll
                for (int t = 0; t < T; ++t)
                    a[q & 1][t] = *reinterpret_cast<const f16x8 *>(xb + t * kTile + 16u * (wt.unit(q) ^ (lr & 7u)));
            };
            if (sb0 + i < sb1) {
                a_read(0);
                a_read(1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[q & 1][t], b, acc[t], 0, 0, 0);
                    // behind them, while they run: the X fragments of the product after the next and the next B
                    if (q < 2) a_read(q + 2);
                    if (q < 3) {
                        b = wt.frag(c, q + 1);
                    } else if (c < 3) {
                        if (c == 1) wt.half(1);
                        b = wt.frag(c + 1, 0);
                    } else {
                        wt.take();
                        b = wt.frag(0, 0);
                    }
                    // one MFMA, then what can issue while it runs: a wave issues in order, and a second MFMA
                    // behind the first would hold it for 32 clocks
#pragma unroll
                    for (int t = 0; t < T; ++t) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                    // MFMA
                        if (q < 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);         // LDS read
                        __builtin_amdgcn_sched_group_barrier(0x002, (28 + T - 1) / T, 0);     // VALU
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    }
    LEV_WAIT_VMCNT(0);   // the request past the end lands before the LDS is used again

    if (KW > 1) {
        // partial tiles of slices 1.. -> LDS, added to the first slice's in slice order
        float *const red = reinterpret_cast<float *>(lds);
        lev_barrier_lds();
        if (kw != 0u) {
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) red[((((kw - 1u) * RW + rw) * T + t) * 16 + i) * 64 + lane] = acc[t][i];
        }
        lev_barrier_lds();
        if (kw != 0u) return;
#pragma unroll
        for (uint32_t k = 1; k < KW; ++k)
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[t][i] += red[((((k - 1u) * RW + rw) * T + t) * 16 + i) * 64 + lane];
    }
    if (row >= rows) return;
    float *const dst = out + (uint64_t)zl * tokens * rows + row;
    if (add) {
#pragma unroll 1
        for (int t = 0; t < T; ++t) {
            const uint32_t first = tok0 + 32u * t + 4u * lh;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const uint32_t tok = first + 8u * (i / 4) + (i % 4);
                float v = 0.f;
#pragma unroll
                for (int k = 0; k < T; ++k) v = k == t ? acc[k][i] : v;
                if (tok < tokens) dst[(uint64_t)tok * rows] += v;
            }
        }
        return;
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t tok = tok0 + 32u * t + 8u * (i / 4) + 4u * lh + (i % 4);
            if (tok < tokens) dst[(uint64_t)tok * rows] = acc[t][i];
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
        // a program is being recorded and the scratch is still too small: a launch for every slice, each added to y where
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
// take, from times measured over 1000 to 32000 rows, 1024 to 12288 columns and 17 to 1000 tokens (us; a step is 64 values
// of K, t = 32-token tiles a wave; of 60 shapes the choice was within 0.2 % of the best on average, 5 % at worst).
//   256-token tiles:  a round of workgroups (one per CU) 6.1 + in_dim / 1024 * (9.8 + 3.8 * share of the CUs it
//                     fills), Q6_K 5.7 + in_dim / 1024 * (19.2 + 3.5 *): 46 to 60 us at 4096 columns of Q4_K;
//   KW = 1:           a round of up to two workgroups a CU; their steps take 1.6 times those of one alone;
//   KW = 2, KW = 4:   a round of one a CU, and with S > 1 splits the kernel that adds and its reads and writes.
// Lower token tiles are more workgroups that decode the same weights: what fills the chip where rows alone do not.
// Beyond 1024 tokens the times of KW = 1 outgrow these, by 1.1 to 1.45, with the tokens that its tiles really hold
// (those of 256 tokens stay within 0.87 to 1.1).  Over 216 shapes of 1025 to 8192 tokens the 256-token tiles were the
// faster ones where nearly every token of them is one and the CUs are full: for Q6_K from 15/16 of the CUs (4096 x 4096 at
// 4096 tokens 174.7 us against 187.2, 32000 x 4096 at 4096 tokens 1361 against 1449), unless there are more than 2^28
// weights (220 MB, about what the Infinity Cache holds: 32000 rows of 12288 at 3072 tokens 4 % more); for Q4_K from 31/32 of them and
// eight token tiles (12288 x 4096 at 4096 tokens 469 us against 505, at 2048 tokens 236 against 242), but not over short
// rows (16384 rows of 1024 at 8192 tokens 2 % more), and where the estimates are within 1.1 (12288 x 4096 at 1500 tokens
// 180 us against 193).  47 shapes of Q6_K and 23 of Q4_K are faster so, by some 4 % on average and none slower by more
// than 0.4 %; Q4_K at 2048 tokens is between 2.7 % faster and 1.5 % slower, by the shape and the card's clock.
// Tall matrices (768 row tiles and more) and rows of fewer than six superblocks are never cut along K, so that
// there every kernel adds in the same order.
lev_gemm_split_plan lev_gemm_split_choose(const lev_ctx *ctx, bool q6, uint32_t in_dim, uint32_t rows, uint32_t tokens,
                                          uint32_t big_rows) {
    const double cus = ctx->num_cus;
    const uint32_t nsb = in_dim / 256u, tiles = (tokens + 31u) / 32u;
    const double big_wgs = (double)((rows + big_rows - 1u) / big_rows) * ((tokens + 255u) / 256u);
    const double big_rounds = std::ceil(big_wgs / cus), fill = big_wgs / (big_rounds * cus);
    lev_gemm_split_plan best{0u, 1u, 1u};
    double least = big_rounds * (q6 ? 5.7 + in_dim / 1024.0 * (19.2 + 3.5 * fill) : 6.1 + in_dim / 1024.0 * (9.8 + 3.8 * fill));
    if (tokens > 1024u) {
        const uint64_t tiled = (tokens + 255ull) / 256u * 256u;
        if (tokens * 32ull >= tiled * 31u && (q6 ? fill >= 15.0 / 16.0 && (uint64_t)in_dim * rows <= 1u << 28
                                                 : fill >= 31.0 / 32.0 && in_dim >= 2048u && tiled >= 2048u))
            return best;
        if (!q6) least /= 1.1;
    }
    struct cost { double start, step, per_tile, full, sum, sum_mb; };
    const cost k1 = q6 ? cost{4.9, 0.383, 0.067, 0.60, 0, 0} : cost{4.0, 0.267, 0.076, 0.66, 0, 0};
    const cost k2 = q6 ? cost{4.3, 0.558, 0.145, 0.16, 3.1, 0.7} : cost{3.9, 0.363, 0.165, 0.08, 2.9, 0.75};
    const cost k4 = q6 ? cost{4.1, 0.534, 0.248, 0.02, 4.8, 0.0} : cost{4.6, 0.206, 0.287, 0.05, 3.1, 0.56};
    auto offer = [&](double us, uint32_t kw, uint32_t splits, uint32_t t) {
        if (us < least) {
            least = us;
            best = lev_gemm_split_plan{kw, splits, t};
        }
    };
    for (uint32_t t = 1; t <= 4u && t <= tiles; ++t) {
        const double tok_tiles = (tiles + t - 1u) / t;
        // workgroups, whole eighths of them on an XCD each
        auto wgs_of = [&](uint32_t rows_wg, uint32_t splits) { return 8.0 * std::ceil((rows + rows_wg - 1u) / rows_wg * tok_tiles * splits / 8.0); };
        {
            const double n = wgs_of(128u, 1u), whole = std::floor(n / (2.0 * cus)), rest = n - whole * 2.0 * cus;
            const double rounds = whole + (rest > 0.0 ? 1.0 : 0.0), pairs = whole + (rest > cus ? 1.0 : 0.0);
            offer(rounds * k1.start + 4.0 * nsb * (k1.step + k1.per_tile * t) * (rounds + k1.full * pairs), 1u, 1u, t);
        }
        if ((rows + 31u) / 32u >= 768u || nsb < 6u) continue;
        for (uint32_t kw = 2; kw <= 4u; kw += 2u) {
            if (kw == 4u && q6 && t == 4u) continue;   // (more LDS than there is)
            const cost &k = kw == 2u ? k2 : k4;
            for (uint32_t s = 1; s <= 8u && s * kw <= nsb; ++s) {
                const double n = wgs_of(kw == 2u ? 128u : 64u, s), rounds = std::ceil(n / cus), full = n / (rounds * cus);
                const double steps = 4.0 * ((nsb + kw * s - 1u) / (kw * s));
                offer(rounds * (k.start + steps * (k.step + k.per_tile * t) * (1.0 + k.full * full)) +
                          (s > 1u ? k.sum + k.sum_mb * 1e-6 * (s + 1.0) * tokens * rows : 0.0), kw, s, t);
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
