// What the prefill GEMMs share: decoding Q4_K and Q6_K weights to fp16 fragments.
#pragma once

#include "lev_common.hpp"

#include <type_traits>

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Of sub-blocks 4 HALF .. 4 HALF + 3 of a superblock: d*sc, times the power of two that q4k_frag wants (2^24 for the sub-blocks
// of the low nibbles, 2^20 for those of the high ones), and dmin*m (lev-cpu/src/lib.rs:64-74, 117-124).
template <int HALF>
__device__ __forceinline__ void q4k_factors(const lev_u32x4 hdr, float d1[8], float mm[8]) {
    const float d = lev_f16_bits_to_f32(hdr.x & 0xFFFFu) * 0x1p20f, d16 = d * 16.f;
    const float dmin = lev_f16_bits_to_f32(hdr.x >> 16);
    const uint32_t s03 = hdr.y, s47 = hdr.z, s811 = hdr.w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t sc = (s03 >> (8 * j)) & 63u, mn = (s47 >> (8 * j)) & 63u;
        if (HALF) {
            const uint32_t a = (s811 >> (8 * j)) & 0xFFu;
            sc = (a & 0x0Fu) | (((s03 >> (8 * j + 6)) & 3u) << 4);
            mn = (a >> 4) | (((s47 >> (8 * j + 6)) & 3u) << 4);
        }
        d1[4 * HALF + j] = (j & 1 ? d : d16) * (float)sc;
        mm[4 * HALF + j] = dmin * (float)mn;
    }
}

// One weight exactly as the reference rounds it: f32(d1*q - mm) first, THEN
// round-to-nearest-even to fp16 (dequant_block_f32 followed by f32_to_f16_bits,
// lev-cli/src/main.rs:1201-1217).  The empty asm pins the f32 value in a
// register so that the compiler cannot merge the multiply-add with the
// conversion into a single-rounding mixed-precision FMA, which differs from
// the two-step rounding in about one weight in ten thousand.
// code: the weight's nibble where it lies in a 16-bit half, which as an fp16 number is q * 2^-24 or, four bits up,
// q * 2^-20; the multiply-add takes it as it is, with no conversion of its own.
__device__ __forceinline__ _Float16 q4k_weight_f16(float d1, _Float16 code, float mm) {
    float w32 = fmaf((float)code, d1, -mm);   // d1*code is exact (17 + 4 bits): one rounding, as in the reference
    asm("" : "+v"(w32));
    return (_Float16)w32;
}

// 8 weights (one per code byte of the two dwords, nibble selected by `hi`)
// -> fp16 B fragment, bit-exact with fp16(f32(d1*q - mm)).
__device__ __forceinline__ f16x8 q4k_frag(uint32_t q0, uint32_t q1, bool hi, float d1, float mm) {
    const uint32_t mask = hi ? 0x00F000F0u : 0x000F000Fu;
    f16x8 f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t q = i ? q1 : q0;
        const f16x2 even = __builtin_bit_cast(f16x2, q & mask), odd = __builtin_bit_cast(f16x2, (q >> 8) & mask);
        f[4 * i + 0] = q4k_weight_f16(d1, even.x, mm);
        f[4 * i + 1] = q4k_weight_f16(d1, odd.x, mm);
        f[4 * i + 2] = q4k_weight_f16(d1, even.y, mm);
        f[4 * i + 3] = q4k_weight_f16(d1, odd.y, mm);
    }
    return f;
}

struct __attribute__((packed, aligned(2))) u32x4_a2 { uint32_t v[4]; };

// Four codes packed in `c` -> fp16 weights out[at..at+3], one instruction per weight
// (Q6.swift:4-62 for the layout).  ds = d * sc has at most 18
// significant bits and q - 32 six, so ds * (q - 32) is exact in f32 and the reference's
// two roundings (f32, then fp16) are one rounding of the exact product.  A code byte
// under the exponent byte 0x64 is the fp16 number 1024 + q; fma(1024 + q, ds, -1056 ds)
// is that exact product, and the mixed-precision FMA rounds it to fp16 once.
__device__ __forceinline__ void q6g_put4_mix(uint32_t c, float ds, float nbm, f16x8 &out, int at) {
    const uint32_t ma = __builtin_amdgcn_perm(0x64646464u, c, 0x04020400u);   // bytes (c0, 0x64, c2, 0x64)
    const uint32_t mb = __builtin_amdgcn_perm(0x64646464u, c, 0x04030401u);   // bytes (c1, 0x64, c3, 0x64)
    const f16x2 a = __builtin_bit_cast(f16x2, ma), b = __builtin_bit_cast(f16x2, mb);
    out[at + 0] = (_Float16)fmaf((float)a.x, ds, nbm);
    out[at + 1] = (_Float16)fmaf((float)b.x, ds, nbm);
    out[at + 2] = (_Float16)fmaf((float)a.y, ds, nbm);
    out[at + 3] = (_Float16)fmaf((float)b.y, ds, nbm);
}

typedef lev_u32x4 u32x4_a4 __attribute__((aligned(4)));   // a vector on a dword boundary

// The weights of a wave's 32 rows, a superblock column at a time: request() the column's bytes, touch() (the
// wait for them), take() them as the current column, frag() its fragments; unit(): the 16-byte unit of the
// step's X row that fragment q meets.  Rows past the end repeat the last row.
struct weights_q4k {
    static constexpr bool kQ6 = false;
    static constexpr int kLoads = 5;
    static constexpr uint32_t kArea = 0u;    // LDS bytes a wave
    const uint8_t *row;
    uint32_t lh;
    lev_u32x4 nhdr, hdr, nqs[4], qs[4];
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
        hdr = nhdr;
        half(0);
    }
    // the factors of half a column
    __device__ __forceinline__ void half(int hf) {
        if (hf) q4k_factors<1>(hdr, d1, mm);
        else q4k_factors<0>(hdr, d1, mm);
    }
    __device__ __forceinline__ void clear() {   // fragments of zeros
#pragma unroll
        for (int c = 0; c < 4; ++c) qs[c] = lev_u32x4{0u, 0u, 0u, 0u};
        hdr = lev_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < 8; ++j) d1[j] = mm[j] = 0.f;
    }
    __device__ __forceinline__ f16x8 frag(int c, int q) const {
        const bool hi = q >= 2;
        return q4k_frag(q & 1 ? qs[c].z : qs[c].x, q & 1 ? qs[c].w : qs[c].y, hi, d1[2 * c + hi], mm[2 * c + hi]);
    }
    static __device__ __forceinline__ uint32_t unit_of(uint32_t half, int q) { return 2u * half + (q < 2 ? q : 2u + q); }
    __device__ __forceinline__ uint32_t unit(int q) const { return unit_of(lh, q); }
};

// Q6_K blocks are 210 bytes on 2-byte boundaries.  A lane that fetches its own row's 37 dwords costs the
// address unit ten misaligned loads a column, 64 rows apart each: 84 us for 77 tokens x 4096 x 12288 on half of
// the chip, 45 without the loads.  So the wave fetches in the order of memory, from the dword that a block
// starts in: 14 pieces of 16 bytes a row (the last one ends with the block: bytes 196 .. 211), seven loads of
// 1 KB, parks them in an area of its own and reads every dword it needs back, shifted by the row's two bytes.
// (Of the dwords in which the matrix begins and ends two bytes may not be its own: read with the others, never used.)
struct weights_q6k {
    static constexpr bool kQ6 = true;
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
    __device__ __forceinline__ void clear() {   // fragments of zeros
#pragma unroll
        for (int j = 0; j < 8; ++j) ql[j] = qh[j] = 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[j] = 0u;
        d = 0.f;
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
    static __device__ __forceinline__ uint32_t unit_of(uint32_t half, int q) { return 4u * half + (uint32_t)q; }
    __device__ __forceinline__ uint32_t unit(int q) const { return unit_of(lh, q); }
};

// Which kernel takes a prefill GEMM (gemm_split.hip).  kw = 0: the one of 256-token tiles (gemm_wide.hip) with `splits` tiles
// of 32 rows a workgroup; else the one for short prompts and small matrices: K slices a workgroup, workgroups that share a
// tile, token tiles of 32 a wave.
struct lev_gemm_split_plan { uint32_t kw, splits, t; };
lev_gemm_split_plan lev_gemm_split_choose(const lev_ctx *ctx, bool q6, uint32_t in_dim, uint32_t rows, uint32_t tokens);
hipError_t lev_gemm_split_launch(lev_ctx *ctx, bool q6, const uint8_t *w, const uint16_t *x, float *y, uint32_t in_dim,
                                 uint32_t rows, uint32_t tokens, const lev_gemm_split_plan &plan);
