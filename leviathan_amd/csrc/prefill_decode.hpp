// What the prefill GEMMs share: decoding Q4_K and Q6_K weights to fp16 fragments.
#pragma once

#include "lev_common.hpp"

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// (d*sc, dmin*m) of the 8 sub-blocks of a superblock (lev-cpu/src/lib.rs:64-74,
// 117-124).
__device__ __forceinline__ void q4k_all_factors(const lev_u32x4 hdr, float d1[8], float mm[8]) {
    const float d = lev_f16_bits_to_f32(hdr.x & 0xFFFFu);
    const float dmin = lev_f16_bits_to_f32(hdr.x >> 16);
    const uint32_t s03 = hdr.y, s47 = hdr.z, s811 = hdr.w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t sc = (s03 >> (8 * j)) & 63u, mn = (s47 >> (8 * j)) & 63u;
        d1[j] = d * (float)sc;
        mm[j] = dmin * (float)mn;
        uint32_t a = (s811 >> (8 * j)) & 0xFFu;
        uint32_t sc2 = (a & 0x0Fu) | (((s03 >> (8 * j + 6)) & 3u) << 4);
        uint32_t mn2 = (a >> 4) | (((s47 >> (8 * j + 6)) & 3u) << 4);
        d1[4 + j] = d * (float)sc2;
        mm[4 + j] = dmin * (float)mn2;
    }
}

// One weight exactly as the reference rounds it: f32(d1*q - mm) first, THEN
// round-to-nearest-even to fp16 (dequant_block_f32 followed by f32_to_f16_bits,
// lev-cli/src/main.rs:1201-1217).  The empty asm pins the f32 value in a
// register so that the compiler cannot merge the multiply-add with the
// conversion into a single-rounding mixed-precision FMA, which differs from
// the two-step rounding in about one weight in ten thousand.
__device__ __forceinline__ _Float16 q4k_weight_f16(float d1, float code, float mm) {
    float w32 = fmaf(d1, code, -mm);   // d1*code is exact (17 + 4 bits): one rounding, as in the reference
    asm("" : "+v"(w32));
    return (_Float16)w32;
}

// 8 weights (one per code byte of the two dwords, nibble selected by `hi`)
// -> fp16 B fragment, bit-exact with fp16(f32(d1*q - mm)).
__device__ __forceinline__ f16x8 q4k_frag(uint32_t q0, uint32_t q1, bool hi, float d1, float mm) {
    uint32_t a = hi ? (q0 >> 4) : q0, b = hi ? (q1 >> 4) : q1;
    a &= 0x0F0F0F0Fu;
    b &= 0x0F0F0F0Fu;
    // opaque from here: the compiler would otherwise fold the mask into four
    // bit-field extracts per dword instead of using v_cvt_f32_ubyte0..3 directly
    asm("" : "+v"(a));
    asm("" : "+v"(b));
    f16x8 f;
    f[0] = q4k_weight_f16(d1, (float)(a & 0xFFu), mm);
    f[1] = q4k_weight_f16(d1, (float)((a >> 8) & 0xFFu), mm);
    f[2] = q4k_weight_f16(d1, (float)((a >> 16) & 0xFFu), mm);
    f[3] = q4k_weight_f16(d1, (float)(a >> 24), mm);
    f[4] = q4k_weight_f16(d1, (float)(b & 0xFFu), mm);
    f[5] = q4k_weight_f16(d1, (float)((b >> 8) & 0xFFu), mm);
    f[6] = q4k_weight_f16(d1, (float)((b >> 16) & 0xFFu), mm);
    f[7] = q4k_weight_f16(d1, (float)(b >> 24), mm);
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

// The GEMM for short prompts and for shapes whose 256-token tiles leave the chip idle (gemm_split.hip):
// kw = 0: the 256-token kernel takes the shape (`big_rows` rows a workgroup); else K slices a workgroup, and
// workgroups that share a tile.
struct lev_gemm_split_plan { uint32_t kw, splits, t; };
lev_gemm_split_plan lev_gemm_split_choose(const lev_ctx *ctx, bool q6, uint32_t in_dim, uint32_t rows, uint32_t tokens,
                                          uint32_t big_rows);
hipError_t lev_gemm_split_launch(lev_ctx *ctx, bool q6, const uint8_t *w, const uint16_t *x, float *y, uint32_t in_dim,
                                 uint32_t rows, uint32_t tokens, const lev_gemm_split_plan &plan);
