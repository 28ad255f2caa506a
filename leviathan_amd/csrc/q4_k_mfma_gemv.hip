// RMSNorm + Q4_K multi-column GEMV on the integer matrix cores, for gfx950.
//
// Stands in for Builder::norm_quant + Builder::matvec with nb columns
// (rust/crates/lev-model/src/gpu.rs:295, 334-370; q4k.matvec,
// lev-forge/src/glsl.rs:157-281 and q8.rs:196-326): the weights are read once
// and applied to every column.
//
// One pass over W; at these sizes the vector ALU, not HBM, sets the time, so
// the formulation minimises instructions per weight.  Per superblock of 256
// weights of a row (w = d*sc_j*q - dmin*m_j, rust/crates/lev-cpu/src/lib.rs:111-154):
//
//   y += d * sum_j sc_j * (sum_k q_k x_k)  -  dmin * sum_j m_j * (sum_k x_k)
//
// Every sum is formed WITHOUT rounding:
//   * per superblock and column the activations become integers
//     X = rint(x * 2^(25-e)), 2^e the power of two above the superblock's largest
//     magnitude: |X| <= 2^25, a step of 2^-25 of that power of two (the top two
//     binades of f32 values are represented exactly).  X is written in four
//     balanced base-256 digits, X = ((b3*256 + b2)*256 + b1)*256 + b0 with every
//     b in [-128, 127] (|b3| <= 2): four int8 planes.
//   * v_mfma_i32_16x16x32_i8 per sub-block: the 16 A rows are 4 columns of x
//     times 4 digit planes, B is 16 weight rows x 32 codes (4-bit, unscaled).
//     The four planes of a column land in the four accumulator registers of one
//     lane, which multiplies them by the sub-block's 6-bit scale and adds them up
//     over the superblock in 32-bit integers (below 2^25 in magnitude per plane).
//   * once per superblock the planes are recombined in f64 (40-bit integers,
//     exact), d, dmin and the power of two are applied in f64, the partial sums of
//     a row are added in f64, and one rounding to f32 ends it.
// The result is the dot product of the dequantized row with the quantized
// activations, rounded once; the order of the additions does not show.
//
// lane (r, g) = (l % 16, l / 16) loads row r's 16-byte header and code bytes
// 8g..8g+7 of each 32-byte chunk (low nibbles: sub-block 2c, high: 2c+1); the
// output lane of weight row r is the lane that loaded its header.
//
// Workgroup = 16 waves, one per CU (the digit planes of four columns of 4096
// activations take 64 KB of LDS).  The waves of a workgroup share 16 weight rows,
// one superblock column each; their partial sums meet in LDS.
//
// Five to eight columns of a matrix of many rows, or three and more of a row of more than sixteen superblocks: the planes are made
// once per launch by a small kernel in front (q4k_planes_kernel, below) instead of by every workgroup.  Fewer superblocks, most
// other shapes: a wave makes the planes of the superblock column that it multiplies (OWN, q4k_own_takes).
//
// Against 64-bit sums, on normal activations: 5e-8 to 6e-8 (2-norm); the f32 chains of the vector-ALU kernel, which
// three and more columns of rows wider than 8192 take without planes, leave 1.4e-7.  A value far below the largest of its
// superblock keeps multiples of 2^-26 of that maximum.
//
// A NaN or infinity in a column of x makes every output of that column NaN.
#include "lev_common.hpp"

#include <cstdlib>

namespace {

constexpr int kMThreads = 1024;
constexpr int kMWaves = kMThreads / LEV_WAVE;
constexpr uint32_t kNZeroBytes = 1024;   // what masked lanes of the narrow kernel read as their A operand

typedef int lev_i4 __attribute__((ext_vector_type(4)));
typedef uint32_t lev_u4 __attribute__((ext_vector_type(4)));
typedef uint32_t lev_u2 __attribute__((ext_vector_type(2)));
typedef double lev_d2 __attribute__((ext_vector_type(2)));

struct q4k_regs {
    lev_u4 hdr, a, b;
};

// Three 16-byte loads per lane: the header, and bytes [16*(g/2), +16) of chunk
// 2i + g%2 for i = 0, 1.  A wave's load covers 64 contiguous bytes per row.
__device__ __forceinline__ void q4k_issue(const uint8_t *__restrict__ w, uint64_t row_bytes, uint32_t row,
                                          uint32_t sb, uint32_t g, q4k_regs &R) {
    const uint8_t *p = w + (uint64_t)row * row_bytes + (uint64_t)sb * 144u;
    R.hdr = *reinterpret_cast<const lev_u4 *>(p);
    const uint8_t *q = p + 16u + 32u * (g & 1u) + 16u * (g >> 1);
    R.a = *reinterpret_cast<const lev_u4 *>(q);
    R.b = *reinterpret_cast<const lev_u4 *>(q + 64u);
}

// The MFMA wants bytes [8g, 8g+8) of every chunk in lane group g.  Lane groups g
// and g^1 (16 lanes apart) hold each other's second piece: the even group's upper
// half is the odd group's piece of chunk 2i, the odd group's lower half the even
// group's piece of chunk 2i+1.  One row swap per dword puts both in place:
// afterwards (x, y) is the lane's piece of chunk 2i and (z, w) of chunk 2i+1.
__device__ __forceinline__ void q4k_exchange(lev_u4 &v) {
    const auto s0 = __builtin_amdgcn_permlane16_swap(v.x, v.z, false, false);
    const auto s1 = __builtin_amdgcn_permlane16_swap(v.y, v.w, false, false);
    v.x = s0[0];
    v.z = s0[1];
    v.y = s1[0];
    v.w = s1[1];
}

// Byte offset of 16-byte unit u (= 8*kg + A row / 2) inside a sub-block's 512 bytes
// of digit planes.  The staging threads of one wave write units 8*kg + 2*(column % 4)
// of many sub-blocks at once; unswizzled, k-groups 0 and 2 and all sub-blocks would
// meet in the same banks.  Flipping bit 0 for the upper two k-groups and bit 1 for
// odd sub-blocks spreads eight consecutive lanes over eight bank groups, and is a
// permutation of the units inside a sub-block, so the MFMA's reads stay conflict-free.
__device__ __forceinline__ uint32_t q4k_unit(uint32_t u, uint32_t kg, uint32_t j) {
    return (u ^ (kg >> 1) ^ ((j & 1u) << 1)) * 16u;
}

// LDS, for SB superblocks and NL = 4*NX layout columns:
//   dig  [8*SB][NX][4 k-groups][16 A rows][8 bytes]   digit planes, A row = 4*(column % 4) + plane
//   sxd  [SB][NL][8] f64                               sum of X per sub-block
//   part [pb][wave][16 rows][NL] f64                   partial sums of a row group
//   psb  [SB][NL] f64                                  2^(e-25) per superblock
//   inv  [NL] f64, bad [NL] u32
//   run  [NL][8*SB] f64                                sums of squares (RMSNorm); in the digit area,
//                                                      which is written once they have been added up
template <int NX>
struct q4k_lds {
    static constexpr uint32_t NL = 4u * NX;
    static __host__ __device__ size_t dig_bytes(uint32_t subs) { return (size_t)subs * NX * 512u; }
    // pb: buffers for the partial sums (two save a barrier per row group)
    static __host__ __device__ size_t total(uint32_t subs, uint32_t pb) {
        return dig_bytes(subs) + (size_t)subs * NL * 8u + (size_t)pb * kMWaves * 16u * NL * 8u +
               (size_t)(subs >> 3) * NL * 8u + (size_t)NL * 12u;
    }
};

// ---------------------------------------------------------------------------
// The digit planes made ONCE per launch instead of once per workgroup.
//
// Turning a column of activations into digit planes costs a compute unit about a
// microsecond whoever does it, and in q4_k_mfma_gemv every workgroup does it for every
// column: at eight columns that is more than half of the kernel's instructions, and from 16384
// values on they do not fit its LDS.  So q4k_planes_kernel (one workgroup per column) writes the planes to device scratch in the order the matrix cores read them, and
// the workgroups of q4_k_mfma_gemv<NC, SHORT, true> load the planes of their wave's
// superblock column straight into registers: no staging, no digit area in LDS, no LDS read
// per product.  The numbers are the same integers, so the outputs are the same bits.
//
// A row of more than sixteen superblocks is cut into slices of at most sixteen (gridDim.y), a workgroup
// taking one: the sums of a row group's slices meet in scratch, in f64, and the last workgroup to get there
// adds them in order (hand-over as in lev_common.hpp; every row group has a counter, cleared with the
// planes).  Six columns of 6095 x 4608 25.5 us with four columns a launch, 14.0 like this; seven of
// 1052 x 8448 40.1 us on the vector ALU, 11.4; eight of 16000 x 12288 199 and 43.
//
// Scratch, for NX groups of four layout columns and SB superblocks:
//   planes [SB][4 sub-block pairs][NX][64 lanes][16 B]   lane (r, g): A row r (4 * (column % 4) + plane,
//          plane 0 the highest digit), k-group g, of sub-blocks 2jp (low 8 bytes) and 2jp + 1 (high)
//   psb    [SB][4 * NX] f64                               2^(e-151) per superblock and column; NaN where one of
//          its activations is NaN or infinite, and with it every output of the column
//   count  [row groups] u32 and sums [slices][row groups][4 * NX][16] f64, where the row is cut
// The sum of X per sub-block (for the mins) is not stored: the matrix cores form
// sum_j m_j * sum_k digit directly, with the min of a sub-block in all of its B bytes.
// ---------------------------------------------------------------------------
constexpr uint32_t kPThreads = 512;   // a run of 8 activations per thread
constexpr uint32_t kPMaxParts = 4u, kPMaxCols = kPMaxParts * 8u * kPThreads;
__host__ __device__ constexpr size_t q4k_planes_bytes(uint32_t sb, uint32_t nx) { return (size_t)sb * nx * 4096u; }
__host__ __device__ constexpr size_t q4k_count_at(uint32_t sb, uint32_t nx) {
    return q4k_planes_bytes(sb, nx) + (size_t)sb * 4u * nx * 8u;
}
__host__ __device__ constexpr size_t q4k_sums_at(uint32_t sb, uint32_t nx, uint32_t groups) {
    return q4k_count_at(sb, nx) + ((size_t)groups + 1u) / 2u * 8u;
}
__host__ __device__ constexpr size_t q4k_planes_total(uint32_t sb, uint32_t nx, uint32_t groups, uint32_t slices) {
    return slices > 1u ? q4k_sums_at(sb, nx, groups) + (size_t)slices * groups * nx * 512u : q4k_count_at(sb, nx);
}

// grid (ncol, PARTS), PARTS parts of the column of 8 * kPThreads values, the last one shorter: a part is one
// workgroup's to convert (four columns of 12288 by one workgroup each: 6.7 us, 4.1 in three parts), the sum of
// squares every part forms for itself.  cols % 256 == 0; x and gain 16-byte aligned.  nclear: counters to clear.
template <int PARTS>
__global__ void __launch_bounds__(kPThreads)
q4k_planes_kernel(const float *__restrict__ x, const float *__restrict__ gain, float eps, uint8_t *__restrict__ scratch,
                  uint32_t cols, uint32_t nx, double rcols, uint32_t nclear) {
    __shared__ double run[PARTS * kPThreads / 4];
    __shared__ double s_inv;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t c = blockIdx.x, SB = cols >> 8, subs = cols >> 5, NL = 4u * nx;
    uint8_t *planes = scratch;
    double *psb = reinterpret_cast<double *>(scratch + q4k_planes_bytes(SB, nx));
    if (c == 0u && blockIdx.y == 0u)
        for (uint32_t i = tid; i < nclear; i += kPThreads)
            reinterpret_cast<uint32_t *>(scratch + q4k_count_at(SB, nx))[i] = 0u;
    const uint32_t part0 = blockIdx.y * kPThreads, runs = cols >> 3;
    auto load = [&](uint32_t k, lev_f32x4 &a, lev_f32x4 &b) {
        const lev_f32x4 *xp = reinterpret_cast<const lev_f32x4 *>(x + (uint64_t)c * cols) + 2u * (k < runs ? k : 0u);
        a = xp[0], b = xp[1];
    };
    const bool real = part0 + tid < runs;
    const uint32_t k8 = real ? part0 + tid : 0u;
    lev_f32x4 va, vb;
    load(part0 + tid, va, vb);
    if (gain) {
        const lev_f32x4 *gp = reinterpret_cast<const lev_f32x4 *>(gain) + 2u * k8;
        const lev_f32x4 ga = gp[0], gb = gp[1];
        // RMSNorm as the reference computes it (rmsnorm, rust/crates/lev-model/src/lib.rs:110-114):
        // mean square and 1/sqrt in f64, then (f32)(x * inv) * gain; the additions in the order of
        // q4_k_mfma_gemv (a sub-block's four runs, the sub-blocks lane by lane, the lanes)
        lev_f32x4 wa[PARTS], wb[PARTS];
#pragma unroll
        for (int i = 0; i < PARTS; ++i) load((uint32_t)i * kPThreads + tid, wa[i], wb[i]);
#pragma unroll
        for (int i = 0; i < PARTS; ++i) {
            const uint32_t k = (uint32_t)i * kPThreads + tid;
            double ss = (double)wa[i].x * (double)wa[i].x;
            ss = fma((double)wa[i].y, (double)wa[i].y, ss); ss = fma((double)wa[i].z, (double)wa[i].z, ss);
            ss = fma((double)wa[i].w, (double)wa[i].w, ss); ss = fma((double)wb[i].x, (double)wb[i].x, ss);
            ss = fma((double)wb[i].y, (double)wb[i].y, ss); ss = fma((double)wb[i].z, (double)wb[i].z, ss);
            ss = fma((double)wb[i].w, (double)wb[i].w, ss);
            ss = lev_group_sum_f64<4>(ss);
            if (k < runs && (k & 3u) == 3u) run[k >> 2] = ss;
        }
        lev_barrier_lds();
        if (wave == 0u) {
            double tot = 0.0;
            for (uint32_t k = lane; k < subs; k += 64u) tot += run[k];
            tot = lev_group_sum_f64<64>(tot);
            const double a = fma(tot, rcols, (double)eps);
            double rs = __builtin_amdgcn_rsq(a);
            rs = rs * fma(-0.5 * a * rs, rs, 1.5);
            rs = rs * fma(-0.5 * a * rs, rs, 1.5);
            if (lane == 63u) s_inv = rs;
        }
        lev_barrier_lds();
        const double inv = s_inv;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            va[k] = (float)((double)va[k] * inv) * ga[k];
            vb[k] = (float)((double)vb[k] * inv) * gb[k];
        }
    }
    const float v[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
    uint32_t mb = 0u;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t bits = __float_as_uint(v[k]) & 0x7FFFFFFFu;
        mb = bits > mb ? bits : mb;
    }
    mb = lev_row16_max_u32(mb);
    {
        const uint32_t o = (uint32_t)__builtin_amdgcn_ds_swizzle((int)mb, 0x401F);   // lane ^ 16: the superblock's 32 runs
        mb = o > mb ? o : mb;
    }
    uint32_t ex = mb >> 23;
    const bool bad = ex == 255u;
    ex = ex < 25u ? 25u : (ex > 254u ? 254u : ex);
    const float scale = __uint_as_float((278u - ex) << 23);   // 2^(151-ex): |x*scale| < 2^25
    uint32_t dw[4][2];                                        // dw[3] = highest digit
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t Y[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) Y[k] = ((uint32_t)(int)rintf(v[4 * h + k] * scale) + 0x00808080u) ^ 0x00808080u;
        const uint32_t t0 = __builtin_amdgcn_perm(Y[1], Y[0], 0x05010400u);
        const uint32_t t1 = __builtin_amdgcn_perm(Y[1], Y[0], 0x07030602u);
        const uint32_t t2 = __builtin_amdgcn_perm(Y[3], Y[2], 0x05010400u);
        const uint32_t t3 = __builtin_amdgcn_perm(Y[3], Y[2], 0x07030602u);
        dw[0][h] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
        dw[1][h] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
        dw[2][h] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
        dw[3][h] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
    }
    if (real) {
        const uint32_t j = k8 >> 2, kg = k8 & 3u;             // sub-block of the row, k-group
        const uint32_t sb = j >> 3, jp = (j & 7u) >> 1, half = j & 1u, q = c >> 2;
        uint8_t *at = planes + ((((size_t)sb * 4u + jp) * nx + q) * 64u + 16u * kg + 4u * (c & 3u)) * 16u + 8u * half;
#pragma unroll
        for (int p = 0; p < 4; ++p) *reinterpret_cast<lev_u2 *>(at + 16 * p) = lev_u2{dw[3 - p][0], dw[3 - p][1]};
        if ((k8 & 31u) == 31u) psb[sb * NL + c] = bad ? (double)__builtin_nanf("") : __hiloint2double((int)((ex + 872u) << 20), 0);   // 2^(ex-151)
    }
}

// NC: columns staged (1, 2, 4 or 8; >= ncol).  SHORT: no wave has more than
// three tasks (every decode-sized matrix); the kernel is then straight-line
// code, so the wait before each task covers exactly that task's loads and each
// task is multiplied while the next streams in.
// PLANES: the digit planes come from q4k_planes_kernel (`x` then points at its scratch; gain
// and eps are not used): the row, or the workgroup's slice of it (SLICED, blockIdx.y), has at most
// sixteen superblocks, so a wave has one superblock column and keeps its A operands in registers; LDS
// holds the partial sums only.  Rows that are not cut have kernels without the slices' arithmetic: with
// it 12288 x 4096 takes 16.6 us by five columns and 16.7 by eight, without 15.5 and 16.0.
// OWN: rows of at most sixteen superblocks: a wave multiplies one superblock column and makes the digits of that one alone, two
// columns a pass, so no barrier stands between the digits and the products, the operands are kept in registers for
// all row groups and the mins are taken as with PLANES.  12288 x 4096 by four columns 10.6 us a call with the digits of all
// superblocks made by all waves, 9.4 like this; by six 15.4 with the planes made in front, 13.4.  The same integers, the same bits.
template <int NC, bool SHORT, bool PLANES = false, bool SLICED = false, bool OWN = false>
__global__ void __launch_bounds__(kMThreads)
q4_k_mfma_gemv(const uint8_t *__restrict__ w, const float *__restrict__ x,
               const float *__restrict__ gain, float eps, float *__restrict__ y, uint32_t cols,
               uint32_t rows, uint32_t ncol, uint32_t pb, double rcols) {
    constexpr int NX = NC > 4 ? 2 : 1;
    using L = q4k_lds<NX>;
    constexpr uint32_t NL = L::NL;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t SB = cols >> 8, subs = PLANES ? 0u : cols >> 5;
    uint8_t *dig = smem;
    double *sxd = reinterpret_cast<double *>(smem + (OWN ? 512u * subs : L::dig_bytes(subs)));
    double *part = sxd + (OWN ? 0u : (size_t)subs * NL);
    double *psb = part + (size_t)pb * kMWaves * 16u * NL;
    double *s_inv = psb + (size_t)SB * NL;
    uint32_t *s_bad = reinterpret_cast<uint32_t *>(s_inv + NL);
    double *run = reinterpret_cast<double *>(smem);

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;

    // ---- geometry of the weight stream ----
    const uint32_t r = lane & 15u, g = lane >> 4;
    const uint64_t row_bytes = (uint64_t)SB * 144u;
    const uint32_t ngroups = (rows + 15u) >> 4;
    const uint32_t slices = SLICED ? gridDim.y : 1u, per_slice = SLICED ? (SB + slices - 1u) / slices : SB;
    const uint32_t sb0 = SLICED ? blockIdx.y * per_slice : 0u;            // the slice's superblocks
    const uint32_t nsb = SLICED && SB - sb0 < per_slice ? SB - sb0 : per_slice;
    constexpr bool REG = PLANES || OWN;      // A operands in registers
    static_assert(!OWN || (!PLANES && NC % 2 == 0), "a wave's lanes take two columns of its superblock at a time");
    const uint32_t tpr = REG ? 1u : (SB + kMWaves - 1u) / kMWaves;    // tasks per row group and wave
    const uint32_t ntasks = ((ngroups - blockIdx.x + gridDim.x - 1u) / gridDim.x) * tpr;
    // A cursor walks the wave's tasks in order: row group rg (stride gridDim.x),
    // within it superblock wave + 16*t for t < tpr.  A task past the end (or
    // past the wave's last superblock) reads the first bytes of the matrix.
    struct cursor {
        uint32_t k, rg, t;
    };
    auto advance = [&](cursor &c) {
        ++c.k;
        if (++c.t == tpr) {
            c.t = 0;
            c.rg += gridDim.x;
        }
    };
    auto issue = [&](cursor &c, q4k_regs &W) {
        const uint32_t sbw = wave + kMWaves * c.t;
        const bool real = c.k < ntasks && sbw < nsb;
        uint32_t row = c.rg * 16u + r;
        row = row < rows ? row : rows - 1u;
        q4k_issue(w, row_bytes, real ? row : 0u, real ? sb0 + sbw : 0u, real ? g : 0u, W);
        advance(c);
    };
    cursor ci{0u, blockIdx.x, 0u}, cc{0u, blockIdx.x, 0u};
    q4k_regs W0, W1, W2;

    // ---- the planes of this wave's superblock column, from q4k_planes_kernel's scratch ----
    lev_i4 Areg[4][NX];      // [sub-block pair][group of four columns]: A of sub-blocks 2jp (x, y) and 2jp + 1 (z, w)
    double pwreg[NX];        // 2^(e-151) of column 4q + g
    if constexpr (PLANES) {
        const uint8_t *scratch = reinterpret_cast<const uint8_t *>(x);
        const uint32_t sbw = sb0 + (wave < nsb ? wave : nsb - 1u);
        const double *psb_g = reinterpret_cast<const double *>(scratch + q4k_planes_bytes(SB, NX));
#pragma unroll
        for (int jp = 0; jp < 4; ++jp)
#pragma unroll
            for (int q = 0; q < NX; ++q)
                Areg[jp][q] = *reinterpret_cast<const lev_i4 *>(
                    scratch + ((((size_t)sbw * 4u + (uint32_t)jp) * NX + (uint32_t)q) * 64u + lane) * 16u);
#pragma unroll
        for (int q = 0; q < NX; ++q) pwreg[q] = psb_g[sbw * NL + 4u * (uint32_t)q + g];
        if (tid < NL) s_bad[tid] = 0u;                       // (the powers of two carry it)
        issue(ci, W0);
        if constexpr (!SHORT) {
            issue(ci, W1);
            issue(ci, W2);
        }
        lev_barrier_lds();
    }
    if constexpr (!PLANES) {
        // ---- stage the activations ----
        // A thread takes runs of 8 consecutive elements (the 8 k-slots one lane
        // feeds to one MFMA).  Slot q = tid + i*1024: the 32 runs of one superblock
        // of one column sit in 32 adjacent lanes (q % 32), superblocks of the NC
        // columns alternate (q / 32 % NC).  The loads are unconditional (clamped) so
        // that they are in flight together; whole passes beyond the data are skipped.
        constexpr int CH = 4;                                   // slots per thread: NC*cols/8 <= 4096
        constexpr uint32_t kLogNC = NC == 8 ? 3u : NC == 4 ? 2u : NC == 2 ? 1u : 0u;
        const uint32_t total_slots = (cols >> 3) * NC;
        auto slot_of = [&](int i, uint32_t &c, uint32_t &k8) {
            if (OWN) {   // two columns of the wave's superblock a pass
                c = 2u * (uint32_t)i + (lane >> 5);
                k8 = (wave << 5) | (lane & 31u);
                return wave < SB && c < ncol;
            }
            const uint32_t q = tid + (uint32_t)i * kMThreads;
            c = (q >> 5) & (NC - 1u);
            k8 = ((q >> (5u + kLogNC)) << 5) | (q & 31u);
            return q < total_slots && c < ncol;
        };
        auto past = [&](int i) { return OWN ? 2 * i >= NC : (uint32_t)i * kMThreads >= total_slots; };   // workgroup-uniform
        lev_f32x4 va[CH], vb[CH];
        {
            lev_f32x4 ga[CH], gb[CH];
    #pragma unroll
            for (int i = 0; i < CH; ++i) {
                if (past(i)) break;
                uint32_t c, k8;
                if (!slot_of(i, c, k8)) c = 0u, k8 = 0u;
                const lev_f32x4 *xp = reinterpret_cast<const lev_f32x4 *>(x + (uint64_t)c * cols) + 2u * k8;
                va[i] = xp[0];
                vb[i] = xp[1];
                if (OWN && i != 0) continue;   // (one superblock: one set of gains)
                if (OWN) k8 = wave < SB ? (wave << 5) | (lane & 31u) : 0u;   // (also where the first pass has no column)
                const lev_f32x4 *gp = reinterpret_cast<const lev_f32x4 *>(gain ? gain : x) + 2u * k8;
                ga[i] = gp[0];
                gb[i] = gp[1];
            }
            if (tid < NL) s_bad[tid] = 0u;
            // RMSNorm as the reference computes it (rmsnorm, rust/crates/lev-model/src/lib.rs:110-114):
            // mean square and 1/sqrt in f64, then (f32)(x * inv) * gain
            if (gain) {
    #pragma unroll
                for (int i = 0; i < CH; ++i) {
                    if (past(i)) break;
                    uint32_t c, k8;
                    const bool real = slot_of(i, c, k8);
                    const lev_f32x4 a = va[i], b = vb[i];
                    double ss = (double)a.x * (double)a.x;
                    ss = fma((double)a.y, (double)a.y, ss); ss = fma((double)a.z, (double)a.z, ss);
                    ss = fma((double)a.w, (double)a.w, ss); ss = fma((double)b.x, (double)b.x, ss);
                    ss = fma((double)b.y, (double)b.y, ss); ss = fma((double)b.z, (double)b.z, ss);
                    ss = fma((double)b.w, (double)b.w, ss);
                    ss = lev_group_sum_f64<4>(ss);   // the four runs of a sub-block sit in four adjacent lanes
                    if (real && (k8 & 3u) == 3u) run[c * subs + (k8 >> 2)] = ss;
                }
            }
            // every wave of the workgroup has its activations: a CU's memory pipeline is
            // one queue, and weight loads of early waves would hold up the activation
            // loads of late ones.  The first weights stream in while the digits are made.
            lev_barrier_lds();
            issue(ci, W0);
            if constexpr (!SHORT) {
                issue(ci, W1);
                issue(ci, W2);
            }
            if (gain) {
                // one wave per column adds the column's sums of squares
                if (wave < ncol) {
                    double ss = 0.0;
                    for (uint32_t k = lane; k < subs; k += 64u) ss += run[wave * subs + k];
                    ss = lev_group_sum_f64<64>(ss);
                    // 1/sqrt(mean + eps): the hardware estimate and two Newton steps (full f64 accuracy)
                    const double a = fma(ss, rcols, (double)eps);
                    double rs = __builtin_amdgcn_rsq(a);
                    rs = rs * fma(-0.5 * a * rs, rs, 1.5);
                    rs = rs * fma(-0.5 * a * rs, rs, 1.5);
                    if (lane == 63u) s_inv[wave] = rs;
                }
                lev_barrier_lds();   // the sums (in the digit area) are dead from here
    #pragma unroll
                for (int i = 0; i < CH; ++i) {
                    if (past(i)) break;
                    uint32_t c, k8;
                    const bool real = slot_of(i, c, k8);
                    const double inv = s_inv[real ? c : 0u];
    #pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        va[i][k] = (float)((double)va[i][k] * inv) * ga[OWN ? 0 : i][k];
                        vb[i][k] = (float)((double)vb[i][k] * inv) * gb[OWN ? 0 : i][k];
                    }
                }
            }
        }
    #pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (past(i)) break;
            uint32_t c, k8;
            const bool real = slot_of(i, c, k8);
            const lev_f32x4 a = va[i], b = vb[i];
            const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            // largest magnitude of the superblock as an integer: NaN and infinity sort above every number
            uint32_t mb = 0u;
    #pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t bits = __float_as_uint(v[k]) & 0x7FFFFFFFu;
                mb = bits > mb ? bits : mb;
            }
            mb = lev_row16_max_u32(mb);   // all 16 lanes of a row hold the row's maximum
            {
                const uint32_t o = (uint32_t)__builtin_amdgcn_ds_swizzle((int)mb, 0x401F);   // lane ^ 16
                mb = o > mb ? o : mb;
            }
            uint32_t ex = mb >> 23;                             // biased exponent: |x| < 2^(ex-126)
            if (real && ex == 255u) atomicOr(&s_bad[c], 1u);
            ex = ex < 25u ? 25u : (ex > 254u ? 254u : ex);      // keeps both powers of two normal numbers
            const float scale = __uint_as_float((278u - ex) << 23);   // 2^(151-ex): |x*scale| < 2^25
            int sum = 0, X[8];
    #pragma unroll
            for (int k = 0; k < 8; ++k) {
                X[k] = (int)rintf(v[k] * scale);
                sum += X[k];
            }
            // balanced base-256 digits: adding 0x80 to each of the low three bytes carries
            // into the next digit where a byte exceeds 127, and flipping bit 7 subtracts the
            // 0x80 again, so the bytes of (X + 0x808080) ^ 0x808080 read as int8 are the
            // digits.  A 4x4 byte transpose puts digit k of four neighbours into one dword.
            uint32_t dw[4][2];                                  // dw[3] = highest digit
    #pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t Y[4];
    #pragma unroll
                for (int k = 0; k < 4; ++k) Y[k] = ((uint32_t)X[4 * h + k] + 0x00808080u) ^ 0x00808080u;
                const uint32_t t0 = __builtin_amdgcn_perm(Y[1], Y[0], 0x05010400u);   // a0 b0 a1 b1
                const uint32_t t1 = __builtin_amdgcn_perm(Y[1], Y[0], 0x07030602u);   // a2 b2 a3 b3
                const uint32_t t2 = __builtin_amdgcn_perm(Y[3], Y[2], 0x05010400u);   // c0 d0 c1 d1
                const uint32_t t3 = __builtin_amdgcn_perm(Y[3], Y[2], 0x07030602u);   // c2 d2 c3 d3
                dw[0][h] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);                // a0 b0 c0 d0
                dw[1][h] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
                dw[2][h] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
                dw[3][h] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
            }
            if constexpr (!OWN) {
                sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xF, 0xF, true);   // 32 values of at most 2^25
                sum += __builtin_amdgcn_update_dpp(0, sum, 0x4E, 0xF, 0xF, true);
            }
            if (real) {
                const uint32_t j = k8 >> 2, kg = k8 & 3u;       // sub-block, k-group
                // 16-byte unit u = 8*kg + (A row)/2 of the sub-block's 512 bytes, stored at q4k_unit(u, kg, j)
                uint8_t *blk = dig + (OWN ? (size_t)j : (size_t)j * NX + (c >> 2)) * 512u;
                const uint32_t u = 8u * kg + 2u * (c & 3u);
                *reinterpret_cast<lev_u4 *>(blk + q4k_unit(u, kg, j)) = lev_u4{dw[3][0], dw[3][1], dw[2][0], dw[2][1]};
                *reinterpret_cast<lev_u4 *>(blk + q4k_unit(u + 1u, kg, j)) = lev_u4{dw[1][0], dw[1][1], dw[0][0], dw[0][1]};
                if (!OWN && kg == 3u) sxd[((j >> 3) * NL + c) * 8u + (j & 7u)] = (double)sum;
                if ((k8 & 31u) == 31u) psb[(j >> 3) * NL + c] = __hiloint2double((int)((ex + 872u) << 20), 0);   // 2^(ex-151)
            }
            if constexpr (OWN) {
                if ((i & 1) == 0 && 2 * i + 2 < NC) continue;
                // Four columns' digits are there (or the last ones'): into registers, the next four take their place.  LDS
                // runs a wave's accesses in order, the fences only keep the compiler from moving them.
                const int q = i >> 1;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const uint32_t sbw = wave < SB ? wave : SB - 1u;
                const uint8_t *ablk = dig + (size_t)sbw * 8u * 512u;
                const uint32_t aoff = q4k_unit(8u * g + (r >> 1), g, 0u) + 8u * (r & 1u);
#pragma unroll
                for (int jp = 0; jp < 4; ++jp) {
                    const lev_u2 lo = *reinterpret_cast<const lev_u2 *>(ablk + 1024u * jp + aoff),
                                 hi = *reinterpret_cast<const lev_u2 *>(ablk + 1024u * jp + 512u + (aoff ^ 32u));
                    Areg[jp][q] = lev_i4{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
                }
                pwreg[q] = wave < SB ? psb[sbw * NL + 4u * (uint32_t)q + g] : 0.0;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        // columns of the layout beyond ncol hold no data: the lanes that read them
        // only feed outputs that are never stored
        if constexpr (!OWN) lev_barrier_lds();
    }
    // ---- stream the weights ----
    uint32_t *count = reinterpret_cast<uint32_t *>(reinterpret_cast<uint64_t>(x) + q4k_count_at(SB, NX));
    double *sums = reinterpret_cast<double *>(reinterpret_cast<uint64_t>(x) + q4k_sums_at(SB, NX, ngroups));
    double yacc[NX];
#pragma unroll
    for (int q = 0; q < NX; ++q) yacc[q] = 0.0;

    // One task: superblock (wave + 16*t) of the 16 rows of group rg.  After the
    // last task of a row group the waves' partial sums meet in LDS.
    uint32_t parity = 0;
    auto compute = [&](cursor &c, const q4k_regs &W) {
        const uint32_t rg = c.rg, t = c.t;
        const uint32_t sbw = wave + kMWaves * t;
        const bool live = sbw < nsb;
        const uint32_t sb = live ? sbw : nsb - 1u;               // (staged planes: the slice is the row)
        // unpack_scale_min, lev-cpu/src/lib.rs:64-74: the eight scales and the eight mins as bytes
        const uint32_t S0 = W.hdr.y, S1 = W.hdr.z, S2 = W.hdr.w;
        const uint32_t sc_w[2] = {S0 & 0x3F3F3F3Fu, (S2 & 0x0F0F0F0Fu) | ((S0 >> 2) & 0x30303030u)};
        const uint32_t mn_w[2] = {S1 & 0x3F3F3F3Fu, ((S2 >> 4) & 0x0F0F0F0Fu) | ((S1 >> 2) & 0x30303030u)};
        int E[NX][4];
        double acc2[NX];
        lev_d2 SX[NX][4];
        double pw[NX];
        lev_i4 M[NX];            // PLANES: sum_j m_j * (sum of the sub-block's digits), per plane
#pragma unroll
        for (int q = 0; q < NX; ++q) {
            E[q][0] = E[q][1] = E[q][2] = E[q][3] = 0;
            acc2[q] = 0.0;
            M[q] = lev_i4{0, 0, 0, 0};
            if constexpr (REG) {
                pw[q] = pwreg[q];
            } else {
                const uint32_t m = sb * NL + 4u * q + g;
                pw[q] = psb[m];
#pragma unroll
                for (int h = 0; h < 4; ++h) SX[q][h] = *reinterpret_cast<const lev_d2 *>(sxd + m * 8u + 2u * h);
            }
        }
        // lane (r, g) reads A row r, k-group g: unit 8g + r/2, its low or high 8 bytes
        const uint8_t *ablk = dig + (size_t)sb * 8u * NX * 512u;
        const uint32_t aoff = q4k_unit(8u * g + (r >> 1), g, 0u) + 8u * (r & 1u);
        lev_u4 ca = W.a, cb = W.b;
        q4k_exchange(ca);
        q4k_exchange(cb);
        const lev_u2 chunk[4] = {lev_u2{ca.x, ca.y}, lev_u2{ca.z, ca.w}, lev_u2{cb.x, cb.y}, lev_u2{cb.z, cb.w}};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int sc = (int)((sc_w[j >> 2] >> (8 * (j & 3))) & 0xFFu);
            const double mnd = (double)((mn_w[j >> 2] >> (8 * (j & 3))) & 0xFFu);
            lev_u2 wv = chunk[j >> 1];
            if (j & 1) wv >>= 4;
            wv &= 0x0F0F0F0Fu;
            const long B = __builtin_bit_cast(long, wv);
#pragma unroll
            for (int q = 0; q < NX; ++q) {
                long A;
                if constexpr (REG) {
                    const lev_i4 a4 = Areg[j >> 1][q];
                    A = __builtin_bit_cast(long, (j & 1) ? lev_u2{(uint32_t)a4.z, (uint32_t)a4.w} : lev_u2{(uint32_t)a4.x, (uint32_t)a4.y});
                } else {
                    A = *reinterpret_cast<const long *>(ablk + ((size_t)j * NX + q) * 512u + (aoff ^ (32u * (j & 1))));
                }
                const lev_i4 D = __builtin_amdgcn_mfma_i32_16x16x32_i8(A, B, lev_i4{0, 0, 0, 0}, 0, 0, 0);
                // |D| <= 32*15*128 < 2^16, sc < 2^6: eight of the products fit 32 bits with room
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    E[q][p] += __mul24(D[p], sc);
                    asm("" : "+v"(E[q][p]));   // one multiply-add per plane: keeps the sums from being regrouped
                }
                if constexpr (!REG) acc2[q] = fma(mnd, SX[q][j >> 1][j & 1], acc2[q]);
            }
            if constexpr (REG) {
                if (j & 1) {
                    // the mins of sub-blocks j - 1 and j in every B byte of their halves of a 64-deep product:
                    // the sum over the pair of m * (sum of the sub-block's digits), per plane (below 2^21 over
                    // the superblock)
                    const uint32_t mw = mn_w[j >> 2];
                    const uint32_t m0 = __builtin_amdgcn_perm(0u, mw, 0x01010101u * (uint32_t)((j - 1) & 3));
                    const uint32_t m1 = __builtin_amdgcn_perm(0u, mw, 0x01010101u * (uint32_t)(j & 3));
                    const lev_i4 Bm = __builtin_bit_cast(lev_i4, lev_u4{m0, m0, m1, m1});
#pragma unroll
                    for (int q = 0; q < NX; ++q)
                        M[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(Areg[j >> 1][q], Bm, M[q], 0, 0, 0);
                }
            }
        }
        // a task past the wave's last superblock contributes nothing
        const double d = live ? (double)lev_f16_bits_to_f32(W.hdr.x & 0xFFFFu) : 0.0;
        const double dmin = live ? (double)lev_f16_bits_to_f32(W.hdr.x >> 16) : 0.0;
#pragma unroll
        for (int q = 0; q < NX; ++q) {
            // plane 0 is the highest digit (at most 2 in magnitude); each plane is below 2^25
            const double hi = fma((double)E[q][0], 256.0, (double)E[q][1]);
            const double lo = fma((double)E[q][2], 256.0, (double)E[q][3]);
            const double dot = fma(hi, 65536.0, lo);
            if constexpr (REG) {
                const double mhi = fma((double)M[q][0], 256.0, (double)M[q][1]);
                const double mlo = fma((double)M[q][2], 256.0, (double)M[q][3]);
                acc2[q] = fma(mhi, 65536.0, mlo);
            }
            yacc[q] = fma(pw[q], fma(d, dot, -dmin * acc2[q]), yacc[q]);
        }

        if (t + 1u == tpr) {   // workgroup-uniform
            double *pp = part + parity * (kMWaves * 16u * NL);
            parity ^= pb - 1u;
#pragma unroll
            for (int q = 0; q < NX; ++q) {
                pp[(wave * 16u + r) * NL + 4u * q + g] = yacc[q];
                yacc[q] = 0.0;
            }
            lev_barrier_lds();
            if (tid < 16u * NL) {
                const uint32_t col = tid >> 4, rr = tid & 15u, row = rg * 16u + rr;
                double sum = 0.0;
#pragma unroll
                for (int kk = 0; kk < kMWaves; ++kk) {
                    if (SLICED && (uint32_t)kk * LEV_WAVE >= blockDim.x) break;
                    sum += pp[((uint32_t)kk * 16u + rr) * NL + col];
                }
                if (SLICED)
                    __hip_atomic_store(sums + (((uint64_t)blockIdx.y * ngroups + rg) * NL + col) * 16u + rr, sum,
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else if (col < ncol && row < rows)
                    y[(uint64_t)col * rows + row] = s_bad[col] ? __builtin_nanf("") : (float)sum;
            }
            if (pb == 1u) lev_barrier_lds();   // the one buffer is written again by the next group
        }
        advance(c);
    };
    // The slices' sums of the workgroup's row groups: those it is the last to bring are added up.
    auto merge = [&]() {
        if (!SLICED) return;
        lev_publish_wait();
        lev_barrier_lds();                                       // every wave's sums have reached memory
        uint32_t *last = reinterpret_cast<uint32_t *>(part);     // one flag per row group (kMaxMerged fit)
        const uint32_t mine = (ngroups - blockIdx.x + gridDim.x - 1u) / gridDim.x;
        for (uint32_t i = tid; i < mine; i += blockDim.x)
            last[i] = __hip_atomic_fetch_add(count + blockIdx.x + i * gridDim.x, 1u, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT) == slices - 1u;
        lev_barrier_lds();
        for (uint32_t e = tid; e < mine * 16u * NL; e += blockDim.x) {
            const uint32_t i = e / (16u * NL), col = (e >> 4) % NL, rg = blockIdx.x + i * gridDim.x;
            const uint32_t row = rg * 16u + (e & 15u);
            if (!last[i] || col >= ncol || row >= rows) continue;
            double sum = 0.0;
            for (uint32_t sl = 0; sl < slices; ++sl)
                sum += __hip_atomic_load(sums + (((uint64_t)sl * ngroups + rg) * NL + col) * 16u + (e & 15u),
                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            y[(uint64_t)col * rows + row] = s_bad[col] ? __builtin_nanf("") : (float)sum;
        }
    };

    if constexpr (SHORT) {
        // A wave that issues a load while the CU's memory queue is full waits until the
        // queue drains: with all three tasks requested up front the waves sat in those
        // waits while the digits were still to be made, and multiplied nothing until
        // the last byte had arrived.  One task is requested before the digits, the
        // next two each just ahead of the multiply that precedes their use.
        issue(ci, W1);
        __builtin_amdgcn_sched_barrier(0);
        compute(cc, W0);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W2);
        __builtin_amdgcn_sched_barrier(0);
        if (ntasks > 1u) compute(cc, W1);
        if (ntasks > 2u) compute(cc, W2);
        merge();
        return;
    }
    // Three tasks in flight per wave.
    // The scheduling barriers keep a refill's loads behind the compute that
    // frees its registers: hoisted above it they would be younger than the
    // data the compute waits for, and the wait would cover them too.
    while (true) {
        compute(cc, W0);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W0);
        __builtin_amdgcn_sched_barrier(0);
        if (cc.k >= ntasks) break;
        compute(cc, W1);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W1);
        __builtin_amdgcn_sched_barrier(0);
        if (cc.k >= ntasks) break;
        compute(cc, W2);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W2);
        __builtin_amdgcn_sched_barrier(0);
        if (cc.k >= ntasks) break;
    }
    merge();
}

// One or two columns: the same sums with half the matrix-core products and half the
// multiply-adds.  v_mfma_i32_16x16x64_i8 takes 64 codes of 16 rows; lane group g
// (l / 16) supplies the 16 codes of ONE half sub-block -- exactly the 16 bytes it
// loaded (low or high nibbles), so nothing is exchanged between lanes -- and A row
// 4*gs + p holds digit plane p of the elements lane group gs supplies and zeros
// elsewhere: output row 4*gs + p is the plane sum over that half sub-block alone, in
// a lane of the group that holds the sub-block's scale.  (With four columns per MFMA,
// as above, three quarters of the lanes of a one-column launch multiply-add columns
// that do not exist.)  The digit planes take 4 bytes per element and column, so rows
// up to 32768 / NC wide are served.
//   dig  [NC][16*SB groups of 16][4 planes][16 bytes]
//   sx16 [NC][16*SB] i32                                sum of X per group of 16
//   part [pb][wave][16 rows][NC] f64, psb [NC][SB] f64, inv [NC] f64, bad [NC] u32
//   run  [NC][8*SB] f64 (RMSNorm), in the digit area
template <int NC>
struct q4k_narrow_lds {
    static __host__ __device__ size_t dig_bytes(uint32_t cols) { return (size_t)NC * cols * 4u; }
    static __host__ __device__ size_t total(uint32_t cols, uint32_t pb) {
        return dig_bytes(cols) + kNZeroBytes + (size_t)NC * (cols >> 4) * 4u +
               (size_t)pb * kMWaves * 16u * NC * 8u + (size_t)NC * (cols >> 8) * 8u + (size_t)NC * 12u + 8u;
    }
};

template <int NC, bool SHORT>
__global__ void __launch_bounds__(kMThreads)
q4_k_mfma_gemv_narrow(const uint8_t *__restrict__ w, const float *__restrict__ x,
               const float *__restrict__ gain, float eps, float *__restrict__ y, uint32_t cols,
               uint32_t rows, uint32_t ncol, uint32_t pb, double rcols) {
    using L = q4k_narrow_lds<NC>;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t SB = cols >> 8, subs = cols >> 5;
    uint8_t *dig = smem;
    uint8_t *zero = smem + L::dig_bytes(cols);
    double *part = reinterpret_cast<double *>(zero + kNZeroBytes);
    double *psb = part + (size_t)pb * kMWaves * 16u * NC;
    double *s_inv = psb + (size_t)SB * NC;
    int32_t *sx16 = reinterpret_cast<int32_t *>(s_inv + NC);
    uint32_t *s_bad = reinterpret_cast<uint32_t *>(sx16 + (size_t)NC * (cols >> 4));
    double *run = reinterpret_cast<double *>(smem);

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;

    // ---- geometry of the weight stream ----
    const uint32_t r = lane & 15u, g = lane >> 4;
    const uint64_t row_bytes = (uint64_t)SB * 144u;
    const uint32_t ngroups = (rows + 15u) >> 4;
    const uint32_t tpr = (SB + kMWaves - 1u) / kMWaves;    // tasks per row group and wave
    const uint32_t ntasks = ((ngroups - blockIdx.x + gridDim.x - 1u) / gridDim.x) * tpr;
    // A cursor walks the wave's tasks in order: row group rg (stride gridDim.x),
    // within it superblock wave + 16*t for t < tpr.  A task past the end (or
    // past the wave's last superblock) reads the first bytes of the matrix.
    struct cursor {
        uint32_t k, rg, t;
    };
    auto advance = [&](cursor &c) {
        ++c.k;
        if (++c.t == tpr) {
            c.t = 0;
            c.rg += gridDim.x;
        }
    };
    auto issue = [&](cursor &c, q4k_regs &W) {
        const uint32_t sbw = wave + kMWaves * c.t;
        const bool real = c.k < ntasks && sbw < SB;
        uint32_t row = c.rg * 16u + r;
        row = row < rows ? row : rows - 1u;
        q4k_issue(w, row_bytes, real ? row : 0u, real ? sbw : 0u, real ? g : 0u, W);
        advance(c);
    };
    cursor ci{0u, blockIdx.x, 0u}, cc{0u, blockIdx.x, 0u};
    q4k_regs W0, W1, W2;

    // ---- stage the activations ----
    // A thread takes runs of 8 consecutive elements (the 8 k-slots one lane
    // feeds to one MFMA).  Slot q = tid + i*1024: the 32 runs of one superblock
    // of one column sit in 32 adjacent lanes (q % 32), superblocks of the NC
    // columns alternate (q / 32 % NC).  The loads are unconditional (clamped) so
    // that they are in flight together; whole passes beyond the data are skipped.
    constexpr int CH = 4;                                   // slots per thread: NC*cols/8 <= 4096
    constexpr uint32_t kLogNC = NC == 8 ? 3u : NC == 4 ? 2u : NC == 2 ? 1u : 0u;
    const uint32_t total_slots = (cols >> 3) * NC;
    auto slot_of = [&](uint32_t q, uint32_t &c, uint32_t &k8) {
        c = (q >> 5) & (NC - 1u);
        k8 = ((q >> (5u + kLogNC)) << 5) | (q & 31u);
        return q < total_slots && c < ncol;
    };
    lev_f32x4 va[CH], vb[CH];
    {
        lev_f32x4 ga[CH], gb[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if ((uint32_t)i * kMThreads >= total_slots) break;   // workgroup-uniform
            uint32_t c, k8;
            if (!slot_of(tid + (uint32_t)i * kMThreads, c, k8)) c = 0u, k8 = 0u;
            const lev_f32x4 *xp = reinterpret_cast<const lev_f32x4 *>(x + (uint64_t)c * cols) + 2u * k8;
            va[i] = xp[0];
            vb[i] = xp[1];
            const lev_f32x4 *gp = reinterpret_cast<const lev_f32x4 *>(gain ? gain : x) + 2u * k8;
            ga[i] = gp[0];
            gb[i] = gp[1];
        }
        if (tid < (uint32_t)NC) s_bad[tid] = 0u;
        if (tid < kNZeroBytes / 4u) reinterpret_cast<uint32_t *>(zero)[tid] = 0u;
        // RMSNorm as the reference computes it (rmsnorm, rust/crates/lev-model/src/lib.rs:110-114):
        // mean square and 1/sqrt in f64, then (f32)(x * inv) * gain
        if (gain) {
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                if ((uint32_t)i * kMThreads >= total_slots) break;
                uint32_t c, k8;
                const bool real = slot_of(tid + (uint32_t)i * kMThreads, c, k8);
                const lev_f32x4 a = va[i], b = vb[i];
                double ss = (double)a.x * (double)a.x;
                ss = fma((double)a.y, (double)a.y, ss); ss = fma((double)a.z, (double)a.z, ss);
                ss = fma((double)a.w, (double)a.w, ss); ss = fma((double)b.x, (double)b.x, ss);
                ss = fma((double)b.y, (double)b.y, ss); ss = fma((double)b.z, (double)b.z, ss);
                ss = fma((double)b.w, (double)b.w, ss);
                ss = lev_group_sum_f64<4>(ss);   // the four runs of a sub-block sit in four adjacent lanes
                if (real && (k8 & 3u) == 3u) run[c * subs + (k8 >> 2)] = ss;
            }
        }
        // every wave of the workgroup has its activations: a CU's memory pipeline is
        // one queue, and weight loads of early waves would hold up the activation
        // loads of late ones.  The first weights stream in while the digits are made.
        lev_barrier_lds();
        issue(ci, W0);
        if constexpr (!SHORT) {
            issue(ci, W1);
            issue(ci, W2);
        }
        if (gain) {
            // one wave per column adds the column's sums of squares
            if (wave < ncol) {
                double ss = 0.0;
                for (uint32_t k = lane; k < subs; k += 64u) ss += run[wave * subs + k];
                ss = lev_group_sum_f64<64>(ss);
                // 1/sqrt(mean + eps): the hardware estimate and two Newton steps (full f64 accuracy)
                const double a = fma(ss, rcols, (double)eps);
                double rs = __builtin_amdgcn_rsq(a);
                rs = rs * fma(-0.5 * a * rs, rs, 1.5);
                rs = rs * fma(-0.5 * a * rs, rs, 1.5);
                if (lane == 63u) s_inv[wave] = rs;
            }
            lev_barrier_lds();   // the sums (in the digit area) are dead from here
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                if ((uint32_t)i * kMThreads >= total_slots) break;
                uint32_t c, k8;
                const bool real = slot_of(tid + (uint32_t)i * kMThreads, c, k8);
                const double inv = s_inv[real ? c : 0u];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    va[i][k] = (float)((double)va[i][k] * inv) * ga[i][k];
                    vb[i][k] = (float)((double)vb[i][k] * inv) * gb[i][k];
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        if ((uint32_t)i * kMThreads >= total_slots) break;
        uint32_t c, k8;
        const bool real = slot_of(tid + (uint32_t)i * kMThreads, c, k8);
        const lev_f32x4 a = va[i], b = vb[i];
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        // largest magnitude of the superblock as an integer: NaN and infinity sort above every number
        uint32_t mb = 0u;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint32_t bits = __float_as_uint(v[k]) & 0x7FFFFFFFu;
            mb = bits > mb ? bits : mb;
        }
        mb = lev_row16_max_u32(mb);   // all 16 lanes of a row hold the row's maximum
        {
            const uint32_t o = (uint32_t)__builtin_amdgcn_ds_swizzle((int)mb, 0x401F);   // lane ^ 16
            mb = o > mb ? o : mb;
        }
        uint32_t ex = mb >> 23;                             // biased exponent: |x| < 2^(ex-126)
        if (real && ex == 255u) atomicOr(&s_bad[c], 1u);
        ex = ex < 25u ? 25u : (ex > 254u ? 254u : ex);      // keeps both powers of two normal numbers
        const float scale = __uint_as_float((278u - ex) << 23);   // 2^(151-ex): |x*scale| < 2^25
        int sum = 0, X[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            X[k] = (int)rintf(v[k] * scale);
            sum += X[k];
        }
        // balanced base-256 digits: adding 0x80 to each of the low three bytes carries
        // into the next digit where a byte exceeds 127, and flipping bit 7 subtracts the
        // 0x80 again, so the bytes of (X + 0x808080) ^ 0x808080 read as int8 are the
        // digits.  A 4x4 byte transpose puts digit k of four neighbours into one dword.
        uint32_t dw[4][2];                                  // dw[3] = highest digit
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t Y[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) Y[k] = ((uint32_t)X[4 * h + k] + 0x00808080u) ^ 0x00808080u;
            const uint32_t t0 = __builtin_amdgcn_perm(Y[1], Y[0], 0x05010400u);   // a0 b0 a1 b1
            const uint32_t t1 = __builtin_amdgcn_perm(Y[1], Y[0], 0x07030602u);   // a2 b2 a3 b3
            const uint32_t t2 = __builtin_amdgcn_perm(Y[3], Y[2], 0x05010400u);   // c0 d0 c1 d1
            const uint32_t t3 = __builtin_amdgcn_perm(Y[3], Y[2], 0x07030602u);   // c2 d2 c3 d3
            dw[0][h] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);                // a0 b0 c0 d0
            dw[1][h] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
            dw[2][h] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
            dw[3][h] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
        }
        sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xF, 0xF, true);   // the two runs of a group of 16
        if (real) {
            // group of 16 = k8 / 2, this run its low or high 8 bytes of every plane
            uint8_t *at = dig + (size_t)c * cols * 4u + (size_t)(k8 >> 1) * 64u + 8u * (k8 & 1u);
#pragma unroll
            for (int p = 0; p < 4; ++p) *reinterpret_cast<lev_u2 *>(at + 16 * p) = lev_u2{dw[p][0], dw[p][1]};
            if (k8 & 1u) sx16[c * (cols >> 4) + (k8 >> 1)] = sum;
            if ((k8 & 31u) == 31u) psb[c * SB + (k8 >> 5)] = __hiloint2double((int)((ex + 872u) << 20), 0);   // 2^(ex-151)
        }
    }
    // columns of the layout beyond ncol hold no data: the lanes that read them
    // only feed outputs that are never stored
    lev_barrier_lds();

    // ---- stream the weights ----
    double yacc[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) yacc[q] = 0.0;
    // lane (r, g): weight row r; its loads a and b are bytes [16*(g/2), +16) of chunks g%2 and
    // 2 + g%2, i.e. for load i and nibble nb the half g/2 of sub-block 2*(2i + g%2) + nb
    const uint32_t gh = g >> 1, gl = g & 1u;
    const bool feeds = (r >> 2) == g;                       // this lane's A row belongs to its own lane group
    const uint32_t a_lane = (4u * gl + gh) * 64u + 16u * (r & 3u);   // + (8i + 2nb) groups of 64 bytes

    // One task: superblock (wave + 16*t) of the 16 rows of group rg.  After the
    // last task of a row group the waves' partial sums meet in LDS.
    uint32_t parity = 0;
    auto compute = [&](cursor &c, const q4k_regs &W) {
        const uint32_t rg = c.rg, t = c.t;
        const uint32_t sbw = wave + kMWaves * t;
        const bool live = sbw < SB;
        const uint32_t sb = live ? sbw : SB - 1u;
        // unpack_scale_min, lev-cpu/src/lib.rs:64-74: the eight scales and the eight mins as bytes
        const uint32_t S0 = W.hdr.y, S1 = W.hdr.z, S2 = W.hdr.w;
        const uint32_t sc_w[2] = {S0 & 0x3F3F3F3Fu, (S2 & 0x0F0F0F0Fu) | ((S0 >> 2) & 0x30303030u)};
        const uint32_t mn_w[2] = {S1 & 0x3F3F3F3Fu, ((S2 >> 4) & 0x0F0F0F0Fu) | ((S1 >> 2) & 0x30303030u)};
        // sub-block j = 4i + 2*gl + nb: byte 2*gl + nb of word i
        int sc[2][2];
        double mnd[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                sc[i][nb] = (int)__builtin_amdgcn_ubfe(sc_w[i], 16u * gl + 8u * (uint32_t)nb, 8u);
                mnd[i][nb] = (double)__builtin_amdgcn_ubfe(mn_w[i], 16u * gl + 8u * (uint32_t)nb, 8u);
            }
        // B operands: the 16 code bytes as loaded, low or high nibbles
        lev_i4 B[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const lev_u4 v = i ? W.b : W.a;
            B[i][0] = __builtin_bit_cast(lev_i4, v & 0x0F0F0F0Fu);
            B[i][1] = __builtin_bit_cast(lev_i4, (v >> 4) & 0x0F0F0F0Fu);
        }
        // a task past the wave's last superblock contributes nothing
        const double d = live ? (double)lev_f16_bits_to_f32(W.hdr.x & 0xFFFFu) : 0.0;
        const double dmin = live ? (double)lev_f16_bits_to_f32(W.hdr.x >> 16) : 0.0;
        const uint32_t goff = 16u * sb + 4u * gl + gh;        // group of 16 of (i, nb) = (0, 0); + 8i + 2nb
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const uint8_t *ab = feeds ? dig + (size_t)q * cols * 4u + (size_t)sb * 1024u + a_lane : zero;
            const int32_t *sxp = sx16 + (size_t)q * (cols >> 4) + goff;
            int E[4] = {0, 0, 0, 0};
            double acc2 = 0.0;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int nb = 0; nb < 2; ++nb) {
                    const lev_i4 A = *reinterpret_cast<const lev_i4 *>(ab + (8 * i + 2 * nb) * 64);
                    const lev_i4 D = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, B[i][nb], lev_i4{0, 0, 0, 0}, 0, 0, 0);
                    // |D| <= 16*15*128 < 2^15, sc < 2^6: the four products per plane fit 32 bits with room
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        E[p] += __mul24(D[p], sc[i][nb]);
                        asm("" : "+v"(E[p]));   // one multiply-add per plane: keeps the sums from being regrouped
                    }
                    acc2 = fma(mnd[i][nb], (double)sxp[8 * i + 2 * nb], acc2);
                }
            }
            // plane 3 is the highest digit (at most 2 in magnitude)
            const double hi = fma((double)E[3], 256.0, (double)E[2]);
            const double lo = fma((double)E[1], 256.0, (double)E[0]);
            const double dot = fma(hi, 65536.0, lo);
            yacc[q] = fma(psb[q * SB + sb], fma(d, dot, -dmin * acc2), yacc[q]);
        }

        if (t + 1u == tpr) {   // workgroup-uniform
            double *pp = part + parity * (kMWaves * 16u * NC);
            parity ^= pb - 1u;
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                // the four lane groups hold the four quarters of the row's share
                double s = yacc[q];
                s += __shfl_xor(s, 16);
                s += __shfl_xor(s, 32);
                if (g == 0u) pp[(wave * 16u + r) * NC + q] = s;
                yacc[q] = 0.0;
            }
            lev_barrier_lds();
            if (tid < 16u * NC) {
                const uint32_t col = tid >> 4, rr = tid & 15u, row = rg * 16u + rr;
                double sum = 0.0;
#pragma unroll
                for (int kk = 0; kk < kMWaves; ++kk) sum += pp[((uint32_t)kk * 16u + rr) * NC + col];
                if (col < ncol && row < rows)
                    y[(uint64_t)col * rows + row] = s_bad[col] ? __builtin_nanf("") : (float)sum;
            }
            if (pb == 1u) lev_barrier_lds();   // the one buffer is written again by the next group
        }
        advance(c);
    };

    if constexpr (SHORT) {
        // A wave that issues a load while the CU's memory queue is full waits until the
        // queue drains: with all three tasks requested up front the waves sat in those
        // waits while the digits were still to be made, and multiplied nothing until
        // the last byte had arrived.  One task is requested before the digits, the
        // next two each just ahead of the multiply that precedes their use.
        issue(ci, W1);
        __builtin_amdgcn_sched_barrier(0);
        compute(cc, W0);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W2);
        __builtin_amdgcn_sched_barrier(0);
        if (ntasks > 1u) compute(cc, W1);
        if (ntasks > 2u) compute(cc, W2);
        return;
    }
    // Three tasks in flight per wave.
    // The scheduling barriers keep a refill's loads behind the compute that
    // frees its registers: hoisted above it they would be younger than the
    // data the compute waits for, and the wait would cover them too.
    while (true) {
        compute(cc, W0);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W0);
        __builtin_amdgcn_sched_barrier(0);
        if (cc.k >= ntasks) break;
        compute(cc, W1);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W1);
        __builtin_amdgcn_sched_barrier(0);
        if (cc.k >= ntasks) break;
        compute(cc, W2);
        __builtin_amdgcn_sched_barrier(0);
        issue(ci, W2);
        __builtin_amdgcn_sched_barrier(0);
        if (cc.k >= ntasks) break;
    }
}

}  // namespace
uint32_t lev_q4_k_mfma_cols(const lev_ctx *ctx, uint32_t in_dim);
namespace {

size_t q4k_mfma_lds_bytes(uint32_t cols, uint32_t nc, uint32_t pb) {
    return nc > 4u ? q4k_lds<2>::total(cols >> 5, pb) : q4k_lds<1>::total(cols >> 5, pb);
}

size_t q4k_lds_limit(const lev_ctx *ctx) {
    return ctx->props.sharedMemPerBlockOptin > ctx->props.sharedMemPerBlock ? ctx->props.sharedMemPerBlockOptin
                                                                            : ctx->props.sharedMemPerBlock;
}

template <int NC, bool SHORT, bool OWN = false>
hipError_t launch_mfma_variant(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain, float eps,
                       float *y, uint32_t cols, uint32_t rows, uint32_t ncol) {
    constexpr uint32_t NL = NC > 4 ? 8u : 4u;
    const uint32_t pb = OWN || q4k_mfma_lds_bytes(cols, NC, 2u) <= q4k_lds_limit(ctx) ? 2u : 1u;
    const size_t lds = OWN ? (cols >> 5) * 512u + pb * kMWaves * 16u * NL * 8u + (cols >> 8) * NL * 8u + NL * 12u   // 97 KB at most
                           : q4k_mfma_lds_bytes(cols, NC, pb);
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&q4_k_mfma_gemv<NC, SHORT, false, false, OWN>), lds); e != hipSuccess) return e;
    uint32_t groups = (rows + 15u) / 16u;
    uint32_t blocks = groups < (uint32_t)ctx->num_cus ? groups : (uint32_t)ctx->num_cus;
    hipLaunchKernelGGL((q4_k_mfma_gemv<NC, SHORT, false, false, OWN>), dim3(blocks), dim3(kMThreads), lds, ctx->stream, w,
                       x, gain, eps, y, cols, rows, ncol, pb, 1.0 / (double)cols);
    return hipGetLastError();
}

template <int NC>
hipError_t launch_mfma(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain, float eps,
                       float *y, uint32_t cols, uint32_t rows, uint32_t ncol) {
    const uint32_t groups = (rows + 15u) / 16u;
    const uint32_t blocks = groups < (uint32_t)ctx->num_cus ? groups : (uint32_t)ctx->num_cus;
    const uint32_t tpr = ((cols >> 8) + kMWaves - 1u) / kMWaves;
    const uint32_t most = ((groups + blocks - 1u) / blocks) * tpr;   // tasks of the busiest wave
    if (most <= 3u) return launch_mfma_variant<NC, true>(ctx, w, x, gain, eps, y, cols, rows, ncol);
    return launch_mfma_variant<NC, false>(ctx, w, x, gain, eps, y, cols, rows, ncol);
}

template <int NC>
hipError_t launch_own(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain, float eps, float *y, uint32_t cols,
                      uint32_t rows, uint32_t ncol) {
    if constexpr (NC <= 4)
        if ((rows + 15u) / 16u > 3u * (uint32_t)ctx->num_cus) return launch_mfma_variant<NC, false, true>(ctx, w, x, gain, eps, y, cols, rows, ncol);
    return launch_mfma_variant<NC, true, true>(ctx, w, x, gain, eps, y, cols, rows, ncol);
}

// Whether the waves make the digits of their own superblock column each (us, recorded, for what took the shape before and for
// this).  Two columns: always (12288 x 4096 10.3, 9.9; 1491 x 2048 5.5, 5.1).  Three and four: rows of more than eight superblocks (12288
// x 4096 11.6, 10.4; 1200 x 2304 7.0, 6.2); of fewer, half of the waves have none to make and all sixteen make them faster
// together (6000 x 2048 7.06, 7.12, 3677 x 1024 5.6, 5.9).  Five and more, which had the planes made in front: three rounds of
// row groups at most, more have no registers for their weights beside two sets of operands (32768 x 4096 by six 28.5, 38.6); by
// five and six always (12288 x 4096 15.4, 13.4; 500 x 2560 8.5, 7.7), by seven and eight up to eight superblocks and from
// two rounds on (12288 x 4096 15.8, 14.8; 1491 x 2048 9.06, 8.77; but 3000 x 3584 9.6, 10.0).
bool q4k_own_takes(const lev_ctx *ctx, uint32_t cols, uint32_t rows, uint32_t ncol) {
    const uint32_t groups = (rows + 15u) / 16u, cus = (uint32_t)ctx->num_cus;
    if (cols > 256u * kMWaves || ncol < 2u || ncol > 8u) return false;
    if (ncol <= 4u) return ncol == 2u || cols > 2048u;
    return groups <= 3u * cus && (ncol <= 6u || cols <= 2048u || groups > cus);
}

constexpr uint32_t kMaxMerged = 4096u;   // row groups a workgroup can merge: a flag each in the LDS of the partial sums

// Slices of a row, waves of a workgroup (one per superblock of its slice) and workgroups of a slice.  A CU holds sixteen
// waves of this kernel.  Of the fewest slices possible and up to three more: the number with the shortest busiest
// workgroup, a round of row groups counted as its waves on a CU and eight more for its latency (4096 x 12288: three
// slices are 85 workgroups and four rounds of 16 waves, four are 64 and four rounds of 12).
struct q4k_grid {
    uint32_t slices, waves, blocks;
};
q4k_grid q4k_planes_grid(const lev_ctx *ctx, uint32_t cols, uint32_t rows) {
    const uint32_t SB = cols >> 8, groups = (rows + 15u) / 16u, W = (uint32_t)kMWaves, cus = (uint32_t)ctx->num_cus;
    if (SB <= W) return q4k_grid{1u, W, groups < cus ? groups : cus};
    q4k_grid best{};
    uint32_t best_cost = 0xFFFFFFFFu;
    const uint32_t least = (SB + W - 1u) / W;
    for (uint32_t sl = least; sl <= least + 3u; ++sl) {
        const uint32_t waves = (SB + sl - 1u) / sl, per_cu = W / waves, room = cus * per_cu / sl;
        const uint32_t blocks = groups < room ? groups : room > 0u ? room : 1u;
        const uint32_t cost = (groups + blocks - 1u) / blocks * (waves * per_cu + 8u);
        if (cost < best_cost) best_cost = cost, best = q4k_grid{sl, waves, blocks};
    }
    return best;
}

// The planes once per launch (q4k_planes_kernel), then the products.  Returns hipErrorOutOfMemory when the scratch
// cannot be had (no memory, or a program is being recorded and the context's scratch is still too small): the caller then takes
// the kernels that stage for themselves.
template <int NC, bool SHORT>
hipError_t launch_planes_variant(lev_ctx *ctx, const uint8_t *w, const uint8_t *scratch, float *y, uint32_t cols,
                                 uint32_t rows, uint32_t ncol, const q4k_grid &grid) {
    constexpr uint32_t NL = NC > 4 ? 8u : 4u, pb = 2u;
    constexpr size_t part = (size_t)pb * kMWaves * 16u * NL * 8u;
    static_assert(part >= kMaxMerged * 4u, "the flags of the merge lie over the partial sums");
    const size_t lds = part + (size_t)(cols >> 8) * NL * 8u + (size_t)NL * 12u;   // 34 KB at sixteen superblocks
    auto kernel = grid.slices > 1u ? q4_k_mfma_gemv<NC, SHORT, true, true> : q4_k_mfma_gemv<NC, SHORT, true, false>;
    hipLaunchKernelGGL(kernel, dim3(grid.blocks, grid.slices), dim3(grid.waves * LEV_WAVE), lds, ctx->stream, w,
                       reinterpret_cast<const float *>(scratch), static_cast<const float *>(nullptr), 0.f, y, cols, rows, ncol,
                       pb, 0.0);
    return hipGetLastError();
}

// From how many columns the planes are made in front (LEV_Q4K_PLANES: 0 never, 3..8 from that many; built-in 5).
uint32_t q4k_planes_min_cols() {
    static const uint32_t v = [] {
        const char *e = getenv("LEV_Q4K_PLANES");
        const int n = e ? atoi(e) : 5;
        return e && e[0] == '0' ? 0xFFFFFFFFu : (uint32_t)(n < 3 ? 3 : n > 8 ? 8 : n);
    }();
    return v;
}

// Rows of at most sixteen superblocks: from five columns on, where q4k_own_takes leaves them.  Wider ones: as soon as the kernel that stages for itself needs a second
// launch (4352 x 16000, four columns: 19.4 us with it, 21.4 with the planes in front).
bool q4k_planes_serves(const lev_ctx *ctx, uint32_t cols, uint32_t rows, uint32_t ncol) {
    const uint32_t from = q4k_planes_min_cols();
    if (ncol < 3u || ncol > 8u || from > 8u || cols % 256u != 0u || cols == 0u || cols > kPMaxCols) return false;
    if (cols <= 256u * kMWaves) return ncol >= from;
    const q4k_grid grid = q4k_planes_grid(ctx, cols, rows);
    return (ncol >= from || ncol > lev_q4_k_mfma_cols(ctx, cols)) && (rows + 15u) / 16u <= grid.blocks * kMaxMerged;
}

hipError_t launch_planes(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain, float eps, float *y,
                         uint32_t cols, uint32_t rows, uint32_t ncol) {
    const uint32_t SB = cols >> 8, nx = ncol > 4u ? 2u : 1u;
    const uint32_t groups = (rows + 15u) / 16u;
    const q4k_grid grid = q4k_planes_grid(ctx, cols, rows);
    uint8_t *scratch = static_cast<uint8_t *>(lev_scratch(ctx, q4k_planes_total(SB, nx, groups, grid.slices)));
    if (!scratch) return hipErrorOutOfMemory;
    const uint32_t nclear = grid.slices > 1u ? groups : 0u;
    const uint32_t parts = (cols + 8u * kPThreads - 1u) / (8u * kPThreads);
    auto planes = parts == 1u ? q4k_planes_kernel<1> : parts == 2u ? q4k_planes_kernel<2> : parts == 3u ? q4k_planes_kernel<3> : q4k_planes_kernel<4>;
    hipLaunchKernelGGL(planes, dim3(ncol, parts), dim3(kPThreads), 0, ctx->stream, x, gain, eps, scratch, cols, nx,
                       1.0 / (double)cols, nclear);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const bool few = (groups + grid.blocks - 1u) / grid.blocks <= 3u;
    if (nx == 2u)
        return few ? launch_planes_variant<8, true>(ctx, w, scratch, y, cols, rows, ncol, grid)
                   : launch_planes_variant<8, false>(ctx, w, scratch, y, cols, rows, ncol, grid);
    return few ? launch_planes_variant<4, true>(ctx, w, scratch, y, cols, rows, ncol, grid)
               : launch_planes_variant<4, false>(ctx, w, scratch, y, cols, rows, ncol, grid);
}

size_t q4k_narrow_lds_bytes(uint32_t cols, uint32_t nc, uint32_t pb) {
    return nc > 1u ? q4k_narrow_lds<2>::total(cols, pb) : q4k_narrow_lds<1>::total(cols, pb);
}

template <int NC, bool SHORT>
hipError_t launch_narrow_variant(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain, float eps,
                                 float *y, uint32_t cols, uint32_t rows, uint32_t ncol) {
    const uint32_t pb = q4k_narrow_lds_bytes(cols, NC, 2u) <= q4k_lds_limit(ctx) ? 2u : 1u;
    const size_t lds = q4k_narrow_lds_bytes(cols, NC, pb);
    if (hipError_t e = lev_allow_lds(ctx, reinterpret_cast<const void *>(&q4_k_mfma_gemv_narrow<NC, SHORT>), lds); e != hipSuccess) return e;
    const uint32_t groups = (rows + 15u) / 16u;
    const uint32_t blocks = groups < (uint32_t)ctx->num_cus ? groups : (uint32_t)ctx->num_cus;
    hipLaunchKernelGGL((q4_k_mfma_gemv_narrow<NC, SHORT>), dim3(blocks), dim3(kMThreads), lds, ctx->stream, w,
                       x, gain, eps, y, cols, rows, ncol, pb, 1.0 / (double)cols);
    return hipGetLastError();
}

template <int NC>
hipError_t launch_narrow(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain, float eps,
                         float *y, uint32_t cols, uint32_t rows, uint32_t ncol) {
    const uint32_t groups = (rows + 15u) / 16u;
    const uint32_t blocks = groups < (uint32_t)ctx->num_cus ? groups : (uint32_t)ctx->num_cus;
    const uint32_t tpr = ((cols >> 8) + kMWaves - 1u) / kMWaves;
    const uint32_t most = ((groups + blocks - 1u) / blocks) * tpr;   // tasks of the busiest wave
    if (most <= 3u) return launch_narrow_variant<NC, true>(ctx, w, x, gain, eps, y, cols, rows, ncol);
    return launch_narrow_variant<NC, false>(ctx, w, x, gain, eps, y, cols, rows, ncol);
}

}  // namespace

// Columns one launch of the MFMA kernel can take for this in_dim (0: not usable).
uint32_t lev_q4_k_mfma_cols(const lev_ctx *ctx, uint32_t in_dim) {
    if (in_dim % 256u != 0u || in_dim == 0u) return 0;
    uint32_t nc = 8;
    const size_t limit = q4k_lds_limit(ctx);
    while (nc >= 1u && ((uint64_t)nc * in_dim > 32768u || q4k_mfma_lds_bytes(in_dim, nc, 1u) > limit))
        nc >>= 1;
    return nc;
}

// Columns the one- and two-column kernel can take for this in_dim (0: not usable).
uint32_t lev_q4_k_mfma_narrow_cols(const lev_ctx *ctx, uint32_t in_dim) {
    static const bool off = [] {
        const char *e = getenv("LEV_Q4K_NARROW");   // LEV_Q4K_NARROW=0: four columns per product, for comparison
        return e && e[0] == '0';
    }();
    if (off || in_dim % 256u != 0u || in_dim == 0u) return 0;
    const size_t limit = q4k_lds_limit(ctx);
    for (uint32_t nc = 2; nc >= 1u; --nc)
        if ((uint64_t)nc * in_dim <= 32768u && q4k_narrow_lds_bytes(in_dim, nc, 1u) <= limit) return nc;
    return 0;
}

bool lev_q4_k_mfma_one_usable(const uint8_t *w, const float *x, const float *gain, uint32_t in_dim, uint32_t ncol);
hipError_t lev_q4_k_mfma_one_launch(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain, float eps,
                                    float *y, uint32_t in_dim, uint32_t rows, uint32_t ncol);

// Whether up to eight columns go through planes made in front of the products.
bool lev_q4_k_mfma_planes(const lev_ctx *ctx, uint32_t in_dim, uint32_t rows, uint32_t ncol) {
    return q4k_planes_serves(ctx, in_dim, rows, ncol);
}

// ncol <= lev_q4_k_mfma_narrow_cols(ctx, in_dim) (the narrow kernel), ncol <= lev_q4_k_mfma_cols(ctx, in_dim) or
// lev_q4_k_mfma_planes (which may report hipErrorOutOfMemory while recording: nothing enqueued); w 16-byte aligned.
hipError_t lev_q4_k_mfma_gemv_launch(lev_ctx *ctx, const uint8_t *w, const float *x, const float *gain,
                                     float eps, float *y, uint32_t in_dim, uint32_t rows,
                                     uint32_t ncol) {
    // one column of at most sixteen superblocks: a wave per superblock column (q4_k_mfma_gemv_one.hip)
    static const bool one_off = [] {
        const char *e = getenv("LEV_Q4K_ONE");   // LEV_Q4K_ONE=0: the narrow kernel at one column too, for comparison
        return e && e[0] == '0';
    }();
    if (!one_off && lev_q4_k_mfma_one_usable(w, x, gain, in_dim, ncol))
        return lev_q4_k_mfma_one_launch(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
    // one column of a longer row: the narrow kernel (9.1 us against 9.7 at 12288 x 4096); two columns: only where the
    // four-column kernel's planes do not fit (it is the faster of the two there: 9.9 against 10.8 us)
    if (ncol <= lev_q4_k_mfma_narrow_cols(ctx, in_dim) && (ncol == 1u || lev_q4_k_mfma_cols(ctx, in_dim) < ncol)) {
        if (ncol > 1) return launch_narrow<2>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
        return launch_narrow<1>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
    }
    static const bool planes_named = getenv("LEV_Q4K_PLANES") != nullptr;   // (then its line holds)
    if (q4k_own_takes(ctx, in_dim, rows, ncol) && !(planes_named && q4k_planes_serves(ctx, in_dim, rows, ncol))) {
        if (ncol > 6u) return launch_own<8>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
        if (ncol > 4u) return launch_own<6>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
        if (ncol > 2u) return launch_own<4>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
        return launch_own<2>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
    }
    if (q4k_planes_serves(ctx, in_dim, rows, ncol)) {
        const hipError_t e = launch_planes(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
        if (e != hipErrorOutOfMemory || ncol > lev_q4_k_mfma_cols(ctx, in_dim)) return e;
    }
    if (ncol > 4) return launch_mfma<8>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
    if (ncol > 2) return launch_mfma<4>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
    if (ncol > 1) return launch_mfma<2>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
    return launch_mfma<1>(ctx, w, x, gain, eps, y, in_dim, rows, ncol);
}
