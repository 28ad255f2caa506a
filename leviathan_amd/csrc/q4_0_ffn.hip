// The shared expert's FFN of one token in Q4_0 (Gemma4.swift:3742-3773): h = rmsnorm(x) * norm,
// [g | u] = [W_gate h | W_up h], act = gelu_tanh(g) * u, shared = rmsnorm(W_down act) * post.
//
// Called operator by operator it is six launches of which four are the launch floor and little else: at
// 2816 / 2112 18.7 us recorded, 29 us enqueued one by one.  Here three: everything up to act, the down GEMV, the
// norm behind it (8.8 us recorded, 9.3 before the scale of the norms by DPP; enqueued 9.0 to 10.4, the host's pace; recorded
// 0.15 more with the only group's weights requested a second time).  The first kernel has the shape of the MoE gate/up
// kernel: a wave owns one 256-value column task of gate row group i and of up row group i, keeps the operands in registers and
// meets the others in LDS; in front of it every workgroup normalises x for itself (a wave its own 256 values,
// the sum of squares crosses the waves once), with its weights already on their way.
#include "moe_scores_few.hpp"
#include "program_nodes.hpp"
#include "q4_0_mfma.hpp"

hipError_t lev_q4_0_gemv_launch(lev_ctx *ctx, const uint8_t *w, const float *x, float *y, uint32_t in_dim, uint32_t rows, bool narrow);

namespace {

// part of a round: [gate, up][wave][row] f32, two of them
constexpr uint32_t kFfnPart = 2u * 16u * 16u * 4u, kFfnUp = kFfnPart / 2u;
constexpr uint32_t kFfnSums = 3u * 64u;   // three sums of squares of sixteen waves
constexpr size_t ffn_lds(int nw) { return 2u * kFfnPart + kFfnSums + (size_t)nw * (kQ4mTaskArea + kQ4mZeroBytes); }

// The wave's 256 values of x, normalised as lev_hip_rmsnorm does it: squares in f32 per wave, f64 across the waves.
template <int NW>
__device__ __forceinline__ void ffn_normalise(const lev_ffn_args &a, lev_f32x4 &v, const lev_f32x4 &gain, bool live, float *s_ss,
                                              double per, uint32_t wave, uint32_t lane) {
    v = q4m_mask_activations(v, live);
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) ss = fmaf(v[c], v[c], ss);
    ss = lev_wave_sum_broadcast(ss);
    if (lane == 0u) s_ss[wave] = ss;
    lev_barrier_lds();
    v = v * lev_norm_scale(s_ss, NW, per, a.eps);
    if (a.gain) v = v * gain;
    if (!live) v = lev_f32x4{0.f, 0.f, 0.f, 0.f};                 // (an infinite inv made NaNs of the zeros past the end)
}

// x itself where a norm and adds make it: as rmsnorm_adds_kernel and rmsnorm_pair_kernel do, a lane the same four values.
// The first workgroup stores it.
struct ffn_front {
    lev_f32x4 b, gb, a, ga, ad[lev_norm_front::kMost];
    bool live;
    __device__ __forceinline__ void request(const lev_norm_front &f, uint32_t T, uint32_t n4) {
        bool unused;
        b = q4m_load_activations(f.y, T, n4, live);
        if (f.wy) gb = q4m_load_activations(f.wy, T, n4, unused);
        if (f.s) a = q4m_load_activations(f.s, T, n4, unused);
        if (f.s && f.ws) ga = q4m_load_activations(f.ws, T, n4, unused);
#pragma unroll
        for (int m = 0; m < lev_norm_front::kMost; ++m)
            if (m < f.adds.count && m != f.own) ad[m] = q4m_load_activations(f.adds.x[m], T, n4, unused);
    }
    template <int NW>
    __device__ __forceinline__ lev_f32x4 value(const lev_norm_front &f, double per, bool active, float *sums, uint32_t wave, uint32_t lane) {
        b = q4m_mask_activations(b, live && active);
        float sb = 0.f, sa = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) sb = fmaf(b[c], b[c], sb);
        if (f.s) {
            a = q4m_mask_activations(a, live && active);
#pragma unroll
            for (int c = 0; c < 4; ++c) sa = fmaf(a[c], a[c], sa);
            sa = lev_wave_sum_broadcast(sa);
        }
        sb = lev_wave_sum_broadcast(sb);
        if (lane == 0u) sums[wave] = sb, sums[16u + wave] = sa;
        lev_barrier_lds();
        lev_f32x4 o = b * lev_norm_scale(sums, NW, per, f.eps), x = {0.f, 0.f, 0.f, 0.f};
        if (f.wy) o = o * gb;
        if (f.s) {
            x = a * lev_norm_scale(sums + 16, NW, per, f.eps_s);
            if (f.ws) x = x * ga;
        }
#pragma unroll
        for (int m = 0; m < lev_norm_front::kMost; ++m) {
            if (m >= f.adds.count) break;
            const lev_f32x4 v = m == f.own ? x : ad[m];
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = fmaf(f.adds.c[m], v[c], o[c]);
        }
        return o;
    }
};

// NW waves, one per column task (at most 16).  SINGLE: a workgroup has one group of 16 rows, nothing to prefetch.
// grid (row chunks).
template <int NW, bool SINGLE, bool FRONT = false>
__device__ __forceinline__ void ffn_gate_up(const lev_ffn_args &a, uint8_t *smem, const lev_norm_front &front = lev_norm_front{}) {
    float *const s_ss = reinterpret_cast<float *>(smem + 2u * kFfnPart);
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t npairs = a.hidden >> 6, ntask = (npairs + 3u) >> 2, n4 = a.hidden >> 2;
    const bool active = wave < ntask;
    const uint32_t T = active ? wave : ntask - 1u;
    bool live;
    lev_f32x4 v, gain = {1.f, 1.f, 1.f, 1.f};
    ffn_front before;
    if (FRONT) {
        before.request(front, T, n4);
        live = before.live;
    } else {
        v = q4m_load_activations(a.x, T, n4, live);
    }
    if (a.gain) {
        bool unused;
        gain = q4m_load_activations(a.gain, T, n4, unused);
    }
    const uint64_t row_bytes = (uint64_t)npairs * 36u;
    const uint32_t i_begin = blockIdx.x * a.rows_per_block, i_end = min(i_begin + a.rows_per_block, a.inter);
    const uint32_t lrow = lane >> 2;                              // fetch order: lane = 4 * row + pair
    auto issue = [&](uint32_t i0, uint32_t (&G)[9], uint32_t (&U)[9]) {
        uint32_t row = i0 + lrow;
        row = row < i_end ? row : i_end - 1u;
        q4m_load_task_part(a.gate + row * row_bytes, 4u * T, npairs, G);
        q4m_load_task_part(a.up + row * row_bytes, 4u * T, npairs, U);
    };
    __builtin_amdgcn_sched_barrier(0);
    uint32_t Ga[9], Ua[9];
    uint32_t i0 = i_begin;
    issue(i0, Ga, Ua);
    double per = 1.0 / (double)a.hidden;
    lev_pin(per);
    __builtin_amdgcn_sched_barrier(0);

    if (FRONT) {
        v = before.value<NW>(front, per, active, s_ss + 16, wave, lane);
        if (blockIdx.x == 0u && active && live) reinterpret_cast<lev_f32x4 *>(front.out)[64u * T + lane] = v;
    }
    ffn_normalise<NW>(a, v, gain, live && active, s_ss, per, wave, lane);
    if (blockIdx.x == 0u && active && live) reinterpret_cast<lev_f32x4 *>(a.h)[64u * T + lane] = v;

    uint8_t *area = smem + 2u * kFfnPart + kFfnSums + (size_t)wave * (kQ4mTaskArea + kQ4mZeroBytes), *zero = area + kQ4mTaskArea;
    if (lane < kQ4mZeroBytes / 4u) reinterpret_cast<uint32_t *>(zero)[lane] = 0u;
    q4m_operand op;
    q4m_stage_task(v, area, zero, active, op);
    __builtin_amdgcn_sched_barrier(0);

    const uint32_t r16 = lane & 15u, q = lane >> 4;
    uint32_t pw = (wave * 16u + lane) * 4u, pr = (q * 16u + r16) * 4u;
    lev_pin(pw);
    lev_pin(pr);
    while (true) {
        uint32_t Gb[9], Ub[9], W[9];
        const uint32_t next = i0 + 16u;
        if (!SINGLE) issue(next < i_end ? next : i0, Gb, Ub);     // unconditional (clamped)
        q4m_turn_task(Ga, W);
        const float vg = lev_row_sum_f32(q4m_task_dot(W, op));
        q4m_turn_task(Ua, W);
        const float vu = lev_row_sum_f32(q4m_task_dot(W, op));
        if (lane < 16u) {
            *reinterpret_cast<float *>(smem + pw) = vg;
            *reinterpret_cast<float *>(smem + pw + kFfnUp) = vu;
        }
        lev_barrier_lds();
        if (wave == 0u) {
            // lane (r16, q) adds waves q, q + 4, .. of row r16
            const float *pg = reinterpret_cast<const float *>(smem + pr), *pu = reinterpret_cast<const float *>(smem + pr + kFfnUp);
            float g = pg[0], u = pu[0];
            for (int k = 1; k < NW / 4; ++k) {
                g += pg[64 * k];
                u += pu[64 * k];
            }
            g = 0.5f * lev_row_sum_f32(g);
            u = 0.5f * lev_row_sum_f32(u);
            const uint32_t row = i0 + r16;
            if (q == 0u && row < i_end) {
                a.gu[row] = g;
                a.gu[a.inter + row] = u;
                a.act[row] = lev_gelu_up_value(g, u);
            }
        }
        if (SINGLE || next >= i_end) break;
        i0 = next;
        pw ^= kFfnPart;
        pr ^= kFfnPart;
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            Ga[k] = Gb[k];
            Ua[k] = Ub[k];
        }
    }
}

template <int NW, bool SINGLE>
__global__ void __launch_bounds__(NW * LEV_WAVE, NW / 4)
q4_0_ffn_gate_up(lev_ffn_args a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    ffn_gate_up<NW, SINGLE>(a, smem);
}

// The same and, by the workgroups from `gate_blocks` on, the router scores of h, which those normalise for themselves as
// well: NW / 4 experts each (recorded programs).  FRONT: every workgroup makes x for itself, from the norm and adds in front
// of the FFN, which as a launch of their own take 2.7 us and a gap.
template <int NW, bool SINGLE, bool FRONT>
__device__ __forceinline__ void ffn_gate_up_and_scores(const lev_ffn_args &a, const lev_scores_args &r, uint32_t gate_blocks, uint8_t *smem,
                                                       const lev_norm_front &front) {
    if (blockIdx.x < gate_blocks) {
        ffn_gate_up<NW, SINGLE, FRONT>(a, smem, front);
        return;
    }
    float *const s_ss = reinterpret_cast<float *>(smem + 2u * kFfnPart), *const s_h = s_ss + kFfnSums / 4u;
    const uint32_t lane = threadIdx.x & 63u, part = threadIdx.x >> 8;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t n4 = a.hidden >> 2, ntask = (a.hidden + 255u) >> 8, T = wave < ntask ? wave : ntask - 1u;
    bool live, unused;
    lev_f32x4 v, gain = {1.f, 1.f, 1.f, 1.f};
    ffn_front before;
    if (FRONT) {
        before.request(front, T, n4);
        live = before.live;
    } else {
        v = q4m_load_activations(a.x, T, n4, live);
    }
    if (a.gain) gain = q4m_load_activations(a.gain, T, n4, unused);
    double per = 1.0 / (double)a.hidden;
    lev_pin(per);
    if (FRONT) v = before.value<NW>(front, per, wave < ntask, s_ss + 16, wave, lane);
    live = live && wave < ntask;
    ffn_normalise<NW>(a, v, gain, live, s_ss, per, wave, lane);
    if (live) reinterpret_cast<lev_f32x4 *>(s_h)[64u * T + lane] = v;
    lev_barrier_lds();
    moe_score_few(r.wr, s_h, r.scores, r.hidden, r.experts, (blockIdx.x - gate_blocks) * (NW / 4) + part, 0u, threadIdx.x & 255u,
                  reinterpret_cast<double *>(smem) + 4u * part);
}

template <int NW, bool SINGLE>
__global__ void __launch_bounds__(NW * LEV_WAVE, NW / 4)
q4_0_ffn_gate_up_and_scores(lev_ffn_args a, lev_scores_args r, uint32_t gate_blocks) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    ffn_gate_up_and_scores<NW, SINGLE, false>(a, r, gate_blocks, smem, lev_norm_front{});
}
template <int NW, bool SINGLE>
__global__ void __launch_bounds__(NW * LEV_WAVE, NW / 4)
q4_0_ffn_norm_gate_up_and_scores(lev_ffn_args a, lev_scores_args r, uint32_t gate_blocks, lev_norm_front front) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    ffn_gate_up_and_scores<NW, SINGLE, true>(a, r, gate_blocks, smem, front);
}

// Whether the first three stages may run at the same time: every workgroup reads all of x, the norm and its own rows
// of the weights while others already write h, gu and act, which the operators one by one only do when all readers are
// through.  act may be one of the halves of gu, whose value a lane replaces with its own.
bool ffn_apart(const lev_ffn_args &a, size_t gate_bytes, size_t up_bytes) {
    const size_t nh = (size_t)a.hidden * 4u, ni = (size_t)a.inter * 4u;
    const lev_span in[] = {{a.x, nh}, {a.gain, nh}, {a.gate, gate_bytes}, {a.up, up_bytes}};
    const lev_span h(a.h, nh), gu(a.gu, 2u * ni), act(a.act, ni);
    for (const lev_span &i : in)
        if (i.meets(h) || i.meets(gu) || i.meets(act)) return false;
    return !h.meets(gu) && !h.meets(act) && (!act.meets(gu) || a.act == a.gu || a.act == a.gu + a.inter);
}

}  // namespace

extern "C" int lev_hip_shared_expert_ffn_q4_0(lev_ctx *ctx, const float *d_x, const float *d_ffn_norm, const void *d_gate_w,
                                              size_t gate_bytes, const void *d_up_w, size_t up_bytes, const void *d_down_w,
                                              size_t down_bytes, const float *d_post_norm, float eps, float *d_h, float *d_gu,
                                              float *d_act, float *d_shared, uint32_t hidden, uint32_t inter) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_x || !d_h || !d_gu || !d_act || !d_shared)
        return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "shared_expert_ffn: null pointer");
    if (!(eps >= 0.f)) return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "shared_expert_ffn: eps %g", (double)eps);
    lev_geom g;
    int st = lev_check_matvec(ctx, "shared_expert_ffn gate", 32, 18, d_gate_w, gate_bytes, 0, d_h, hidden, hidden, d_gu,
                              (size_t)2 * inter, inter, hidden, inter, &g);
    if (st == LEV_OK)
        st = lev_check_matvec(ctx, "shared_expert_ffn up", 32, 18, d_up_w, up_bytes, 0, d_h, hidden, hidden, d_gu,
                              (size_t)2 * inter, inter, hidden, inter, &g);
    if (st == LEV_OK)
        st = lev_check_matvec(ctx, "shared_expert_ffn down", 32, 18, d_down_w, down_bytes, 0, d_act, inter, inter, d_shared,
                              hidden, hidden, inter, hidden, &g);
    if (st != LEV_OK) return st;
    const uintptr_t al4 = reinterpret_cast<uintptr_t>(d_gate_w) | reinterpret_cast<uintptr_t>(d_up_w);
    const uintptr_t al16 = reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(d_h) | reinterpret_cast<uintptr_t>(d_ffn_norm);
    lev_ffn_args a = {static_cast<const uint8_t *>(d_gate_w), static_cast<const uint8_t *>(d_up_w), d_x, d_ffn_norm, d_h,
                  d_gu, d_act, hidden, inter, 0u, eps};
    // A schedule installed for the gate/up GEMV keeps the operators apart, so that it is the one that runs.
    const bool fused = hidden % 64u == 0u && hidden <= 4096u && (al4 & 3u) == 0u && (al16 & 15u) == 0u &&
                       ffn_apart(a, gate_bytes, up_bytes) && !lev_selected(ctx, LEV_OP_Q4_0_GEMV, hidden, inter, 1);
    if (fused) {
        const uint32_t cus = (uint32_t)ctx->num_cus, per = (inter + 16u * cus - 1u) / (16u * cus);
        const uint32_t rows = per == 1u ? (inter + cus - 1u) / cus : (inter + 16u * cus - 1u) / (16u * cus) * 16u;
        a.rows_per_block = rows;
        const dim3 grid((inter + rows - 1u) / rows);
#define LEV_FFN(NW)                                                                                                    \
    if (rows <= 16u) hipLaunchKernelGGL((q4_0_ffn_gate_up<NW, true>), grid, dim3(NW * LEV_WAVE), ffn_lds(NW), ctx->stream, a); \
    else hipLaunchKernelGGL((q4_0_ffn_gate_up<NW, false>), grid, dim3(NW * LEV_WAVE), ffn_lds(NW), ctx->stream, a)
        if (hidden <= 2048u) { LEV_FFN(8); }
        else if (hidden <= 3072u) { LEV_FFN(12); }
        else { LEV_FFN(16); }
#undef LEV_FFN
        if (ctx->recording) ctx->folded_nodes += 3u;   // norm, gate, up and geluUp are one node
        st = lev_hip_check(ctx, hipGetLastError(), "shared_expert_ffn gate/up launch");
    } else {
        st = lev_hip_rmsnorm(ctx, d_x, d_h, hidden, 1, d_ffn_norm, eps);
        if (st == LEV_OK)
            st = lev_hip_check(ctx, lev_q4_0_gemv_launch(ctx, static_cast<const uint8_t *>(d_gate_w), d_h, d_gu, hidden, inter, false),
                               "shared_expert_ffn gate launch");
        if (st == LEV_OK)
            st = lev_hip_check(ctx, lev_q4_0_gemv_launch(ctx, static_cast<const uint8_t *>(d_up_w), d_h, d_gu + inter, hidden, inter, false),
                               "shared_expert_ffn up launch");
        if (st == LEV_OK) st = lev_hip_gelu_up(ctx, d_gu, d_act, inter);
    }
    if (st == LEV_OK)
        // narrow rows of the down projection on the matrix cores too: as a launch the two kernels are alike (3968 x 1216 12.1 us
        // a call and 10.5, others 0 to 6 %), but the MoE layer's gate/up takes this one along in recorded programs, 94 us and 72
        // for four layers of 1664 / 320 and 1216; the error against 64 bits is less than half (rms 1.9e-7 and 7.4e-8), beside
        // outliers a hundredth (q4_0_mfma.hpp)
        st = lev_hip_check(ctx, lev_q4_0_gemv_launch(ctx, static_cast<const uint8_t *>(d_down_w), d_act, d_shared, inter, hidden, true),
                           "shared_expert_ffn down launch");
    if (st == LEV_OK) st = lev_hip_rmsnorm(ctx, d_shared, d_shared, hidden, 1, d_post_norm, eps);
    return st;
}

// ---- what recorded programs know of the first kernel (program_nodes.hpp) ----
namespace {
// (the FFN's own kernel or the one with scores)
template <int NW, bool SINGLE>
bool with_scores(const void *func, lev_ffn_node *n) {
    void *const both = reinterpret_cast<void *>(&q4_0_ffn_gate_up_and_scores<NW, SINGLE>);
    if (func != reinterpret_cast<const void *>(&q4_0_ffn_gate_up<NW, SINGLE>) && func != both) return false;
    n->with_scores = lev_fused_launch{both, 0u, NW * LEV_WAVE, (uint32_t)ffn_lds(NW)};
    n->with_front = n->with_scores;
    n->with_front.func = reinterpret_cast<void *>(&q4_0_ffn_norm_gate_up_and_scores<NW, SINGLE>);
    return true;
}
}  // namespace

bool lev_ffn_gate_up_node(const void *func, void **args, lev_ffn_node *out) {
    if (!with_scores<8, true>(func, out) && !with_scores<8, false>(func, out) && !with_scores<12, true>(func, out) &&
        !with_scores<12, false>(func, out) && !with_scores<16, true>(func, out) && !with_scores<16, false>(func, out))
        return false;
    const lev_ffn_args &a = out->args = *static_cast<const lev_ffn_args *>(args[0]);
    const size_t nh = 4u * (size_t)a.hidden, ni = 4u * (size_t)a.inter, w = (size_t)a.inter * (a.hidden / 32u) * 18u;
    out->touches = lev_footprint{};
    out->touches.reads[0] = lev_span(a.x, nh);
    out->touches.reads[1] = lev_span(a.gain, nh);
    out->touches.reads[2] = lev_span(a.gate, w);
    out->touches.reads[3] = lev_span(a.up, w);
    out->touches.writes[0] = lev_span(a.h, nh);
    out->touches.writes[1] = lev_span(a.gu, 2u * ni);
    out->touches.writes[2] = lev_span(a.act, ni);
    return true;
}
