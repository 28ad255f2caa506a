// Context, buffers, argument validation and the small elementwise operators
// of the C ABI declared in include/leviathan_hip.h.
#include "lev_common.hpp"
#include "program_nodes.hpp"

#include <cmath>
#include <new>
#include <vector>

// ---------------------------------------------------------------------------
// errors
// ---------------------------------------------------------------------------

int lev_fail(lev_ctx *ctx, int status, const char *fmt, ...) {
    if (ctx) {
        char buf[512];
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(buf, sizeof(buf), fmt, ap);
        va_end(ap);
        ctx->last_error = buf;
    }
    return status;
}

// The runtime keeps a failed call's error until it is fetched, and what fetches it is the check behind the next launch: an
// error that is reported or answered in another way is taken out here, so that it is not the next call's as well.
int lev_hip_check(lev_ctx *ctx, hipError_t err, const char *what) {
    if (err == hipSuccess) return LEV_OK;
    (void)hipGetLastError();
    return lev_fail(ctx, LEV_ERR_COMMAND_FAILED, "%s: %s", what, hipGetErrorString(err));
}

void *lev_scratch(lev_ctx *ctx, size_t bytes) {
    if (bytes <= ctx->scratch_bytes) return ctx->scratch;
    if (ctx->recording) return nullptr;   // no allocation while a program is being recorded
    // Growing replaces the buffer; earlier kernels on the stream may still be
    // using the old one, so drain the stream first.
    if (ctx->scratch) {
        if (ctx->live_programs > 0) {
            // a recorded program may hold this address: keep the memory alive
            ctx->retired_scratch.push_back(ctx->scratch);
        } else {
            if (hipStreamSynchronize(ctx->stream) != hipSuccess) return nullptr;   // (an error that stays: the stream's)
            (void)hipFree(ctx->scratch);
        }
        ctx->scratch = nullptr;
        ctx->scratch_bytes = 0;
    }
    size_t want = (bytes + 0xFFFFFu) & ~(size_t)0xFFFFFu;
    void *p = nullptr;
    if (hipMalloc(&p, want) != hipSuccess) {
        (void)hipGetLastError();   // (most callers do without)
        return nullptr;
    }
    ctx->scratch = p;
    ctx->scratch_bytes = want;
    return p;
}

namespace {
__global__ void __launch_bounds__(256) zero_kernel(uint32_t *p, size_t n) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * 256;
    for (; i < n; i += stride) p[i] = 0u;
}
}  // namespace

hipError_t lev_zero_async(lev_ctx *ctx, void *d_ptr, size_t bytes) {
    size_t n = bytes / 4;
    if (n == 0) return hipSuccess;
    unsigned blocks = (unsigned)((n + 255) / 256);
    if (blocks > 4096u) blocks = 4096u;
    hipLaunchKernelGGL(zero_kernel, dim3(blocks), dim3(256), 0, ctx->stream,
                       static_cast<uint32_t *>(d_ptr), n);
    return hipGetLastError();
}

extern "C" int lev_hip_abi_version(void) { return 2; }

extern "C" const char *lev_hip_status_name(int status) {
    switch (status) {
        case LEV_OK: return "ok";
        case LEV_ERR_BAD_DIMENSIONS: return "badDimensions";
        case LEV_ERR_WRONG_INPUT_COUNT: return "wrongInputCount";
        case LEV_ERR_NON_FINITE_INPUT: return "nonFiniteInput";
        case LEV_ERR_NON_FINITE_SCALE: return "nonFiniteScale";
        case LEV_ERR_NON_FINITE_OUTPUT: return "nonFiniteOutput";
        case LEV_ERR_EXCEEDS_MODEL_WORKLOAD: return "exceedsModelWorkload";
        case LEV_ERR_INTEGER_OVERFLOW: return "integerOverflow";
        case LEV_ERR_DEVICE_UNAVAILABLE: return "deviceUnavailable";
        case LEV_ERR_KERNEL_LOAD_FAILED: return "kernelLoadFailed";
        case LEV_ERR_FUNCTION_MISSING: return "functionMissing";
        case LEV_ERR_COMMAND_FAILED: return "commandFailed";
        case LEV_ERR_EXCEEDS_MAX_BUFFER_LENGTH: return "exceedsMaxBufferLength";
        case LEV_ERR_EXCEEDS_WORKING_SET: return "exceedsWorkingSet";
        case LEV_ERR_INVALID_ARGUMENT: return "invalidArgument";
        default: return "unknown";
    }
}

// ---------------------------------------------------------------------------
// context + buffers
// ---------------------------------------------------------------------------

extern "C" int lev_hip_ctx_create(int device, void *stream, lev_ctx **out) {
    if (!out) return LEV_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0 || device < 0 || device >= count)
        return LEV_ERR_DEVICE_UNAVAILABLE;
    if (hipSetDevice(device) != hipSuccess) return LEV_ERR_DEVICE_UNAVAILABLE;
    lev_ctx *ctx = new (std::nothrow) lev_ctx();
    if (!ctx) return LEV_ERR_DEVICE_UNAVAILABLE;
    ctx->device = device;
    if (hipGetDeviceProperties(&ctx->props, device) != hipSuccess) {
        delete ctx;
        return LEV_ERR_DEVICE_UNAVAILABLE;
    }
    // This library carries gfx950 code objects only.
    if (std::strncmp(ctx->props.gcnArchName, "gfx950", 6) != 0) {
        delete ctx;
        return LEV_ERR_KERNEL_LOAD_FAILED;
    }
    ctx->num_cus = ctx->props.multiProcessorCount;
    if (stream != LEV_HIP_OWN_STREAM) {
        ctx->stream = static_cast<hipStream_t>(stream);
    } else {
        if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess) {
            delete ctx;
            return LEV_ERR_DEVICE_UNAVAILABLE;
        }
        ctx->owns_stream = true;
    }
    if (hipMalloc(&ctx->argmax_partials, (size_t)lev_ctx::kArgmaxPartials * 16u) != hipSuccess ||
        hipMalloc(reinterpret_cast<void **>(&ctx->d_flag), lev_ctx::kFlagWords * sizeof(int)) != hipSuccess ||
        hipHostMalloc(reinterpret_cast<void **>(&ctx->h_flag), sizeof(int), hipHostMallocDefault) !=
            hipSuccess ||
        hipMemset(ctx->d_flag, 0, lev_ctx::kFlagWords * sizeof(int)) != hipSuccess) {
        lev_hip_ctx_destroy(ctx);
        return LEV_ERR_DEVICE_UNAVAILABLE;
    }
    *ctx->h_flag = 0;
    if (lev_moe_static_scratch_init(ctx) != LEV_OK) {
        lev_hip_ctx_destroy(ctx);
        return LEV_ERR_KERNEL_LOAD_FAILED;
    }
    *out = ctx;
    return LEV_OK;
}

extern "C" int lev_hip_ctx_destroy(lev_ctx *ctx) {
    if (!ctx) return LEV_OK;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    if (ctx->scratch) (void)hipFree(ctx->scratch);
    for (void *p : ctx->retired_scratch) (void)hipFree(p);
    if (ctx->argmax_partials) (void)hipFree(ctx->argmax_partials);
    if (ctx->d_flag) (void)hipFree(ctx->d_flag);
    if (ctx->h_flag) (void)hipHostFree(ctx->h_flag);
    if (ctx->owns_stream && ctx->stream) (void)hipStreamDestroy(ctx->stream);
    (void)hipGetLastError();   // (also what ended ctx_create)
    delete ctx;
    return LEV_OK;
}

extern "C" int lev_hip_sync(lev_ctx *ctx) {
    LEV_REQUIRE_CTX(ctx);
    if (ctx->recording) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "sync while recording a program");
    LEV_HIP(ctx, hipMemcpyAsync(ctx->h_flag, ctx->d_flag, sizeof(int), hipMemcpyDeviceToHost,
                                ctx->stream));
    LEV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (*ctx->h_flag != 0) {
        int flag = *ctx->h_flag;
        *ctx->h_flag = 0;
        LEV_HIP(ctx, lev_zero_async(ctx, ctx->d_flag, sizeof(int)));
        LEV_HIP(ctx, hipStreamSynchronize(ctx->stream));
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS,
                        "a kernel rejected device-resident arguments (code %d; bit 0: expert ids must be "
                        "distinct and below the expert count, bit 1: non-finite router score, bit 2: token id "
                        "beyond the embedding table)",
                        flag);
    }
    return LEV_OK;
}

extern "C" const char *lev_hip_last_error(lev_ctx *ctx) {
    return ctx ? ctx->last_error.c_str() : "null context";
}

extern "C" int lev_hip_device_name(lev_ctx *ctx, char *out, size_t cap) {
    LEV_REQUIRE_CTX(ctx);
    if (!out || cap == 0) return LEV_ERR_INVALID_ARGUMENT;
    std::snprintf(out, cap, "%s (%s)", ctx->props.name, ctx->props.gcnArchName);
    return LEV_OK;
}

extern "C" int lev_hip_buf_alloc(lev_ctx *ctx, size_t bytes, void **d_out) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_out) return LEV_ERR_INVALID_ARGUMENT;
    *d_out = nullptr;
    if (bytes == 0) return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "buf_alloc of 0 bytes");
    if (bytes > ctx->props.totalGlobalMem)
        return lev_fail(ctx, LEV_ERR_EXCEEDS_MAX_BUFFER_LENGTH, "buf_alloc %zu bytes > device %zu",
                        bytes, (size_t)ctx->props.totalGlobalMem);
    hipError_t e = hipMalloc(d_out, bytes);
    const int st = lev_hip_check(ctx, e, "hipMalloc");
    if (e == hipErrorOutOfMemory)
        return lev_fail(ctx, LEV_ERR_EXCEEDS_WORKING_SET, "buf_alloc %zu bytes: out of memory", bytes);
    return st;
}

extern "C" int lev_hip_buf_free(lev_ctx *ctx, void *d_ptr) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_ptr) return LEV_OK;
    LEV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return lev_hip_check(ctx, hipFree(d_ptr), "hipFree");
}

extern "C" int lev_hip_buf_upload(lev_ctx *ctx, void *d_dst, const void *host_src, size_t bytes) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_dst || !host_src) return LEV_ERR_INVALID_ARGUMENT;
    LEV_HIP(ctx, hipMemcpyAsync(d_dst, host_src, bytes, hipMemcpyHostToDevice, ctx->stream));
    return lev_hip_check(ctx, hipStreamSynchronize(ctx->stream), "upload");
}

extern "C" int lev_hip_buf_download(lev_ctx *ctx, void *host_dst, const void *d_src, size_t bytes) {
    LEV_REQUIRE_CTX(ctx);
    if (!host_dst || !d_src) return LEV_ERR_INVALID_ARGUMENT;
    LEV_HIP(ctx, hipMemcpyAsync(host_dst, d_src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    return lev_hip_check(ctx, hipStreamSynchronize(ctx->stream), "download");
}

// ---------------------------------------------------------------------------
// shared geometry validation
// ---------------------------------------------------------------------------

int lev_check_matvec(lev_ctx *ctx, const char *op, uint32_t block_values, uint32_t block_bytes,
                     const void *d_w, size_t w_bytes, uint64_t w_off, const void *d_x,
                     size_t x_count, uint64_t x_needed, const void *d_y, size_t y_capacity,
                     uint64_t y_needed, uint64_t in_dim, uint64_t out_rows, lev_geom *g) {
    if (!d_w || !d_x || !d_y) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "%s: null pointer", op);
    if (in_dim == 0 || out_rows == 0 || in_dim % block_values != 0 ||
        in_dim > LEV_MAX_Q4_INPUT_DIM || out_rows > LEV_MAX_Q4_OUTPUT_DIM)
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "%s: inDim %llu, outDim %llu", op,
                        (unsigned long long)in_dim, (unsigned long long)out_rows);
    g->blocks_per_row = in_dim / block_values;
    uint64_t row_bytes, weight_bytes, w_end;
    if (__builtin_mul_overflow(g->blocks_per_row, (uint64_t)block_bytes, &row_bytes) ||
        __builtin_mul_overflow(out_rows, row_bytes, &weight_bytes) ||
        __builtin_add_overflow(w_off, weight_bytes, &w_end))
        return lev_fail(ctx, LEV_ERR_INTEGER_OVERFLOW, "%s: weight extent overflows", op);
    if (weight_bytes > LEV_MAX_Q4_WEIGHT_BYTES)
        return lev_fail(ctx, LEV_ERR_EXCEEDS_MODEL_WORKLOAD, "%s: %llu weight bytes", op,
                        (unsigned long long)weight_bytes);
    if (w_end > w_bytes)
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS,
                        "%s: weight bytes [%llu, %llu) beyond buffer extent %zu", op,
                        (unsigned long long)w_off, (unsigned long long)w_end, w_bytes);
    if (x_count != x_needed)
        return lev_fail(ctx, LEV_ERR_WRONG_INPUT_COUNT, "%s: input %zu, expected %llu", op, x_count,
                        (unsigned long long)x_needed);
    if (y_capacity < y_needed)
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "%s: y holds %zu floats, needs %llu", op,
                        y_capacity, (unsigned long long)y_needed);
    g->row_bytes = row_bytes;
    g->weight_bytes = weight_bytes;
    return LEV_OK;
}

// ---------------------------------------------------------------------------
// elementwise operators
// ---------------------------------------------------------------------------

namespace {

using norm_adds = lev_norm_adds;

// One workgroup of up to 16 waves per vector.  Sum of squares in f32 per lane, wave DPP sums, f64 across
// waves; y = x * inv * w.  A call on one vector is latency and nothing else (11 KB at n = 2816), so the
// vector and the gains are requested together, 16 bytes a lane, and x stays in registers between the two
// passes: one memory round trip.  V = 16-byte pieces a lane holds; V = 0 takes any length and alignment,
// a float at a time, and reads x twice.  Measured in a recorded chain of 56 operators with three of these a
// layer: 276 us with 256 threads that read x twice and the library's 1 / sqrt in f64, 189 with this.
template <int V, bool ADDS>
__device__ __forceinline__ void rmsnorm_vector(const float *__restrict__ x, float *__restrict__ y, const float *__restrict__ w,
                                               uint32_t n, float eps, const norm_adds &adds) {
    __shared__ float part[16];
    const uint32_t t = threadIdx.x, nt = blockDim.x, n4 = n >> 2;
    const float *xv = x + (uint64_t)blockIdx.x * n;
    float *yv = y + (uint64_t)blockIdx.x * n;
    const lev_f32x4 *x4 = reinterpret_cast<const lev_f32x4 *>(xv), *w4 = reinterpret_cast<const lev_f32x4 *>(w);
    constexpr int R = V ? V : 1;
    lev_f32x4 v[R], g[R], ad[norm_adds::kMost][R];
    double per = 1.0 / (double)n;
    float ss = 0.f;
    if (V) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t i = t + nt * k;
            v[k] = i < n4 ? x4[i] : lev_f32x4{0.f, 0.f, 0.f, 0.f};
        }
        if (w) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t i = t + nt * k;
                g[k] = w4[i < n4 ? i : 0u];
            }
        }
        if (ADDS) {
#pragma unroll
            for (int a = 0; a < norm_adds::kMost; ++a) {
                if (a >= adds.count) break;
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    const uint32_t i = t + nt * k;
                    ad[a][k] = reinterpret_cast<const lev_f32x4 *>(adds.x[a])[i < n4 ? i : 0u];
                }
            }
        }
        lev_pin(per);
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int c = 0; c < 4; ++c) ss = fmaf(v[k][c], v[k][c], ss);
    } else {
        for (uint32_t i = t; i < n; i += nt) {
            const float f = xv[i];
            ss = fmaf(f, f, ss);
        }
    }
    ss = lev_wave_sum_broadcast(ss);
    if ((t & 63u) == 0u) part[t >> 6] = ss;
    lev_barrier_lds();   // (the gains may still be on their way)
    const float inv = lev_norm_scale(part, nt >> 6, per, eps);
    if (V) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t i = t + nt * k;
            lev_f32x4 o = v[k] * inv;
            if (w) o = o * g[k];
            if (ADDS) {
#pragma unroll
                for (int a = 0; a < norm_adds::kMost; ++a) {
                    if (a >= adds.count) break;
#pragma unroll
                    for (int c = 0; c < 4; ++c) o[c] = fmaf(adds.c[a], ad[a][k][c], o[c]);
                }
            }
            if (i < n4) reinterpret_cast<lev_f32x4 *>(yv)[i] = o;
        }
    } else {
        for (uint32_t i = t; i < n; i += nt) {
            const float f = xv[i] * inv;
            yv[i] = w ? f * w[i] : f;
        }
    }
}

template <int V>
__global__ void __launch_bounds__(1024)
rmsnorm_kernel(const float *__restrict__ x, float *__restrict__ y, const float *__restrict__ w, uint32_t n, float eps) {
    rmsnorm_vector<V, false>(x, y, w, n, eps, norm_adds{});
}

template <int V>
__global__ void __launch_bounds__(1024)
rmsnorm_adds_kernel(const float *__restrict__ x, float *__restrict__ y, const float *__restrict__ w, uint32_t n, float eps,
                    norm_adds adds) {
    rmsnorm_vector<V, true>(x, y, w, n, eps, adds);
}

// Two norms of one length in one launch: x = rmsnorm(x) * wx in place, then what rmsnorm_adds_kernel does with y, of whose
// addends number `own` is that x (see pair_norms).  One memory round trip for both.  A piece of four values a lane: the length is
// the width of a MoE layer whose kernels pair_norms knows, 4096 at most.
struct norm_pair {
    float *x;
    const float *wx;
    float eps;
    int own;
};
__global__ void __launch_bounds__(1024)
rmsnorm_pair_kernel(norm_pair p, const float *__restrict__ y, float *__restrict__ out, const float *__restrict__ wy, uint32_t n, float eps,
                    norm_adds adds) {
    __shared__ float part[2][16];
    const uint32_t t = threadIdx.x, nt = blockDim.x, n4 = n >> 2, i = t < n4 ? t : 0u;
    auto vec = [](const float *q) { return reinterpret_cast<const lev_f32x4 *>(q); };
    lev_f32x4 ga, gb, ad[norm_adds::kMost];
    const lev_f32x4 a = t < n4 ? vec(p.x)[t] : lev_f32x4{0.f, 0.f, 0.f, 0.f};
    const lev_f32x4 b = t < n4 ? vec(y)[t] : lev_f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.wx) ga = vec(p.wx)[i];
    if (wy) gb = vec(wy)[i];
#pragma unroll
    for (int m = 0; m < norm_adds::kMost; ++m)
        if (m < adds.count && m != p.own) ad[m] = vec(adds.x[m])[i];
    double per = 1.0 / (double)n;
    lev_pin(per);
    float sa = 0.f, sb = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        sa = fmaf(a[c], a[c], sa);
        sb = fmaf(b[c], b[c], sb);
    }
    sa = lev_wave_sum_broadcast(sa);
    sb = lev_wave_sum_broadcast(sb);
    if ((t & 63u) == 0u) part[0][t >> 6] = sa, part[1][t >> 6] = sb;
    lev_barrier_lds();   // (gains and addends may still be on their way)
    const float ia = lev_norm_scale(part[0], nt >> 6, per, p.eps), ib = lev_norm_scale(part[1], nt >> 6, per, eps);
    lev_f32x4 x = a * ia, o = b * ib;
    if (p.wx) x = x * ga;
    if (wy) o = o * gb;
#pragma unroll
    for (int m = 0; m < norm_adds::kMost; ++m) {
        if (m >= adds.count) break;
        const lev_f32x4 v = m == p.own ? x : ad[m];
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = fmaf(adds.c[m], v[c], o[c]);
    }
    if (t < n4) {
        reinterpret_cast<lev_f32x4 *>(p.x)[t] = x;
        reinterpret_cast<lev_f32x4 *>(out)[t] = o;
    }
}

__global__ void __launch_bounds__(256)
gelu_up_kernel(const float *__restrict__ gu, float *__restrict__ y, uint32_t n) {
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = lev_gelu_up_value(gu[i], gu[n + i]);
}

__global__ void __launch_bounds__(256)
axpy_kernel(const float *__restrict__ x, float *__restrict__ y, float c, uint32_t n) {
    uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = fmaf(c, x[i], y[i]);
}

__global__ void __launch_bounds__(256)
f32_to_f16_kernel(const float *__restrict__ x, uint16_t *__restrict__ out, size_t n) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = __builtin_bit_cast(uint16_t, (_Float16)x[i]);
}

}  // namespace

extern "C" int lev_hip_rmsnorm(lev_ctx *ctx, const float *d_x, float *d_y, uint32_t n,
                               uint32_t vectors, const float *d_weight, float eps) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_x || !d_y) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "rmsnorm: null pointer");
    if (n == 0 || vectors == 0 || !(eps >= 0.f))
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "rmsnorm: n %u, vectors %u, eps %g", n, vectors,
                        (double)eps);
    const bool vec = n % 4u == 0u && n <= 16384u &&
                     ((reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(d_y) |
                       reinterpret_cast<uintptr_t>(d_weight)) & 15u) == 0u;
    // as many waves as the vector fills with one 16-byte piece a lane: they all request at once
    const uint32_t pieces = vec ? (n / 4u + 63u) / 64u : 16u, threads = 64u * (pieces < 16u ? pieces : 16u);
#define LEV_RMS(V) \
    hipLaunchKernelGGL((rmsnorm_kernel<V>), dim3(vectors), dim3(threads), 0, ctx->stream, d_x, d_y, d_weight, n, eps)
    if (!vec) LEV_RMS(0);
    else if (pieces <= 16u) LEV_RMS(1);
    else if (pieces <= 32u) LEV_RMS(2);
    else LEV_RMS(4);
#undef LEV_RMS
    return lev_hip_check(ctx, hipGetLastError(), "rmsnorm launch");
}

extern "C" int lev_hip_gelu_up(lev_ctx *ctx, const float *d_gu, float *d_y, uint32_t n) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_gu || !d_y) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "gelu_up: null pointer");
    if (n == 0) return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "gelu_up: n 0");
    hipLaunchKernelGGL(gelu_up_kernel, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, d_gu, d_y, n);
    return lev_hip_check(ctx, hipGetLastError(), "gelu_up launch");
}

extern "C" int lev_hip_axpy(lev_ctx *ctx, const float *d_x, float *d_y, float c, uint32_t n) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_x || !d_y) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "axpy: null pointer");
    if (n == 0) return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "axpy: n 0");
    if (!std::isfinite(c)) return lev_fail(ctx, LEV_ERR_NON_FINITE_INPUT, "axpy: coefficient");
    hipLaunchKernelGGL(axpy_kernel, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, d_x, d_y, c, n);
    return lev_hip_check(ctx, hipGetLastError(), "axpy launch");
}

extern "C" int lev_hip_f32_to_f16(lev_ctx *ctx, const float *d_x, uint16_t *d_out, size_t n) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_x || !d_out) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "f32_to_f16: null pointer");
    if (n == 0 || n > ((size_t)1 << 40)) return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "f32_to_f16: n");
    hipLaunchKernelGGL(f32_to_f16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       ctx->stream, d_x, d_out, n);
    return lev_hip_check(ctx, hipGetLastError(), "f32_to_f16 launch");
}

// ---------------------------------------------------------------------------
// streaming-read probe: what a plain 128-bit read loop achieves on this
// device, stated next to the nominal HBM peak (the reference's `vk-bw`
// command, rust/crates/lev-cli/src/main.rs:1876-1935).
// ---------------------------------------------------------------------------

namespace {

__global__ void __launch_bounds__(256)
stream_read_kernel(const lev_u32x4 *__restrict__ src, uint64_t n16, uint32_t *__restrict__ sink) {
    uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    lev_u32x4 a = {0, 0, 0, 0}, b = {0, 0, 0, 0}, c = {0, 0, 0, 0}, d = {0, 0, 0, 0};
    for (; i + 3 * stride < n16; i += 4 * stride) {
        lev_u32x4 v0 = src[i], v1 = src[i + stride], v2 = src[i + 2 * stride],
                  v3 = src[i + 3 * stride];
        a ^= v0;
        b ^= v1;
        c ^= v2;
        d ^= v3;
    }
    for (; i < n16; i += stride) a ^= src[i];
    a ^= b ^ c ^ d;
    uint32_t r = a.x ^ a.y ^ a.z ^ a.w;
    if (r == 0x9E3779B9u) sink[0] = r;   // practically never: keeps the loads alive
}

__global__ void empty_kernel() {}

}  // namespace

extern "C" int lev_hip_stream_read_probe(lev_ctx *ctx, const void *d_src, size_t bytes,
                                         uint32_t *d_sink, uint32_t workgroups) {
    LEV_REQUIRE_CTX(ctx);
    if (!d_src || !d_sink) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "probe: null pointer");
    if (bytes < 16 || (reinterpret_cast<uintptr_t>(d_src) & 15u))
        return lev_fail(ctx, LEV_ERR_BAD_DIMENSIONS, "probe: needs >= 16 bytes, 16-byte aligned");
    if (workgroups == 0) workgroups = (uint32_t)ctx->num_cus * 8u;
    hipLaunchKernelGGL(stream_read_kernel, dim3(workgroups), dim3(256), 0, ctx->stream,
                       static_cast<const lev_u32x4 *>(d_src), (uint64_t)(bytes / 16), d_sink);
    return lev_hip_check(ctx, hipGetLastError(), "probe launch");
}

extern "C" int lev_hip_empty_launch(lev_ctx *ctx) {
    LEV_REQUIRE_CTX(ctx);
    hipLaunchKernelGGL(empty_kernel, dim3(1), dim3(64), 0, ctx->stream);
    return lev_hip_check(ctx, hipGetLastError(), "empty launch");
}

// ---------------------------------------------------------------------------
// recorded programs: record once, replay (Program / Step of
// rust/crates/lev-vulkan/src/engine.rs:94-141; the deferred segment of
// Gemma4.swift:2313-2376).  A program is a HIP graph captured from the
// context's stream.
// ---------------------------------------------------------------------------

namespace {

// Operators of a recorded program that one kernel does as well: an RMSNorm of one vector and the axpys right behind it
// that add to its result (a layer's norm and residuals).  A launch of its own costs such an operator some 2 us at any
// size.  Taken: kernel nodes with one dependency and one dependent each, so that nothing else sees the intermediate
// values; an addend that does not overlap the result.  The same values, rounded at the same places.  Anything this
// cannot see through stays as it was recorded.  Recorded decode step of four layers at 2816: 135 us with
// the operators at the end of a layer apart, 123 with this; seven kernels a layer.
// Three more rules look through the shared expert and the MoE layer behind it, whose kernels otherwise run one after the other
// although they share only the normalised input and the sum at the end (weave_shared_expert, pair_norms), and through the
// norm and residuals in front of an FFN (front_norms).  Four kernels a layer and three for the next, 115 us and 89 for the same
// four layers (weights of two such states in turn; 92 with the norms apart, 100 where the launches of the middle do not fit the
// chip together).  1.15 to 1.56 times as fast over 26 drawn ones.
struct node_view {
    const void *func;
    void **args;
    hipKernelNodeParams params;
};
bool kernel_node(hipGraphNode_t node, node_view *out) {
    hipGraphNodeType type;
    if (hipGraphNodeGetType(node, &type) != hipSuccess || type != hipGraphNodeTypeKernel) return false;
    if (hipGraphKernelNodeGetParams(node, &out->params) != hipSuccess) return false;
    out->func = out->params.func;
    out->args = out->params.kernelParams;
    return out->args != nullptr;
}
template <typename T>
T arg_of(const node_view &v, int k) {
    return *static_cast<const T *>(v.args[k]);
}
// The only dependent of `node` if that has no other dependency.
bool only_next(hipGraphNode_t node, hipGraphNode_t *next) {
    size_t n = 0, m = 0;
    if (hipGraphNodeGetDependentNodes(node, nullptr, &n) != hipSuccess || n != 1) return false;
    if (hipGraphNodeGetDependentNodes(node, next, &n) != hipSuccess || n != 1) return false;
    return hipGraphNodeGetDependencies(*next, nullptr, &m) == hipSuccess && m == 1;
}

// Another launch in the place of a node's own.  (Not a new node for the old one: the runtime walks the nodes in the order in
// which they were added, and with the first of a graph replaced by a later one it deals one chain over two queues: the four
// layers took 130 us instead of 93.)  `args` must not lie in the node.
hipError_t become(hipGraphNode_t node, void *func, uint32_t blocks, uint32_t threads, uint32_t lds, void **args, uint32_t blocks_y = 1u) {
    hipKernelNodeParams kp{};
    kp.func = func;
    kp.gridDim = dim3(blocks, blocks_y);
    kp.blockDim = dim3(threads);
    kp.sharedMemBytes = lds;
    kp.kernelParams = args;
    return hipGraphKernelNodeSetParams(node, &kp);
}
// What waits for `last` waits for `one` as well.
hipError_t hand_on(hipGraph_t graph, hipGraphNode_t last, hipGraphNode_t one) {
    size_t n = 0;
    hipError_t e = hipGraphNodeGetDependentNodes(last, nullptr, &n);
    if (e != hipSuccess || n == 0) return e;
    std::vector<hipGraphNode_t> behind(n);
    if ((e = hipGraphNodeGetDependentNodes(last, behind.data(), &n)) != hipSuccess) return e;
    const std::vector<hipGraphNode_t> from(n, one);
    return hipGraphAddDependencies(graph, from.data(), behind.data(), n);
}

hipError_t fuse_norm_chains(hipGraph_t graph) {
    const void *const norms[3] = {reinterpret_cast<const void *>(&rmsnorm_kernel<1>), reinterpret_cast<const void *>(&rmsnorm_kernel<2>),
                                  reinterpret_cast<const void *>(&rmsnorm_kernel<4>)};
    void *const fused[3] = {reinterpret_cast<void *>(&rmsnorm_adds_kernel<1>), reinterpret_cast<void *>(&rmsnorm_adds_kernel<2>),
                            reinterpret_cast<void *>(&rmsnorm_adds_kernel<4>)};
    size_t count = 0;
    if (hipGraphGetNodes(graph, nullptr, &count) != hipSuccess || count == 0) return hipSuccess;
    std::vector<hipGraphNode_t> nodes(count);
    if (hipGraphGetNodes(graph, nodes.data(), &count) != hipSuccess) return hipSuccess;
    auto kind = [&](const node_view &v) {
        for (int k = 0; k < 3; ++k)
            if (v.func == norms[k] && v.params.gridDim.x == 1u) return k;
        return -1;
    };
    // the norms first: a fusion destroys nodes behind its norm
    std::vector<hipGraphNode_t> heads;
    for (hipGraphNode_t node : nodes) {
        node_view v;
        if (kernel_node(node, &v) && kind(v) >= 0) heads.push_back(node);
    }
    for (hipGraphNode_t first : heads) {
        node_view norm;
        if (!kernel_node(first, &norm)) continue;
        const int which = kind(norm);
        const float *x = arg_of<const float *>(norm, 0), *w = arg_of<const float *>(norm, 2);
        float *y = arg_of<float *>(norm, 1);
        uint32_t n = arg_of<uint32_t>(norm, 3);
        float eps = arg_of<float>(norm, 4);
        norm_adds adds{};
        std::vector<hipGraphNode_t> chain;
        hipGraphNode_t last = first, next;
        node_view add;
        while (adds.count < norm_adds::kMost && only_next(last, &next) && kernel_node(next, &add) &&
               add.func == reinterpret_cast<const void *>(&axpy_kernel)) {
            const float *ax = arg_of<const float *>(add, 0);
            const uintptr_t a0 = reinterpret_cast<uintptr_t>(ax), y0 = reinterpret_cast<uintptr_t>(y), bytes = (uintptr_t)n * 4u;
            if (arg_of<float *>(add, 1) != y || arg_of<uint32_t>(add, 3) != n || (a0 & 15u) != 0u ||
                (a0 < y0 + bytes && y0 < a0 + bytes))
                break;
            adds.x[adds.count] = ax;
            adds.c[adds.count++] = arg_of<float>(add, 2);
            chain.push_back(next);
            last = next;
        }
        if (chain.empty()) continue;
        void *args[6] = {&x, &y, &w, &n, &eps, &adds};
        hipError_t e = become(first, fused[which], 1u, norm.params.blockDim.x, 0u, args);
        if (e == hipSuccess) e = hand_on(graph, last, first);
        for (hipGraphNode_t gone : chain)
            if (e == hipSuccess) e = hipGraphDestroyNode(gone);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

const void *norm_of(int k) {
    return k == 0 ? reinterpret_cast<const void *>(&rmsnorm_kernel<1>) : k == 1 ? reinterpret_cast<const void *>(&rmsnorm_kernel<2>)
                                                                             : reinterpret_cast<const void *>(&rmsnorm_kernel<4>);
}
// A norm of one vector: 0, 1, 2 by its pieces a lane; else -1.
int norm_kind(const node_view &v) {
    for (int k = 0; k < 3; ++k)
        if (v.func == norm_of(k) && v.params.gridDim.x == 1u) return k;
    return -1;
}
lev_footprint norm_touches(const node_view &v) {
    const size_t bytes = 4u * (size_t)arg_of<uint32_t>(v, 3);
    lev_footprint t;
    t.reads[0] = lev_span(arg_of<const float *>(v, 0), bytes);
    t.reads[1] = lev_span(arg_of<const float *>(v, 2), bytes);
    t.writes[0] = lev_span(arg_of<float *>(v, 1), bytes);
    return t;
}

lev_footprint scores_touches(const node_view &v) {   // of one token
    const size_t hidden = arg_of<uint32_t>(v, 3), experts = arg_of<uint32_t>(v, 4);
    lev_footprint t;
    t.reads[0] = lev_span(arg_of<const float *>(v, 0), 4u * hidden * experts);
    t.reads[1] = lev_span(arg_of<const float *>(v, 1), 4u * hidden);
    t.writes[0] = lev_span(arg_of<float *>(v, 2), 4u * experts);
    return t;
}

lev_gemv_args gemv_args_of(const node_view &v) {
    return lev_gemv_args{arg_of<const uint8_t *>(v, 0), arg_of<const float *>(v, 1), arg_of<float *>(v, 2), arg_of<uint32_t>(v, 3),
                         arg_of<uint32_t>(v, 4), arg_of<uint32_t>(v, 5), arg_of<uint32_t>(v, 6), arg_of<uint64_t>(v, 7),
                         arg_of<uint64_t>(v, 8)};
}
lev_footprint gemv_touches(const lev_gemv_args &g) {
    lev_footprint t;
    t.reads[0] = lev_span(g.w, (size_t)g.rows * (g.in_dim / 32u) * 18u);
    t.reads[1] = lev_span(g.x, 4u * (size_t)g.in_dim);
    t.writes[0] = lev_span(g.y, 4u * (size_t)g.rows);
    return t;
}

// The shared expert's FFN (gate/up, down, norm) and the scores and gate/up kernel of a MoE layer on the same h behind it, whose
// kernels only share that h: the scores join the FFN's gate/up kernel, which normalises it, and the down projection the
// layer's gate/up.  Where the layer's gate/up takes no GEMV along (more than one group of rows a workgroup, a down projection
// of more columns than it has waves, too many workgroups) the scores join the down projection; where they are not those of h, too.
hipError_t weave_shared_expert(hipGraph_t graph, const std::vector<hipGraphNode_t> &heads, const lev_ctx *ctx) {
    for (hipGraphNode_t first : heads) {   // down projections
        node_view g, n, r, u, f;
        hipGraphNode_t norm, scores, gate_up, ffn, next;
        if (!kernel_node(first, &g) || !only_next(first, &norm) || !kernel_node(norm, &n) || norm_kind(n) < 0 || !only_next(norm, &scores) ||
            !kernel_node(scores, &r) || r.func != lev_moe_scores_few() || r.params.gridDim.y != 1u)
            continue;
        lev_gemv_args ga = gemv_args_of(g);
        lev_scores_args sa{arg_of<const float *>(r, 0), arg_of<const float *>(r, 1), arg_of<float *>(r, 2), arg_of<uint32_t>(r, 3),
                           arg_of<uint32_t>(r, 4)};
        const lev_footprint gt = gemv_touches(ga), nt = norm_touches(n), st = scores_touches(r);
        if (!st.apart(gt) || !st.apart(nt)) continue;
        size_t ndeps = 0;
        lev_ffn_node fn;
        lev_footprint ut, wt = st;
        wt.reads[1] = lev_span();          // (h, which the workgroups of the scores form for themselves)
        lev_gate_up_gemv gu;
        lev_gemv_args gg = ga;
        hipError_t e;
        if (hipGraphNodeGetDependencies(first, nullptr, &ndeps) == hipSuccess && ndeps == 1u &&
            hipGraphNodeGetDependencies(first, &ffn, &ndeps) == hipSuccess && only_next(ffn, &next) && kernel_node(ffn, &f) &&
            lev_ffn_gate_up_node(f.func, f.args, &fn) && sa.x == fn.args.h && sa.hidden == fn.args.hidden && wt.apart(fn.touches) &&
            only_next(scores, &gate_up) && kernel_node(gate_up, &u) && u.params.gridDim.z == 1u &&
            lev_moe_expert_node(ctx, u.func, u.args, &ut) && ut.apart(gt) && ut.apart(nt) &&
            lev_moe_gate_up_and_gemv(ctx, u.func, u.args, &gg, &gu)) {
            const uint32_t each = fn.with_scores.threads / 256u;
            uint32_t blocks = f.params.gridDim.x;
            void *with_scores[3] = {&fn.args, &sa, &blocks}, *with_gemv[14];
            for (int k = 0; k < 9; ++k) with_gemv[k] = u.args[k];
            with_gemv[9] = &gu.rows_per_block, with_gemv[10] = &gg, with_gemv[11] = &gu.extra, with_gemv[12] = &gu.gemv_blocks;
            lev_norm_tail none{};
            with_gemv[13] = &none;
            e = become(ffn, fn.with_scores.func, blocks + (sa.experts + each - 1u) / each, fn.with_scores.threads, fn.with_scores.lds, with_scores);
            if (e == hipSuccess) e = become(first, gu.launch.func, gu.launch.blocks, gu.launch.threads, gu.launch.lds, with_gemv, gu.top_k);
            if (e == hipSuccess) e = hand_on(graph, gate_up, norm);
            if (e == hipSuccess) e = hipGraphDestroyNode(gate_up);
        } else {
            uint32_t blocks = g.params.gridDim.x;
            const lev_fused_launch l = lev_q4_0_gemv_and_scores(blocks, g.params.blockDim.x, sa.experts);
            void *args[3] = {&ga, &sa, &blocks};
            e = become(first, l.func, l.blocks, l.threads, l.lds, args);
            if (e == hipSuccess) e = hand_on(graph, scores, norm);
        }
        if (e == hipSuccess) e = hipGraphDestroyNode(scores);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// A norm in place, kernels of the MoE layer of one token, and a norm of the same length that adds the first one's result:
// the first norm goes into the second one's launch where the layer does not touch what it does (the shared expert's norm and
// the layer's; of 4096 values at most, as the layer).
hipError_t pair_norms(hipGraph_t graph, const std::vector<hipGraphNode_t> &nodes, const lev_ctx *ctx) {
    const void *const adds_kernel = reinterpret_cast<const void *>(&rmsnorm_adds_kernel<1>);
    for (hipGraphNode_t first : nodes) {
        node_view n, s;
        hipGraphNode_t behind, last;
        if (!kernel_node(first, &n) || norm_kind(n) != 0 || arg_of<const float *>(n, 0) != arg_of<float *>(n, 1) ||
            !only_next(first, &behind))
            continue;
        const lev_footprint nt = norm_touches(n);
        bool fits = true;
        last = behind;
        for (int layer = 0; layer < 3 && kernel_node(last, &s) && s.func != adds_kernel; ++layer) {   // scores, gate/up, down
            lev_footprint t;
            if (s.func == lev_moe_scores_few() && s.params.gridDim.y == 1u) t = scores_touches(s);
            else if (!lev_moe_expert_node(ctx, s.func, s.args, &t)) fits = false;
            fits = fits && nt.apart(t) && only_next(last, &last);
            if (!fits) break;
        }
        if (!fits || last == behind || !kernel_node(last, &s) || s.func != adds_kernel || s.params.gridDim.x != 1u ||
            arg_of<uint32_t>(s, 3) != arg_of<uint32_t>(n, 3) || !nt.apart(norm_touches(s)))
            continue;
        norm_adds adds = arg_of<norm_adds>(s, 5);
        norm_pair p{arg_of<float *>(n, 1), arg_of<const float *>(n, 2), arg_of<float>(n, 4), -1};
        for (int k = 0; k < adds.count; ++k) {
            if (adds.x[k] == p.x && p.own < 0) p.own = k;
            else if (lev_span(adds.x[k], nt.writes[0].bytes).meets(nt.writes[0])) fits = false;
        }
        if (!fits || p.own < 0) continue;
        const float *y = arg_of<const float *>(s, 0), *wy = arg_of<const float *>(s, 2);
        float *out = arg_of<float *>(s, 1);
        uint32_t len = arg_of<uint32_t>(s, 3);
        float eps = arg_of<float>(s, 4);
        void *args[7] = {&p, &y, &out, &wy, &len, &eps, &adds};
        size_t nbefore = 0;
        hipError_t e = become(last, reinterpret_cast<void *>(&rmsnorm_pair_kernel), 1u, s.params.blockDim.x, 0u, args);
        if (e == hipSuccess) e = hipGraphNodeGetDependencies(first, nullptr, &nbefore);
        if (e == hipSuccess && nbefore) {
            std::vector<hipGraphNode_t> before(nbefore);
            const std::vector<hipGraphNode_t> to(nbefore, behind);
            e = hipGraphNodeGetDependencies(first, before.data(), &nbefore);
            if (e == hipSuccess) e = hipGraphAddDependencies(graph, before.data(), to.data(), nbefore);
        }
        if (e == hipSuccess) e = hipGraphDestroyNode(first);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// The norm and adds in front of an FFN whose gate/up computes the scores too: every workgroup of it makes x for itself, with its
// weights on their way (2432 / 512 and 1280 four layers 78.9 us and 76.3, 3712 / 320 and 1408 79.4 and 73.3; 19 programs of
// several layers 0.92 to 1.01 of the time).  The
// norm of the pair that goes in place (the shared expert's of the layer before) is stored by the launch behind, unless that
// writes a new value there.
hipError_t front_norms(hipGraph_t graph, const std::vector<hipGraphNode_t> &heads, const lev_ctx *ctx) {
    for (hipGraphNode_t norm : heads) {
        node_view n, f, u;
        hipGraphNode_t ffn, behind;
        lev_ffn_node fn;
        lev_footprint ut;
        if (!kernel_node(norm, &n) || !only_next(norm, &ffn) || !kernel_node(ffn, &f) || !lev_ffn_gate_up_node(f.func, f.args, &fn) ||
            f.func != fn.with_scores.func || !only_next(ffn, &behind) || !kernel_node(behind, &u))
            continue;
        lev_norm_front front{};
        uint32_t len;
        front.own = -1;
        if (n.func == reinterpret_cast<const void *>(&rmsnorm_adds_kernel<1>)) {
            front.y = arg_of<const float *>(n, 0), front.out = arg_of<float *>(n, 1), front.wy = arg_of<const float *>(n, 2);
            len = arg_of<uint32_t>(n, 3), front.eps = arg_of<float>(n, 4), front.adds = arg_of<norm_adds>(n, 5);
        } else {
            const norm_pair p = arg_of<norm_pair>(n, 0);
            front.s = p.x, front.ws = p.wx, front.eps_s = p.eps, front.own = p.own;
            front.y = arg_of<const float *>(n, 1), front.out = arg_of<float *>(n, 2), front.wy = arg_of<const float *>(n, 3);
            len = arg_of<uint32_t>(n, 4), front.eps = arg_of<float>(n, 5), front.adds = arg_of<norm_adds>(n, 6);
        }
        lev_scores_args sa = arg_of<lev_scores_args>(f, 1);
        uint32_t blocks = arg_of<uint32_t>(f, 2);
        if (n.params.gridDim.x != 1u || front.out != fn.args.x || len != fn.args.hidden || front.adds.count > lev_norm_front::kMost) continue;
        int per_cu = 0;   // (more registers: what was on the chip at once has to be so still)
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn.with_front.func, (int)fn.with_front.threads, fn.with_front.lds) != hipSuccess ||
            (uint32_t)(per_cu * ctx->num_cus) < f.params.gridDim.x)
            continue;
        // what the norm reads, whose values no workgroup of the FFN's may change, and its result beside what those touch
        const size_t bytes = 4u * (size_t)len;
        lev_footprint rt, wt, ft = fn.touches;
        rt.reads[0] = lev_span(front.y, bytes), rt.reads[1] = lev_span(front.wy, bytes), rt.reads[2] = lev_span(front.s, bytes),
        rt.reads[3] = lev_span(front.ws, bytes);
        for (int k = 0; k < front.adds.count; ++k)
            if (k != front.own) rt.reads[4 + k] = lev_span(front.adds.x[k], bytes);
        wt.writes[0] = lev_span(front.out, bytes);
        ft.reads[0] = lev_span();                                          // (x, which is made)
        ft.reads[4] = lev_span(sa.wr, 4u * (size_t)sa.experts * sa.hidden);
        ft.writes[3] = lev_span(sa.scores, 4u * (size_t)sa.experts);
        if (!rt.apart(ft) || !wt.apart(ft) || !wt.apart(rt)) continue;
        if (front.s) {
            const lev_norm_tail tail{const_cast<float *>(front.s), front.ws, len, front.eps_s};
            if (!lev_moe_gate_up_and_gemv_is(u.func) || !lev_moe_expert_node(ctx, u.func, u.args, &ut)) continue;
            lev_footprint tt;
            tt.writes[0] = lev_span(front.s, bytes);
            tt.reads[0] = lev_span(front.ws, bytes);
            if (!tt.apart(ft)) continue;                                   // (the FFN, which would read s as it was before this norm)
            const lev_gemv_args g = arg_of<lev_gemv_args>(u, 10);
            if (!(g.y == front.s && g.rows >= len)) {
                if (!tt.apart(ut) || !tt.apart(gemv_touches(g))) continue;
                const hipError_t e = lev_moe_gate_up_and_gemv_tail(behind, tail);
                if (e == hipErrorNotSupported) continue;
                if (e != hipSuccess) return e;
            }
        }
        size_t nbefore = 0;
        void *args[4] = {&fn.args, &sa, &blocks, &front};
        hipError_t e = become(ffn, fn.with_front.func, f.params.gridDim.x, fn.with_front.threads, fn.with_front.lds, args);
        if (e == hipSuccess) e = hipGraphNodeGetDependencies(norm, nullptr, &nbefore);
        if (e == hipSuccess && nbefore) {
            std::vector<hipGraphNode_t> before(nbefore);
            const std::vector<hipGraphNode_t> to(nbefore, ffn);
            e = hipGraphNodeGetDependencies(norm, before.data(), &nbefore);
            if (e == hipSuccess) e = hipGraphAddDependencies(graph, before.data(), to.data(), nbefore);
        }
        if (e == hipSuccess) e = hipGraphDestroyNode(norm);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t fuse_nodes(hipGraph_t graph, const lev_ctx *ctx) {
    hipError_t e = fuse_norm_chains(graph);
    for (int rule = 0; rule < 3 && e == hipSuccess; ++rule) {
        size_t count = 0;
        if (hipGraphGetNodes(graph, nullptr, &count) != hipSuccess || count == 0) return hipSuccess;
        std::vector<hipGraphNode_t> nodes(count);
        if (hipGraphGetNodes(graph, nodes.data(), &count) != hipSuccess) return hipSuccess;
        // the heads of the pattern alone: a fusion destroys nodes that are no heads, or the head itself
        auto is_head = [&](const node_view &v) {
            if (rule == 0) return v.func == lev_q4_0_gemv_one_round();
            if (rule == 1) return norm_kind(v) == 0;
            return v.func == reinterpret_cast<const void *>(&rmsnorm_adds_kernel<1>) || v.func == reinterpret_cast<const void *>(&rmsnorm_pair_kernel);
        };
        std::vector<hipGraphNode_t> heads;
        for (hipGraphNode_t node : nodes) {
            node_view v;
            if (kernel_node(node, &v) && is_head(v)) heads.push_back(node);
        }
        e = rule == 0 ? weave_shared_expert(graph, heads, ctx) : rule == 1 ? pair_norms(graph, heads, ctx) : front_norms(graph, heads, ctx);
    }
    return e;
}

}  // namespace

struct lev_program {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    size_t nodes = 0;
};

extern "C" int lev_hip_program_begin(lev_ctx *ctx) {
    LEV_REQUIRE_CTX(ctx);
    if (ctx->stream == nullptr)
        return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT,
                        "program_begin: the default (null) stream cannot be captured; create the "
                        "context on a stream of its own");
    if (ctx->recording) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "program_begin: already recording");
    LEV_HIP(ctx, hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    ctx->recording = true;
    ctx->folded_nodes = 0;
    return LEV_OK;
}

extern "C" int lev_hip_program_end(lev_ctx *ctx, lev_program **out) {
    LEV_REQUIRE_CTX(ctx);
    if (!out) return LEV_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    if (!ctx->recording) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "program_end: not recording");
    ctx->recording = false;
    hipGraph_t graph = nullptr;
    LEV_HIP(ctx, hipStreamEndCapture(ctx->stream, &graph));
    lev_program *p = new (std::nothrow) lev_program();
    if (!p) {
        (void)hipGraphDestroy(graph);
        return lev_fail(ctx, LEV_ERR_DEVICE_UNAVAILABLE, "program_end: out of host memory");
    }
    p->graph = graph;
    (void)hipGraphGetNodes(graph, nullptr, &p->nodes);
    p->nodes += ctx->folded_nodes;   // counted as recorded: an operator each
    hipError_t e;
    try {
        e = fuse_nodes(graph, ctx);
    } catch (const std::bad_alloc &) {   // (its lists of nodes; nothing leaves a C entry as an exception)
        e = hipErrorOutOfMemory;
    }
    if (e == hipSuccess) (void)hipGetLastError();   // (of a question to the graph that had no answer: the nodes stayed as they were)
    if (e == hipSuccess) e = hipGraphInstantiate(&p->exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(graph);
        delete p;
        return lev_hip_check(ctx, e, "hipGraphInstantiate");
    }
    ++ctx->live_programs;
    *out = p;
    return LEV_OK;
}

extern "C" int lev_hip_program_run(lev_ctx *ctx, lev_program *program) {
    LEV_REQUIRE_CTX(ctx);
    if (!program || !program->exec) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "program_run: null program");
    if (ctx->recording) return lev_fail(ctx, LEV_ERR_INVALID_ARGUMENT, "program_run: still recording");
    return lev_hip_check(ctx, hipGraphLaunch(program->exec, ctx->stream), "hipGraphLaunch");
}

extern "C" int lev_hip_program_destroy(lev_ctx *ctx, lev_program *program) {
    LEV_REQUIRE_CTX(ctx);
    if (!program) return LEV_OK;
    LEV_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (program->exec) (void)hipGraphExecDestroy(program->exec);
    if (program->graph) (void)hipGraphDestroy(program->graph);
    delete program;
    if (ctx->live_programs > 0 && --ctx->live_programs == 0) {
        // no program is left that could hold a parked scratch address
        for (void *p : ctx->retired_scratch) (void)hipFree(p);
        ctx->retired_scratch.clear();
    }
    return LEV_OK;
}

extern "C" int lev_hip_program_node_count(lev_program *program, size_t *out) {
    if (!program || !out) return LEV_ERR_INVALID_ARGUMENT;
    *out = program->nodes;
    return LEV_OK;
}
