// What the library makes of HIP calls that fail, on a machine without a GPU: this program defines the HIP runtime's functions
// that the library calls (the dynamic linker takes them from here), hands out host memory, lets allocations fail from a given
// size on and counts launches instead of making them.  As in the runtime a failed call's error stays until hipGetLastError
// fetches it, whoever asks.
#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__
#endif
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "leviathan_hip.h"

namespace {
hipError_t last = hipSuccess;
size_t refused_from = (size_t)-1;      // bytes of an allocation
int failures = 0;
std::vector<std::string> launched;
std::map<const void *, std::string> &names() {
    static std::map<const void *, std::string> n;
    return n;
}
hipError_t fails(hipError_t e) { return last = e; }

struct call_config { dim3 grid, block; size_t lds; hipStream_t stream; } pushed;

void expect(bool ok, const char *what, int line) {
    if (ok) return;
    std::printf("line %d: %s\n", line, what);
    ++failures;
}
#define EXPECT(c) expect((c), #c, __LINE__)

// the launches since the last call whose kernel's name holds `part`
size_t launches_of(const char *part) {
    size_t n = 0;
    for (const std::string &k : launched) n += k.find(part) != std::string::npos;
    return n;
}
}  // namespace

extern "C" {
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->name, "none");
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = (size_t)288 << 30;
    p->sharedMemPerBlock = 160 << 10;
    p->sharedMemPerMultiprocessor = 160 << 10;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
    if (bytes >= refused_from) return fails(hipErrorOutOfMemory);
    // (what the library allocates here is never read)
    *p = std::malloc(bytes > 4096 ? 4096 : bytes);
    return *p ? hipSuccess : fails(hipErrorOutOfMemory);
}
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return *p = std::calloc(1, bytes), hipSuccess; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = reinterpret_cast<hipStream_t>(16), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = std::malloc(16), hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) { return std::memset(a, 0, sizeof(*a)), hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
    launched.push_back(names()[f]);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { return pushed = {g, b, lds, s}, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = pushed.grid, *b = pushed.block, *lds = pushed.lds, *s = pushed.stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipRegisterFunction(void **, const void *host, char *, const char *device, unsigned, void *, void *, void *, void *, int *) {
    names()[host] = device;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}

int main() {
    lev_ctx *ctx = nullptr;
    if (lev_hip_ctx_create(0, LEV_HIP_OWN_STREAM, &ctx) != LEV_OK) {
        std::printf("no context\n");
        return 1;
    }
    // operands are not read: only their addresses and sizes count
    alignas(16) static char w[16], x[16], y[16];
    const size_t huge = (size_t)1 << 34;
    auto *const xf = reinterpret_cast<float *>(x), *const yf = reinterpret_cast<float *>(y);
    auto prefill = [&](bool q6, uint32_t in_dim, uint32_t rows, uint32_t tokens) {
        launched.clear();
        auto *const call = q6 ? lev_hip_q6_k_gemm_prefill : lev_hip_q4_k_gemm_prefill;
        return call(ctx, w, huge, 0, reinterpret_cast<const uint16_t *>(x), (size_t)in_dim * tokens, yf, huge, in_dim, rows, tokens);
    };
    auto next = [&] { return lev_hip_axpy(ctx, xf, yf, 1.f, 64); };   // a call that has nothing to do with the failed one

    // no memory for the fragments of X: the kernel for short prompts serves the call
    for (int q6 = 0; q6 < 2; ++q6) {
        refused_from = 1 << 20;
        EXPECT(prefill(q6, 4096, 12288, 512) == LEV_OK);
        EXPECT(launches_of("gemm_split_kernel") == 1 && launched.size() == 1);
        EXPECT(next() == LEV_OK);
        // slices along K without a place for their sums: a launch each
        EXPECT(prefill(q6, 12288, 4096, 77) == LEV_OK);
        EXPECT(launches_of("gemm_split_kernel") == launched.size() && launched.size() > 1);
        EXPECT(next() == LEV_OK);
    }
    // int8 activations in slices, planes of f32 columns: the kernels that need no scratch
    launched.clear();
    EXPECT(lev_hip_q6_k_gemv_q8(ctx, w, huge, 0, reinterpret_cast<int8_t *>(x), xf, 7 * 12288, yf, huge, 12288, 4096, 7) == LEV_OK);
    EXPECT(launched.size() > 1);
    EXPECT(next() == LEV_OK);
    launched.clear();
    EXPECT(lev_hip_q4_k_gemv_ncol(ctx, w, huge, 0, xf, 4 * 12288, nullptr, 1e-6f, yf, huge, 12288, 4096, 4) == LEV_OK);
    EXPECT(launches_of("q4k_planes_kernel") == 0 && !launched.empty());
    EXPECT(next() == LEV_OK);
    // what cannot be served fails, and the call behind it does not
    lev_moe_experts pools{};
    pools.d_base = w, pools.base_bytes = (size_t)1 << 40;
    pools.hidden = 2816, pools.inter = 704, pools.experts = 128;
    pools.gate_stride = pools.up_stride = pools.down_stride = (uint64_t)2816 * 704 / 32 * 18;
    pools.up_off = 128 * pools.gate_stride, pools.down_off = 2 * pools.up_off;
    int32_t ids[8];
    refused_from = 1;
    EXPECT(lev_hip_moe_layer_q4_0(ctx, &pools, xf, nullptr, xf, yf, ids, yf, 8, 1000) == LEV_ERR_EXCEEDS_WORKING_SET);
    EXPECT(next() == LEV_OK);
    void *buffer = nullptr;
    EXPECT(lev_hip_buf_alloc(ctx, 4096, &buffer) == LEV_ERR_EXCEEDS_WORKING_SET && !buffer);
    EXPECT(next() == LEV_OK);
    // with memory again the kernels that want it run
    refused_from = (size_t)-1;
    EXPECT(prefill(false, 4096, 12288, 512) == LEV_OK);
    EXPECT(launches_of("gemm_x_fragments") == 1 && launches_of("gemm_wide_kernel") == 1 && launched.size() == 2);
    // an error that is there when a context is made or given back is not the next one's
    refused_from = 1;
    lev_ctx *none = nullptr;
    EXPECT(lev_hip_ctx_create(0, LEV_HIP_OWN_STREAM, &none) == LEV_ERR_DEVICE_UNAVAILABLE && !none);
    EXPECT(next() == LEV_OK);
    lev_hip_ctx_destroy(ctx);
    std::printf(failures ? "%d failed\n" : "ok\n", failures);
    return failures != 0;
}
