// Session creation against a device with little memory, on the CPU: this program
// defines the HIP calls that context and session creation make (allocations from
// host memory up to a limit, launches that do nothing), so libtokhip's take effect
// here instead of the runtime's.  Exit status 0: the sessions are created wherever
// their required buffers fit, and report what they hold.  Test infrastructure.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>

#include "tokhip.h"

namespace {
std::map<void *, size_t> g_blocks;
size_t g_used = 0, g_limit = SIZE_MAX;
hipError_t g_last = hipSuccess;
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    if (n > g_limit - g_used) return g_last = hipErrorOutOfMemory;
    *p = std::malloc(16);
    g_blocks[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    g_used -= g_blocks[p];
    g_blocks.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipGetLastError(); }
}

namespace {

// Creates a session with at most `spare` bytes left beside what it needs; its Q
// scratch in slots, or 0 when it could not be created.
uint64_t slots(uint64_t chunk, uint64_t layers, tkh_dtype storage, size_t spare) {
    tkh_error e{};
    tkh_context *ctx = nullptr;
    tkh_session_options o{};
    o.capacity = 2 * chunk;
    o.prefill_chunk_size = chunk;
    o.vocab_size = 64;
    o.layers = layers;
    o.query_heads = 32;
    o.kv_heads = 8;
    o.head_dim = 128;
    o.storage = storage;
    o.score_scale = 0.125f;
    o.norm_epsilon = 1e-6f;
    o.rotary = TKH_ROTARY_SPLIT_HALF;
    o.theta = 10000.0f;
    o.factor = 1.0f;
    o.low_freq_factor = 1.0f;
    o.high_freq_factor = 4.0f;
    o.original_max_positions = 8192;
    const uint64_t slot = chunk * 32 * 128 * (storage == TKH_F32 ? 4 : 2), rope = 2 * chunk * 64 * 8;
    const uint64_t kv = layers * 2 * 2 * chunk * 8 * 128 * (storage == TKH_F32 ? 4 : 2);
    g_limit = SIZE_MAX;
    if (tkh_context_create(0, nullptr, 1 << 20, 1, &ctx, &e) != TKH_OK) {
        std::printf("FAIL context: %s\n", e.message);
        return 0;
    }
    g_limit = spare == SIZE_MAX ? spare : g_used + kv + slot + rope + 4096 + spare;
    tkh_session *s = nullptr;
    const uint32_t rc = tkh_session_create(ctx, &o, nullptr, &s, &e);
    uint64_t n = 0;
    if (rc != TKH_OK) {
        std::printf("session of %llu layers, chunk %llu: %s\n", (unsigned long long)layers, (unsigned long long)chunk,
                    e.message);
    } else {
        tkh_session_state st{};
        tkh_session_state_get(s, &st);
        n = (st.scratch_bytes - rope) / slot;
        if (hipGetLastError() != hipSuccess) {
            std::printf("an error is left for the next call\n");
            n = 0;
        }
        tkh_session_destroy(s);
    }
    tkh_context_destroy(ctx);
    if (g_used != 0) {
        std::printf("%zu bytes not freed\n", g_used);
        return 0;
    }
    std::printf("%llu layers, chunk %llu, spare %zu: %llu slots\n", (unsigned long long)layers, (unsigned long long)chunk,
                spare, (unsigned long long)n);
    return n;
}

}  // namespace

int main() {
    bool ok = slots(128, 6, TKH_BF16, SIZE_MAX) == 6;
    ok &= slots(128, 20, TKH_BF16, SIZE_MAX) == 8;
    ok &= slots(128, 6, TKH_F32, SIZE_MAX) == 1;
    ok &= slots(128, 6, TKH_BF16, 0) == 1;          // just what the session needs
    ok &= slots(128, 6, TKH_BF16, 5 << 20) == 1;    // not beside the first slot
    ok &= slots(8192, 6, TKH_F16, SIZE_MAX) == 4;   // 64 MiB each
    ok &= slots(65536, 6, TKH_BF16, SIZE_MAX) == 1;  // 512 MiB each
    std::printf("%s\n", ok ? "OK" : "FAIL");
    return ok ? 0 : 1;
}
