// Error text and version entry points of libmoe_gfx950.so.
#include "common.h"

#include <atomic>
#include <chrono>
#if defined(__x86_64__)
#include <immintrin.h>
#endif

static thread_local char g_err[512] = {0};

char* moe_err_buf() { return g_err; }

int moe_fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int moe_check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return moe_fail(MOE_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
    return MOE_OK;
}

// Reading the word over and over notices the store within a microsecond; waiting for an event or the stream takes the runtime some
// ten (and, through torch's objects, the interpreter as many again).  After 200 us the wait is left to the runtime.
extern "C" int moe_wait_i32(const int32_t* value, int32_t pending, moe_stream_t stream) {
    MOE_REQUIRE(value, MOE_ERR_INVALID, "wait: null pointer");
    const volatile int32_t* v = value;
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    bool there = false;
    do {
        for (int i = 0; i < 64 && !there; ++i) {
            there = *v != pending;
#if defined(__x86_64__)
            if (!there) _mm_pause();
#endif
        }
    } while (!there && std::chrono::steady_clock::now() < until);
    if (!there) {
        const hipError_t e = hipStreamSynchronize((hipStream_t)stream);
        if (e != hipSuccess) return moe_fail(MOE_ERR_LAUNCH, "wait: %s", hipGetErrorString(e));
        if (*v == pending) return moe_fail(MOE_ERR_LAUNCH, "wait: the stream ended without the value");
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return MOE_OK;
}

extern "C" int moe_abi_version(void) { return 3; }

extern "C" const char* moe_last_error(void) { return g_err; }
