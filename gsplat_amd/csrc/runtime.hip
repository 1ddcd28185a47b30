// Error plumbing, version string and small utility kernels shared by the
// extern "C" entry points of libgsplat_hip.so.
#include "common.h"

namespace gs {

namespace {
thread_local std::string g_last_error;
}

void set_error(const std::string &msg) { g_last_error = msg; }
void clear_error() { g_last_error.clear(); }

int fail(int code, const std::string &msg) {
    set_error(msg);
    return code;
}

int check_launch(const char *what) {
    hipError_t err = hipGetLastError();
    if (err != hipSuccess)
        return fail(GSPLAT_ERR_LAUNCH,
                    std::string(what) + ": " + hipGetErrorString(err));
    return GSPLAT_OK;
}

__global__ void clear_lookback_kernel(uint32_t *ticket, uint64_t *status,
                                      int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0)
        *ticket = 0u;
    if (i < n)
        status[i] = 0ull;
}

int clear_lookback(void *ws, int64_t n_blocks, hipStream_t stream) {
    Lookback lb = lookback_from(ws);
    const int64_t n = n_blocks > 0 ? n_blocks : 1;
    clear_lookback_kernel<<<(unsigned)ceil_div(n, 256), 256, 0, stream>>>(
        lb.ticket, lb.status, n_blocks);
    return check_launch("clear_lookback");
}

}  // namespace gs

extern "C" const char *gsplat_last_error(void) {
    return gs::g_last_error.c_str();
}

extern "C" const char *gsplat_version(void) {
    return "gsplat_hip 0.1.0 gfx950";
}

extern "C" int gsplat_wait_count(const int64_t *word, int64_t *value,
                                 gsplat_stream_t stream) {
    gs::clear_error();
    GS_REQUIRE(word != nullptr && value != nullptr, "wait_count: NULL word or value");
    for (uint32_t spin = 1;; ++spin) {
        const int64_t v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
        if (v >= 0) {
            *value = v;
            return GSPLAT_OK;
        }
        if ((spin & 4095u) != 0) {
            __builtin_ia32_pause();
            continue;
        }
        const hipError_t err = hipStreamQuery(gs::as_stream(stream));
        if (err == hipErrorNotReady)
            continue;
        (void)hipGetLastError();
        if (err != hipSuccess)
            return gs::fail(GSPLAT_ERR_LAUNCH,
                            std::string("wait_count: ") + hipGetErrorString(err));
        // the stream has drained: the word is written now, or never
        const int64_t last = __atomic_load_n(word, __ATOMIC_ACQUIRE);
        if (last < 0)
            return gs::fail(GSPLAT_ERR_INVALID_ARGUMENT,
                            "wait_count: nothing queued on the stream writes the word");
        *value = last;
        return GSPLAT_OK;
    }
}

// The build passes the digest of include/gsplat_hip.h's declarations.
#ifndef GSPLAT_ABI_HASH
#error "GSPLAT_ABI_HASH must be defined by the build (digest of include/gsplat_hip.h)"
#endif

extern "C" const char *gsplat_abi_version(void) {
    return GSPLAT_ABI_HASH;
}
