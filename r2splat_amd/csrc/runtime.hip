// Error reporting and small utility kernels shared by every entry point.
#include "common.hpp"

#include <chrono>
#include <cstdarg>
#include <limits>
#include <thread>

namespace r2s {

static thread_local char g_error[1024] = "";

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
}

int check_launch(const char* where) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: kernel launch failed: %s", where, hipGetErrorString(e));
        return R2S_ERR_HIP;
    }
    return R2S_OK;
}

}  // namespace r2s

extern "C" int r2s_abi_version(void) { return 5; }

extern "C" const char* r2s_last_error(void) { return r2s::g_error; }

// ---------------------------------------------------------------------------
// Value checks: one workgroup row (blockIdx.y) per check, a grid-stride scan
// of its buffer, and flags[check] = 1 from any wave that saw a bad element
// (every such store writes the same value, so their order does not matter).
// ---------------------------------------------------------------------------
namespace r2s {

constexpr int kCheckThreads = 256;
constexpr uint32_t kCheckPacks = 4;
constexpr uint32_t kCheckBlocks = 4096;  // enough workgroups per check to stream a large buffer at HBM rate

struct ValueCheckTable {
    r2s_value_check c[R2S_MAX_VALUE_CHECKS];
};

template <typename S>
__device__ __forceinline__ bool bad_element(S x, int kind) {  // (kind is uniform: selects, no branches)
    const bool nonfinite = !(fabs(x) <= std::numeric_limits<S>::max());
    const bool nonpositive = x <= S(0), negative = x < S(0);
    return kind == R2S_CHECK_NONFINITE ? nonfinite : kind == R2S_CHECK_NONPOSITIVE ? nonpositive : negative;
}

template <typename S>
__device__ __forceinline__ bool scan_check(const r2s_value_check& c) {
    const S* p = static_cast<const S*>(c.data);
    const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
    bool bad = false;
    if (c.kind >= R2S_CHECK_ZERO_ROW) {
        const uint64_t rows = c.n / c.row;
        for (uint64_t r = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; r < rows; r += stride) {
            const S* m = p + r * c.row;
            bool b;
            if (c.kind == R2S_CHECK_K_FOCAL) {
                b = m[0] <= S(0) || m[4] <= S(0);
            } else if (c.kind == R2S_CHECK_K_PINHOLE) {
                b = m[1] != S(0) || m[3] != S(0) || m[6] != S(0) || m[7] != S(0) || m[8] != S(1);
            } else if (c.kind == R2S_CHECK_VIEW_ROW) {
                b = m[12] != S(0) || m[13] != S(0) || m[14] != S(0) || m[15] != S(1);
            } else {
                b = true;
                for (uint32_t k = 0; k < c.row; ++k) b = b && m[k] == S(0);
            }
            bad = bad || b;
        }
    } else {
        // 16-byte packs, kCheckPacks in flight a thread (one element at a time, the checks
        // of 256 views of 512^2 and 500k primitives took 338 us, now 202); the tail, or a
        // buffer off the alignment, by elements
        constexpr uint32_t kPack = 16 / sizeof(S);
        struct __align__(16) Pack {
            S v[kPack];
        };
        const uint64_t packs = reinterpret_cast<uintptr_t>(p) % 16 == 0 ? c.n / kPack : 0;
        const uint64_t first = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
        for (uint64_t i = first; i < packs; i += kCheckPacks * stride) {
            Pack q[kCheckPacks];
#pragma unroll
            for (uint32_t j = 0; j < kCheckPacks; ++j)  // past the end: the thread's first pack again
                q[j] = reinterpret_cast<const Pack*>(p)[i + j * stride < packs ? i + j * stride : i];
#pragma unroll
            for (uint32_t j = 0; j < kCheckPacks; ++j)
#pragma unroll
                for (uint32_t k = 0; k < kPack; ++k) bad |= bad_element(q[j].v[k], c.kind);
        }
        for (uint64_t i = packs * kPack + first; i < c.n; i += stride) bad = bad || bad_element(p[i], c.kind);
    }
    return bad;
}

__global__ void __launch_bounds__(kWave) value_checks_clear_kernel(uint32_t n_checks, uint32_t* __restrict__ flags) {
    if (threadIdx.x < n_checks) flags[threadIdx.x] = 0u;
}

__global__ void __launch_bounds__(kCheckThreads) value_checks_kernel(ValueCheckTable table,
                                                                     uint32_t* __restrict__ flags) {
    const r2s_value_check& c = table.c[blockIdx.y];
    const bool bad = c.dtype == R2S_F64 ? scan_check<double>(c) : scan_check<float>(c);
    // (the flags may lie in pinned host memory: a system-scope store)
    if (__ballot(bad) != 0 && threadIdx.x % kWave == 0) {
        __hip_atomic_store(flags + blockIdx.y, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __threadfence_system();
    }
}

}  // namespace r2s

namespace r2s {

static int launch_checks(const r2s_value_check* checks, uint32_t n_checks, uint32_t* flags, hipStream_t stream) {
    ValueCheckTable table = {};
    uint64_t most = 0;
    for (uint32_t i = 0; i < n_checks; ++i) {
        const r2s_value_check& c = checks[i];
        R2S_REQUIRE(c.dtype == R2S_F32 || c.dtype == R2S_F64, "check %u: dtype must be R2S_F32 or R2S_F64", i);
        R2S_REQUIRE(c.kind >= R2S_CHECK_NONFINITE && c.kind <= R2S_CHECK_VIEW_ROW, "check %u: unknown kind %d", i,
                    c.kind);
        R2S_REQUIRE(c.n == 0 || c.data, "check %u: data must be non-null", i);
        R2S_REQUIRE(c.kind < R2S_CHECK_ZERO_ROW || (c.row > 0 && c.n % c.row == 0),
                    "check %u: row must be positive and divide n", i);
        R2S_REQUIRE((c.kind != R2S_CHECK_K_FOCAL && c.kind != R2S_CHECK_K_PINHOLE) || c.row == 9,
                    "check %u: intrinsics rows hold 9 elements", i);
        R2S_REQUIRE(c.kind != R2S_CHECK_VIEW_ROW || c.row == 16, "check %u: viewmat rows hold 16 elements", i);
        table.c[i] = c;
        most = std::max<uint64_t>(most, c.kind >= R2S_CHECK_ZERO_ROW ? c.n / c.row : c.n);
    }
    constexpr uint64_t kPerBlock = kCheckThreads * kCheckPacks * 4;  // (4 floats a pack)
    const uint64_t want = std::max<uint64_t>(1, (most + kPerBlock - 1) / kPerBlock);
    const uint32_t blocks = uint32_t(std::min<uint64_t>(kCheckBlocks, want));
    value_checks_kernel<<<dim3(blocks, n_checks), kCheckThreads, 0, stream>>>(table, flags);
    return check_launch("value_checks");
}

// ---------------------------------------------------------------------------
// Words handed to the host while the stream goes on: a one-wave kernel copies
// them (or nothing: the value checks set their flags there themselves) to pinned
// host memory and raises the first word, which the host polls. Against a copy
// to pageable memory and a stream synchronisation this leaves out the copy
// launch and the wake-up, and work launched after the hand-over runs while the
// host waits.
// ---------------------------------------------------------------------------
constexpr uint32_t kMaxFetch = 64;

__global__ void __launch_bounds__(kWave)
fetch_kernel(const uint32_t* __restrict__ src, uint32_t n, uint32_t* host) {
    if (threadIdx.x < n) __hip_atomic_store(host + 1 + threadIdx.x, src[threadIdx.x], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();  // one wave: every lane's words precede the first word
    if (threadIdx.x == 0) __hip_atomic_store(host, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

int fetch_begin(const uint32_t* src, uint32_t n, uint32_t* host, hipStream_t stream) {
    __atomic_store_n(host, 0u, __ATOMIC_RELEASE);
    fetch_kernel<<<1, kWave, 0, stream>>>(src, n, host);
    return check_launch("fetch");
}

}  // namespace r2s

extern "C" int r2s_value_checks(const r2s_value_check* checks, uint32_t n_checks, uint32_t* flags,
                                r2s_stream_t stream) {
    using namespace r2s;
    if (n_checks == 0) return R2S_OK;
    R2S_REQUIRE(checks && flags, "checks and flags must be non-null");
    R2S_REQUIRE(n_checks <= R2S_MAX_VALUE_CHECKS, "at most %d value checks per call", R2S_MAX_VALUE_CHECKS);
    value_checks_clear_kernel<<<1, kWave, 0, stream>>>(n_checks, flags);
    if (int rc = check_launch("value_checks_clear")) return rc;
    return launch_checks(checks, n_checks, flags, stream);
}

extern "C" int r2s_value_checks_begin(const r2s_value_check* checks, uint32_t n_checks, uint32_t* host,
                                      r2s_stream_t stream) {
    using namespace r2s;
    R2S_REQUIRE(checks && host, "checks and host must be non-null");
    R2S_REQUIRE(n_checks > 0 && n_checks <= R2S_MAX_VALUE_CHECKS, "1 to %d value checks per call",
                R2S_MAX_VALUE_CHECKS);
    for (uint32_t i = 0; i < n_checks; ++i) host[1 + i] = 0u;
    if (int rc = launch_checks(checks, n_checks, host + 1, stream)) return rc;
    const int rc = fetch_begin(nullptr, 0, host, stream);
    if (rc) (void)hipStreamSynchronize(stream);  // the checks write to `host`, which the caller takes back
    return rc;
}

extern "C" int r2s_fetch_begin(const uint32_t* src, uint32_t n, uint32_t* host, r2s_stream_t stream) {
    using namespace r2s;
    R2S_REQUIRE(src && host, "src and host must be non-null");
    R2S_REQUIRE(n > 0 && n <= kMaxFetch, "1 to %u words per call", kMaxFetch);
    return fetch_begin(src, n, host, stream);
}

// Polls the first word: without pause for 4 ms (a sleep of 20 us lasts 75 us
// with the timer's slack: waits of 0.1-0.7 ms ended 45 us late with a spin of
// 50 us), then every 50 us or so, asking the runtime whether the stream has ended
// (an error, or all work done) so that a failed launch ends the wait.
extern "C" int r2s_fetch_wait(const uint32_t* host, r2s_stream_t stream) {
    using namespace r2s;
    using clock = std::chrono::steady_clock;
    R2S_REQUIRE(host, "host must be non-null");
    const auto raised = [&] { return __atomic_load_n(host, __ATOMIC_ACQUIRE) != 0u; };
    const auto spin_end = clock::now() + std::chrono::milliseconds(4);
    do {
        for (int k = 0; k < 64; ++k) {
            if (raised()) return R2S_OK;
            __builtin_ia32_pause();
        }
    } while (clock::now() < spin_end);
    while (!raised()) {
        hipError_t e = hipStreamQuery(stream);
        if (e == hipErrorNotReady) {
            // (the query's own state alone: an earlier call's error stays for its reader)
            if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError();
            std::this_thread::sleep_for(std::chrono::microseconds(50));
            continue;
        }
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e == hipSuccess && raised()) return R2S_OK;
        if (e != hipSuccess) (void)hipGetLastError();  // reported here
        set_error("fetch: %s", e == hipSuccess ? "the stream ended without the words" : hipGetErrorString(e));
        return R2S_ERR_HIP;
    }
    return R2S_OK;
}
