// Shared device/host helpers for the gfx950 CT splatting kernels.
//
// Everything in this library is plain HIP for CDNA4 (wave64). Host entry points
// are `extern "C"` and take raw device pointers, sizes and a hipStream_t; the
// caller owns every allocation (outputs and workspaces), so no entry point
// allocates device memory and all of them can be captured into a hipGraph.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <cmath>
#include <algorithm>

#include "../../include/r2splat_hip.h"

namespace r2s {

constexpr int kWave = 64;

// A dispatch's grid size counts work-items in 32 bits, so blocks * threads
// must stay below 2^32. Kernels with one wave per element (intersections can
// number in the hundreds of millions) loop over a grid capped at this many
// blocks instead of launching one block per few elements.
constexpr uint32_t kIsectBlocks = 1u << 16;

// ---------------------------------------------------------------------------
// Error reporting: thread-local message + status code.
// ---------------------------------------------------------------------------
void set_error(const char* fmt, ...);
int check_launch(const char* where);
// Copies n words of device memory to host[1..n] (pinned) behind the stream's work, then raises host[0].
int fetch_begin(const uint32_t* src, uint32_t n, uint32_t* host, hipStream_t stream);

#define R2S_REQUIRE(cond, ...)                 \
    do {                                       \
        if (!(cond)) {                         \
            ::r2s::set_error(__VA_ARGS__);     \
            return R2S_ERR_INVALID;            \
        }                                      \
    } while (0)

#define R2S_HIP(call)                                                         \
    do {                                                                      \
        hipError_t _e = (call);                                               \
        if (_e != hipSuccess) {                                               \
            ::r2s::set_error("%s failed: %s", #call, hipGetErrorString(_e));  \
            return R2S_ERR_HIP;                                               \
        }                                                                     \
    } while (0)

inline uint32_t ceil_div(uint64_t a, uint64_t b) { return static_cast<uint32_t>((a + b - 1) / b); }

// ---------------------------------------------------------------------------
// Precision-dependent math. Float uses the hardware transcendental units
// (v_exp_f32 / v_log_f32 are base-2); double uses the IEEE library routines.
// ---------------------------------------------------------------------------
template <typename S> struct Math;

template <> struct Math<float> {
    static __device__ __forceinline__ float exp(float x) { return __expf(x); }
    static __device__ __forceinline__ float log(float x) { return __logf(x); }
    static __device__ __forceinline__ float pow(float b, float e) { return __expf(e * __logf(b)); }
    static __device__ __forceinline__ float sqrt(float x) { return sqrtf(x); }
    static __device__ __forceinline__ float fma(float a, float b, float c) { return fmaf(a, b, c); }
};

template <> struct Math<double> {
    static __device__ __forceinline__ double exp(double x) { return ::exp(x); }
    static __device__ __forceinline__ double log(double x) { return ::log(x); }
    static __device__ __forceinline__ double pow(double b, double e) { return ::pow(b, e); }
    static __device__ __forceinline__ double sqrt(double x) { return ::sqrt(x); }
    static __device__ __forceinline__ double fma(double a, double b, double c) { return ::fma(a, b, c); }
};

// Type-dispatch helper for the C-ABI dtype code.
template <typename F>
inline int dispatch_dtype(int dtype, F&& f) {
    if (dtype == R2S_F32) return f(float{});
    if (dtype == R2S_F64) return f(double{});
    set_error("unsupported dtype code %d (expected R2S_F32 or R2S_F64)", dtype);
    return R2S_ERR_INVALID;
}

// ---------------------------------------------------------------------------
// Wave64 reductions (butterfly over 64 lanes; the compiler lowers the xor
// shuffles to DPP / ds_swizzle on gfx950).
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// Inclusive scan over the 64 lanes by data-parallel-primitive moves (within
// rows of 16, then across rows): no LDS traffic, every lane active.
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return x;
}

// LDS written by some lanes of a wave is visible to its other lanes.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inclusive maximum over the lanes up to this one (unsigned).
__device__ __forceinline__ uint32_t wave_max_scan(uint32_t x) {
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x111, 0xf, 0xf, false)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x112, 0xf, 0xf, false)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x114, 0xf, 0xf, false)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x118, 0xf, 0xf, false)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x142, 0xa, 0xf, false)));
    x = max(x, uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x143, 0xc, 0xf, false)));
    return x;
}

// Lanes of `among` that hold the same value as this lane, for values of up to
// `bits` bits: each ballot keeps the lanes that agree with this lane's bit
// (four bits per loop: bits past the value are 0 in every lane).
__device__ __forceinline__ uint64_t wave_match(uint32_t value, uint32_t bits, uint64_t among) {
    uint32_t lo = uint32_t(among), hi = uint32_t(among >> 32);
    for (uint32_t b = 0; b < bits; b += 4) {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t own = uint32_t(__builtin_amdgcn_sbfe(int(value >> j), 0, 1));  // all ones where set
            const uint64_t m = __ballot(own != 0u);
            lo &= ~(uint32_t(m) ^ own);
            hi &= ~(uint32_t(m >> 32) ^ own);
        }
        value >>= 4;
    }
    return (uint64_t(hi) << 32) | lo;
}

// Device atomics on float / double with hardware fp atomics (-munsafe-fp-atomics).
template <typename S>
__device__ __forceinline__ void atomic_add(S* p, S v) { atomicAdd(p, v); }

// ITEMS consecutive words of a thread's run, from word i of p (0 past word n), and
// back. A run loaded word by word costs each instruction a cache line per lane
// (a one-workgroup scan of 12k words took 10 us); where p + i and p + i + ITEMS are
// 16-byte aligned (i is a multiple of ITEMS, so p decides) and the run is whole, it
// moves in 16-byte pieces.
__device__ __forceinline__ bool runs_aligned(const uint32_t* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

template <int ITEMS>
__device__ __forceinline__ void load_run(const uint32_t* __restrict__ p, size_t i, size_t n, bool aligned,
                                         uint32_t (&v)[ITEMS]) {
    static_assert(ITEMS % 4 == 0, "whole 16-byte pieces");
    if (aligned && i + ITEMS <= n) {
#pragma unroll
        for (int k = 0; k < ITEMS; k += 4) {
            const uint4 q = *reinterpret_cast<const uint4*>(p + i + k);
            v[k] = q.x;
            v[k + 1] = q.y;
            v[k + 2] = q.z;
            v[k + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) v[k] = i + k < n ? p[i + k] : 0u;
    }
}
template <int ITEMS>
__device__ __forceinline__ void store_run(uint32_t* __restrict__ p, size_t i, size_t n, bool aligned,
                                          const uint32_t (&v)[ITEMS]) {
    if (aligned && i + ITEMS <= n) {
#pragma unroll
        for (int k = 0; k < ITEMS; k += 4)
            *reinterpret_cast<uint4*>(p + i + k) = make_uint4(v[k], v[k + 1], v[k + 2], v[k + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (i + k < n) p[i + k] = v[k];
    }
}

}  // namespace r2s
