// Volume TV loss (anisotropic, edge-mean normalised; isotropic, voxel-mean
// normalised) and mean-L1 image loss.
// Semantics: r2splat/cuda/csrc/VolumeLossFwd.cu:39-153, VolumeLossBwd.cu:46-115,
// Loss.cpp:115-188, ImageLossFwd.cu:20-31, ImageLossBwd.cu:14-30.
#include "common.hpp"
#include "raster_common.hpp"

#include <type_traits>

namespace r2s {

// The losses stream their buffers: a thread takes VEC consecutive elements of
// a row (16-byte loads; VEC = 1 where a row's length or a pointer is not a
// multiple of 16 bytes), and what bounds them is memory traffic as long as
// three things stay small, each of which the first form of these kernels paid
// for: the sums end in one partial per workgroup (or, without a buffer for
// them, one atomic: same-address atomics retire one every 12.7 ns), so the grid
// is capped (65536 workgroups took 833 us for a 256^3 float volume, the capped
// one 24 us, 5.6 TB/s); row and plane
// indices come from 32-bit divisions per VEC elements instead of 64-bit ones
// per element (anisotropic gradient 91 -> 30 us); and the isotropic gradient
// marches along z, so that a voxel costs 2.25 square roots instead of four
// (126 -> 66 us, and by sharing terms between threads to 54, bound by the
// correctly rounded square roots and divisions).
constexpr int kLossThreads = 256;
constexpr int kSumThreads = 1024;
constexpr uint32_t kSumBlocks = 512;  // two per CU
constexpr uint32_t kMarch = 8;        // planes per thread of the isotropic gradient

template <typename S>
__device__ __forceinline__ S sgn(S x) { return x > S(0) ? S(1) : (x < S(0) ? S(-1) : S(0)); }

// Where a sum goes. With `partials`: each block's entry of them, added in order
// by loss_total_kernel (or, of a single block, at once), which writes the mean
// sum / divisor and the loss lambda mean: no elementwise launches behind the sum
// (both regularisers of a small volume, forward and backward, whose launches are
// the time: 85 -> 61 us; 256^3: 167 -> 154). Without them one atomic per block
// into *sum.
template <typename S>
struct Reduced {
    S* sum;
    double* partials;
    S *mean, *loss;
    double divisor;
    S lambda;
    __device__ __forceinline__ void finish(double t) const {
        const S m = S(t / divisor);
        *mean = m;
        *loss = lambda * m;
    }
};

// Block sum of one value per thread (in double).
template <typename S>
__device__ __forceinline__ void block_sum(S v, const Reduced<S>& out) {
    __shared__ double part[kSumThreads / kWave];
    const double w = wave_sum(double(v));
    if (lane_id() == 0) part[threadIdx.x / kWave] = w;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < kSumThreads / kWave; ++k) t += part[k];
        if (!out.partials) atomic_add(out.sum, S(t));
        else if (gridDim.x == 1) out.finish(t);
        else out.partials[blockIdx.x] = t;
    }
}

// The sum of m <= kSumBlocks partials, in double and a fixed order.
template <typename S>
__global__ void __launch_bounds__(kSumBlocks)
loss_total_kernel(Reduced<S> out, uint32_t m) {
    __shared__ double part[kSumBlocks / kWave];
    const double w = wave_sum(threadIdx.x < m ? out.partials[threadIdx.x] : 0.0);
    if (lane_id() == 0) part[threadIdx.x / kWave] = w;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (uint32_t k = 0; k < kSumBlocks / kWave; ++k) t += part[k];
        out.finish(t);
    }
}

template <typename S, int VEC>
struct __align__(VEC * sizeof(S)) Pack {
    S v[VEC];
};

template <typename S, int VEC>
__device__ __forceinline__ Pack<S, VEC> load_pack(const S* __restrict__ p) {
    return *reinterpret_cast<const Pack<S, VEC>*>(p);
}
template <typename S, int VEC>
__device__ __forceinline__ void store_pack(S* __restrict__ p, const Pack<S, VEC>& x) {
    *reinterpret_cast<Pack<S, VEC>*>(p) = x;
}

// A volume [B, D, H, W] as rows of `quads` = W / VEC packs; I is the index type
// (32-bit unless the pack count needs 64).
template <typename I>
struct Volume {
    I quads, total;  // packs per row, packs in all
    uint32_t D, H, W;
};

// Pack i -> its first element, and its place: x (first column), h, d.
template <typename I, int VEC>
__device__ __forceinline__ size_t locate(const Volume<I>& g, I i, uint32_t& x, uint32_t& h, uint32_t& d) {
    const I row = i / g.quads;
    const I plane = row / I(g.H);
    x = uint32_t(i - row * g.quads) * VEC;
    h = uint32_t(row - plane * I(g.H));
    d = uint32_t(plane % I(g.D));
    return size_t(row) * g.W + x;
}

// One pack's forward differences along z, y and x (0 past the last index of an
// axis); `right` is the element after the pack in its row.
template <typename S, int VEC>
__device__ __forceinline__ void differences(const Pack<S, VEC>& c, const Pack<S, VEC>& zn, const Pack<S, VEC>& yn,
                                            S right, bool has_z, bool has_y, bool has_x, S (&dz)[VEC], S (&dy)[VEC],
                                            S (&dx)[VEC]) {
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        dz[k] = has_z ? zn.v[k] - c.v[k] : S(0);
        dy[k] = has_y ? yn.v[k] - c.v[k] : S(0);
        if (k + 1 < VEC)
            dx[k] = c.v[k + 1 < VEC ? k + 1 : k] - c.v[k];
        else
            dx[k] = has_x ? right - c.v[k] : S(0);
    }
}

// tv_map and its sum: anisotropic |dz| + |dy| + |dx|, or (ISO) the isotropic
// sqrt(dz^2 + dy^2 + dx^2 + eps), with forward differences.
template <typename S, typename I, int VEC, bool ISO>
__global__ void __launch_bounds__(kSumThreads)
tv_fwd_kernel(const S* __restrict__ vol, Volume<I> g, S eps, S* __restrict__ tv_map, Reduced<S> out) {
    S sum = S(0);
    const size_t sd = size_t(g.H) * g.W, sh = g.W;
    for (I i = I(blockIdx.x) * kSumThreads + threadIdx.x; i < g.total; i += I(gridDim.x) * kSumThreads) {
        uint32_t x, h, d;
        const size_t o = locate<I, VEC>(g, i, x, h, d);
        const bool has_z = d + 1 < g.D, has_y = h + 1 < g.H, has_x = x + VEC < g.W;
        const Pack<S, VEC> c = load_pack<S, VEC>(vol + o);
        const Pack<S, VEC> zn = has_z ? load_pack<S, VEC>(vol + o + sd) : c;
        const Pack<S, VEC> yn = has_y ? load_pack<S, VEC>(vol + o + sh) : c;
        const S right = has_x ? vol[o + VEC] : S(0);
        S dz[VEC], dy[VEC], dx[VEC];
        differences<S, VEC>(c, zn, yn, right, has_z, has_y, has_x, dz, dy, dx);
        Pack<S, VEC> t;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            if constexpr (ISO) t.v[k] = sqrt(dz[k] * dz[k] + dy[k] * dy[k] + dx[k] * dx[k] + eps);
            else t.v[k] = fabs(dz[k]) + fabs(dy[k]) + fabs(dx[k]);
            sum += t.v[k];
        }
        store_pack<S, VEC>(tv_map + o, t);
    }
    block_sum(sum, out);
}

// grad = ((sign sum) * (g / edges)) * lambda: the reference's rounding order
// (the kernel's g / edges product, then the host-side multiply by lambda).
template <typename S, typename I, int VEC>
__global__ void __launch_bounds__(kLossThreads)
tv_bwd_kernel(const S* __restrict__ vol, const S* __restrict__ grad_out, Volume<I> g, S edges, S lambda,
              S* __restrict__ grad) {
    const I i = I(blockIdx.x) * kLossThreads + threadIdx.x;
    if (i >= g.total) return;
    uint32_t x, h, d;
    const size_t o = locate<I, VEC>(g, i, x, h, d), sd = size_t(g.H) * g.W, sh = g.W;
    const bool has_zn = d + 1 < g.D, has_zp = d > 0, has_yn = h + 1 < g.H, has_yp = h > 0;
    const Pack<S, VEC> c = load_pack<S, VEC>(vol + o);
    // a missing neighbour equals the voxel: its sign is 0
    const Pack<S, VEC> zn = has_zn ? load_pack<S, VEC>(vol + o + sd) : c;
    const Pack<S, VEC> zp = has_zp ? load_pack<S, VEC>(vol + o - sd) : c;
    const Pack<S, VEC> yn = has_yn ? load_pack<S, VEC>(vol + o + sh) : c;
    const Pack<S, VEC> yp = has_yp ? load_pack<S, VEC>(vol + o - sh) : c;
    const bool has_xn = x + VEC < g.W, has_xp = x > 0;
    const S right = has_xn ? vol[o + VEC] : S(0), left = has_xp ? vol[o - 1] : S(0);
    const S per_edge = grad_out[0] / edges;
    Pack<S, VEC> out;
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        const S v = c.v[k];
        S s = S(0);
        if (has_zn) s -= sgn(zn.v[k] - v);
        if (has_zp) s += sgn(v - zp.v[k]);
        if (has_yn) s -= sgn(yn.v[k] - v);
        if (has_yp) s += sgn(v - yp.v[k]);
        if (k + 1 < VEC) s -= sgn(c.v[k + 1 < VEC ? k + 1 : k] - v);
        else if (has_xn) s -= sgn(right - v);
        if (k > 0) s += sgn(v - c.v[k > 0 ? k - 1 : k]);
        else if (has_xp) s += sgn(v - left);
        out.v[k] = (s * per_edge) * lambda;
    }
    store_pack<S, VEC>(grad + o, out);
}

// d/dV(v) of sum_u t(u), t the isotropic term: -(dz + dy + dx)(v) / t(v) plus
// dz(v - ez) / t(v - ez), dy(v - ey) / t(v - ey) and dx(v - ex) / t(v - ex)
// where those voxels exist. A thread takes a pack's column over kMarch planes:
// plane d's dz / t is what plane d + 1 needs, a pack's last dx / t what the next
// lane needs, and its dy / t what the thread of the row above needs (through LDS,
// `quads` threads on), so that a voxel costs one correctly rounded square root and
// four divisions, which bound the kernel; only a workgroup's first row, a wave's
// first lane and a march's first plane evaluate a neighbour's terms (each thread
// evaluating its neighbours: 67 us for 256^3 floats, now 54). `total` counts
// (plane chunk, row, pack).
constexpr int kMarchThreads = 512;

template <typename S, typename I, int VEC>
__global__ void __launch_bounds__(kMarchThreads)
tv_iso_bwd_kernel(const S* __restrict__ vol, const S* __restrict__ grad_out, Volume<I> g, uint32_t chunks, S eps,
                  S scale, S* __restrict__ grad) {
    __shared__ Pack<S, VEC> shared_y[2][kMarchThreads];  // dy / t, by the parity of the plane
    const I mine = I(blockIdx.x) * kMarchThreads + threadIdx.x;
    const bool valid = mine < g.total;  // (the others repeat the last pack and store nothing)
    const I i = valid ? mine : g.total - 1;
    const I row = i / g.quads, slab = row / I(g.H);
    const uint32_t x = uint32_t(i - row * g.quads) * VEC, h = uint32_t(row - slab * I(g.H));
    const I b = slab / I(chunks);
    const uint32_t d0 = uint32_t(slab - b * I(chunks)) * kMarch, d1 = min(g.D, d0 + kMarch);
    const size_t sd = size_t(g.H) * g.W, sh = g.W;
    const bool has_yn = h + 1 < g.H, has_yp = h > 0, has_xn = x + VEC < g.W, has_xp = x > 0;
    // the threads of the packs to the left and in the row above, if in this wave and workgroup
    const bool left_lane = valid && has_xp && threadIdx.x % kWave != 0;
    const bool row_thread = valid && has_yp && I(threadIdx.x) >= g.quads;
    const S gs = grad_out[0] * scale;
    size_t o = ((size_t(b) * g.D + d0) * g.H + h) * g.W + x;
    Pack<S, VEC> c = load_pack<S, VEC>(vol + o);
    S below[VEC];  // dz / t of the plane below
#pragma unroll
    for (int k = 0; k < VEC; ++k) below[k] = S(0);
    if (d0 > 0) {
        const size_t q = o - sd;
        const Pack<S, VEC> p = load_pack<S, VEC>(vol + q);
        const Pack<S, VEC> yn = has_yn ? load_pack<S, VEC>(vol + q + sh) : p;
        const S right = has_xn ? vol[q + VEC] : S(0);
        S dz[VEC], dy[VEC], dx[VEC];
        differences<S, VEC>(p, c, yn, right, true, has_yn, has_xn, dz, dy, dx);
#pragma unroll
        for (int k = 0; k < VEC; ++k) below[k] = dz[k] / sqrt(dz[k] * dz[k] + dy[k] * dy[k] + dx[k] * dx[k] + eps);
    }
    for (uint32_t step = 0; step < kMarch; ++step, o += sd) {  // every thread takes every step: barriers
        const uint32_t d = d0 + step;
        const bool active = d < d1;
        Pack<S, VEC> zn = c, yt;
        S out[VEC], xt[VEC], carry_x = S(0);  // -(dz + dy + dx) / t, dx / t; dx / t of the voxel to the left
        const bool has_z = d + 1 < g.D;
        if (active) {
            if (has_z) zn = load_pack<S, VEC>(vol + o + sd);
            const Pack<S, VEC> yn = has_yn ? load_pack<S, VEC>(vol + o + sh) : c;
            const S right = has_xn ? vol[o + VEC] : S(0);
            S dz[VEC], dy[VEC], dx[VEC];
            differences<S, VEC>(c, zn, yn, right, has_z, has_yn, has_xn, dz, dy, dx);
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                const S t = sqrt(dz[k] * dz[k] + dy[k] * dy[k] + dx[k] * dx[k] + eps);
                out[k] = -(dz[k] + dy[k] + dx[k]) / t;
                out[k] += below[k];
                below[k] = dz[k] / t;
                yt.v[k] = dy[k] / t;
                xt[k] = dx[k] / t;
            }
            shared_y[step % 2][threadIdx.x] = yt;
            carry_x = __shfl_up(xt[VEC - 1], 1, kWave);  // (the left pack's lane takes the same steps)
            if (!left_lane) {
                carry_x = S(0);
                if (has_xp) {
                    const S l = vol[o - 1];
                    const S lz = has_z ? vol[o + sd - 1] - l : S(0), ly = has_yn ? vol[o + sh - 1] - l : S(0);
                    const S lx = c.v[0] - l;
                    carry_x = lx / sqrt(lz * lz + ly * ly + lx * lx + eps);
                }
            }
        }
        __syncthreads();  // (the other buffer's readers passed it before the last one)
        if (active) {
            S from_y[VEC];  // dy / t of the voxel at y - 1
#pragma unroll
            for (int k = 0; k < VEC; ++k) from_y[k] = S(0);
            if (row_thread) {
                const Pack<S, VEC> p = shared_y[step % 2][threadIdx.x - uint32_t(g.quads)];
#pragma unroll
                for (int k = 0; k < VEC; ++k) from_y[k] = p.v[k];
            } else if (has_yp) {
                const size_t q = o - sh;
                const Pack<S, VEC> p = load_pack<S, VEC>(vol + q);
                const Pack<S, VEC> pz = has_z ? load_pack<S, VEC>(vol + q + sd) : p;
                const S pr = has_xn ? vol[q + VEC] : S(0);
                S az[VEC], ay[VEC], ax[VEC];
                differences<S, VEC>(p, pz, c, pr, has_z, true, has_xn, az, ay, ax);
#pragma unroll
                for (int k = 0; k < VEC; ++k)
                    from_y[k] = ay[k] / sqrt(az[k] * az[k] + ay[k] * ay[k] + ax[k] * ax[k] + eps);
            }
            Pack<S, VEC> w;
#pragma unroll
            for (int k = 0; k < VEC; ++k) {
                S s = out[k];
                s += from_y[k];
                s += k > 0 ? xt[k > 0 ? k - 1 : 0] : carry_x;
                w.v[k] = s * gs;
            }
            if (valid) store_pack<S, VEC>(grad + o, w);
            c = zn;
        }
    }
}

template <typename S, int VEC>
__global__ void __launch_bounds__(kSumThreads)
l1_fwd_kernel(const S* __restrict__ p, const S* __restrict__ t, uint64_t n, S* __restrict__ map,
              Reduced<S> out) {
    S s = S(0);
    for (uint64_t i = uint64_t(blockIdx.x) * kSumThreads + threadIdx.x; i < n / VEC;
         i += uint64_t(gridDim.x) * kSumThreads) {
        const Pack<S, VEC> a = load_pack<S, VEC>(p + i * VEC), b = load_pack<S, VEC>(t + i * VEC);
        Pack<S, VEC> m;
#pragma unroll
        for (int k = 0; k < VEC; ++k) {
            m.v[k] = fabs(a.v[k] - b.v[k]);
            s += m.v[k];
        }
        store_pack<S, VEC>(map + i * VEC, m);
    }
    block_sum(s, out);
}

template <typename S>
__global__ void __launch_bounds__(kLossThreads)
l1_bwd_kernel(const S* __restrict__ p, const S* __restrict__ t, const S* __restrict__ g, uint64_t n,
              S lambda, S* __restrict__ out) {
    const size_t idx = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    out[idx] = g[0] * lambda * sgn(p[idx] - t[idx]) / S(n);  // the reference's operation order
}

// Whether `length` and the pointers allow 16-byte packs of S.
template <typename S>
static bool packed16(uint64_t length, const void* a, const void* b, const void* c = nullptr) {
    const uintptr_t bits = reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) |
                           reinterpret_cast<uintptr_t>(c);
    return length % (16 / sizeof(S)) == 0 && bits % 16 == 0;
}

static uint32_t sum_blocks(uint64_t items) {
    return std::min<uint32_t>(kSumBlocks, std::max<uint32_t>(1u, ceil_div(items, kSumThreads)));
}

// Calls f(I{}, std::integral_constant<int, VEC>{}) with the pack width that W
// and the pointers allow and 32-bit indices where `rows` packed rows fit them
// (grid-stride loops step up to 2^19 past the last index).
template <typename S, typename F>
static int with_packs(uint64_t rows, uint32_t W, const void* a, const void* b, F&& f) {
    constexpr int kWide = 16 / int(sizeof(S));
    const bool wide = packed16<S>(W, a, b);
    const bool small = rows * (wide ? W / kWide : W) < (1ull << 32) - (1ull << 20);
    if (wide && small) return f(uint32_t{}, std::integral_constant<int, kWide>{});
    if (wide) return f(uint64_t{}, std::integral_constant<int, kWide>{});
    if (small) return f(uint32_t{}, std::integral_constant<int, 1>{});
    return f(uint64_t{}, std::integral_constant<int, 1>{});
}

// A loss forward's outputs as the entry points take them.
struct LossOutputs {
    void* sum;
    double* partials;
    void *mean, *loss;
    double divisor, lambda;
    template <typename S>
    Reduced<S> as() const {
        return {static_cast<S*>(sum), partials, static_cast<S*>(mean), static_cast<S*>(loss), divisor, S(lambda)};
    }
};

// Before the sum: cleared where blocks add to it, finished where there are none.
template <typename S>
static int begin_sum(const Reduced<S>& out, uint64_t total, hipStream_t stream, const char* where) {
    if (!out.partials) return fill_zero<S>(out.sum, 1, stream);
    if (total == 0) loss_total_kernel<S><<<1, kSumBlocks, 0, stream>>>(out, 0);
    return check_launch(where);
}
template <typename S>
static int end_sum(const Reduced<S>& out, uint32_t blocks, hipStream_t stream, const char* where) {
    if (out.partials && blocks > 1) loss_total_kernel<S><<<1, kSumBlocks, 0, stream>>>(out, blocks);
    return check_launch(where);
}

static int tv_fwd(int dtype, bool iso, const void* volume, uint32_t B, uint32_t D, uint32_t H, uint32_t W, double eps,
                  void* tv_map, const LossOutputs& outputs, hipStream_t stream, const char* where) {
    const uint64_t rows = uint64_t(B) * D * H;
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        const S* vol = (const S*)volume;
        const Reduced<S> out = outputs.as<S>();
        if (int rc = begin_sum<S>(out, rows * W, stream, where)) return rc;
        if (rows * W == 0) return R2S_OK;
        return with_packs<S>(rows, W, volume, tv_map, [&](auto index, auto vec) {
            using I = decltype(index);
            constexpr int VEC = decltype(vec)::value;
            const Volume<I> g{I(W / VEC), I(rows * (W / VEC)), D, H, W};
            const uint32_t blocks = sum_blocks(g.total);
            auto k = iso ? tv_fwd_kernel<S, I, VEC, true> : tv_fwd_kernel<S, I, VEC, false>;
            k<<<blocks, kSumThreads, 0, stream>>>(vol, g, S(eps), (S*)tv_map, out);
            if (int rc = check_launch(where)) return rc;
            return end_sum<S>(out, blocks, stream, where);
        });
    });
}

static int l1_fwd(int dtype, const void* prediction, const void* target, uint64_t n, void* l1_map,
                  const LossOutputs& outputs, hipStream_t stream) {
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        constexpr int kWide = 16 / int(sizeof(S));
        const Reduced<S> out = outputs.as<S>();
        if (int rc = begin_sum<S>(out, n, stream, "image_l1_fwd")) return rc;
        if (n == 0) return R2S_OK;
        const bool wide = packed16<S>(n, prediction, target, l1_map);
        const uint32_t blocks = sum_blocks(wide ? n / kWide : n);
        auto k = wide ? l1_fwd_kernel<S, kWide> : l1_fwd_kernel<S, 1>;
        k<<<blocks, kSumThreads, 0, stream>>>((const S*)prediction, (const S*)target, n, (S*)l1_map, out);
        if (int rc = check_launch("image_l1_fwd")) return rc;
        return end_sum<S>(out, blocks, stream, "image_l1_fwd");
    });
}

}  // namespace r2s

using namespace r2s;

extern "C" int r2s_volume_tv_fwd(int dtype, const void* volume, uint32_t B, uint32_t D, uint32_t H,
                                 uint32_t W, void* tv_map, void* tv_sum, r2s_stream_t stream) {
    return tv_fwd(dtype, false, volume, B, D, H, W, 0.0, tv_map, {tv_sum}, stream, "volume_tv_fwd");
}

extern "C" int r2s_volume_tv_bwd(int dtype, const void* volume, const void* grad_output, uint32_t B,
                                 uint32_t D, uint32_t H, uint32_t W, float lambda_tv,
                                 void* grad_volume, r2s_stream_t stream) {
    const size_t total = size_t(B) * D * H * W;
    if (total == 0) return R2S_OK;
    const int64_t edges64 = int64_t(B) * ((int64_t(D) - 1) * H * W + int64_t(D) * (H - 1) * W +
                                          int64_t(D) * H * (W - 1));
    const int64_t edges = edges64 < 1 ? 1 : edges64;
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        const uint64_t rows = uint64_t(B) * D * H;
        return with_packs<S>(rows, W, volume, grad_volume, [&](auto index, auto vec) {
            using I = decltype(index);
            constexpr int VEC = decltype(vec)::value;
            const Volume<I> g{I(W / VEC), I(rows * (W / VEC)), D, H, W};
            tv_bwd_kernel<S, I, VEC><<<ceil_div(g.total, kLossThreads), kLossThreads, 0, stream>>>(
                (const S*)volume, (const S*)grad_output, g, S(edges), S(lambda_tv), (S*)grad_volume);
            return check_launch("volume_tv_bwd");
        });
    });
}

extern "C" int r2s_volume_tv_iso_fwd(int dtype, const void* volume, uint32_t B, uint32_t D, uint32_t H,
                                     uint32_t W, double eps, void* tv_map, void* tv_sum, r2s_stream_t stream) {
    R2S_REQUIRE(eps > 0.0, "isotropic TV needs eps > 0 (got %g)", eps);
    return tv_fwd(dtype, true, volume, B, D, H, W, eps, tv_map, {tv_sum}, stream, "volume_tv_iso_fwd");
}

extern "C" int r2s_volume_tv_iso_bwd(int dtype, const void* volume, const void* grad_output, uint32_t B,
                                     uint32_t D, uint32_t H, uint32_t W, double eps, double lambda_tv,
                                     void* grad_volume, r2s_stream_t stream) {
    R2S_REQUIRE(eps > 0.0, "isotropic TV needs eps > 0 (got %g)", eps);
    const size_t total = size_t(B) * D * H * W;
    if (total == 0) return R2S_OK;
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        const uint32_t chunks = ceil_div(D, kMarch);
        const uint64_t rows = uint64_t(B) * chunks * H;  // one per (plane chunk, row)
        return with_packs<S>(rows, W, volume, grad_volume, [&](auto index, auto vec) {
            using I = decltype(index);
            constexpr int VEC = decltype(vec)::value;
            const Volume<I> g{I(W / VEC), I(rows * (W / VEC)), D, H, W};
            tv_iso_bwd_kernel<S, I, VEC><<<ceil_div(g.total, kMarchThreads), kMarchThreads, 0, stream>>>(
                (const S*)volume, (const S*)grad_output, g, chunks, S(eps), S(lambda_tv / double(total)),
                (S*)grad_volume);
            return check_launch("volume_tv_iso_bwd");
        });
    });
}

extern "C" int r2s_image_l1_fwd(int dtype, const void* prediction, const void* target, uint64_t n,
                                void* l1_map, void* l1_sum, r2s_stream_t stream) {
    return l1_fwd(dtype, prediction, target, n, l1_map, {l1_sum}, stream);
}

extern "C" int r2s_image_l1_bwd(int dtype, const void* prediction, const void* target,
                                const void* grad_output, uint64_t n, float lambda_l1,
                                void* grad_prediction, r2s_stream_t stream) {
    if (n == 0) return R2S_OK;
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        l1_bwd_kernel<S><<<ceil_div(n, kLossThreads), kLossThreads, 0, stream>>>(
            (const S*)prediction, (const S*)target, (const S*)grad_output, n, S(lambda_l1),
            (S*)grad_prediction);
        return check_launch("image_l1_bwd");
    });
}

extern "C" size_t r2s_loss_partials_bytes(void) { return kSumBlocks * sizeof(double); }

extern "C" int r2s_volume_tv_fwd_ordered(int dtype, int isotropic, const void* volume, uint32_t B, uint32_t D,
                                         uint32_t H, uint32_t W, double eps, double divisor, double lambda,
                                         void* tv_map, void* tv, void* loss, void* partials,
                                         r2s_stream_t stream) {
    R2S_REQUIRE(partials && tv && loss, "volume_tv_fwd_ordered: tv, loss and partials are required");
    R2S_REQUIRE(!isotropic || eps > 0.0, "isotropic TV needs eps > 0 (got %g)", eps);
    return tv_fwd(dtype, isotropic != 0, volume, B, D, H, W, eps, tv_map,
                  {nullptr, static_cast<double*>(partials), tv, loss, divisor, lambda}, stream,
                  "volume_tv_fwd_ordered");
}

extern "C" int r2s_image_l1_fwd_ordered(int dtype, const void* prediction, const void* target, uint64_t n,
                                        double divisor, double lambda, void* l1_map, void* l1, void* loss,
                                        void* partials, r2s_stream_t stream) {
    R2S_REQUIRE(partials && l1 && loss, "image_l1_fwd_ordered: l1, loss and partials are required");
    return l1_fwd(dtype, prediction, target, n, l1_map,
                  {nullptr, static_cast<double*>(partials), l1, loss, divisor, lambda}, stream);
}
