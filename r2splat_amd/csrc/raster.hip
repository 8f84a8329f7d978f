// 2D CT rasterization: each pixel sums opacity * mu * profile over the
// primitives binned to its tile (additive line integrals, no compositing).
//
// Operator-level kernels for every tile size and both float/double:
//  * tile-parallel forward (mean, mean+variance): tiles of 8, 16 and 32 pixels
//    share their list over several waves and skip the rows a primitive does not
//    reach; other sizes stage the list through LDS in batches, a pixel per thread;
//  * tile-parallel ("pixel" mode) VJP and the uncertainty VJP: one wave64
//    reduction per (wave, primitive) followed by one atomic per field;
//  * intersection-parallel ("primitive" mode) VJP: tiles of 8, 16 and 32 pixels
//    one lane per intersection, walking the rows it reaches; other sizes and
//    absolute gradients one wave64 per intersection, lanes striding the tile's
//    pixels; one atomic per field.
// Profiles follow r2splat/cuda/csrc/RasterizeToPixelsFwd.cu:155-180 (Gaussian)
// and :664-680 (Beta), and the VJPs RasterizeToPixelsBwd.cu:169-265,421-501,
// 674-706,909-945.
#include "common.hpp"
#include "raster_common.hpp"
#include "sorted_chunk.hpp"

#include <type_traits>

namespace r2s {

constexpr uint32_t kBatch = 256;

template <typename S>
struct PrimLDS {
    S* mx; S* my; S* a; S* b; S* c; S* opac; S* mu; S* beta; S* q; int32_t* id;
};

template <typename S>
__device__ __forceinline__ PrimLDS<S> carve_lds(unsigned char* smem, uint32_t batch) {
    PrimLDS<S> p;
    S* f = reinterpret_cast<S*>(smem);
    p.mx = f; p.my = f + batch; p.a = f + 2 * batch; p.b = f + 3 * batch; p.c = f + 4 * batch;
    p.opac = f + 5 * batch; p.mu = f + 6 * batch; p.beta = f + 7 * batch; p.q = f + 8 * batch;
    p.id = reinterpret_cast<int32_t*>(f + 9 * batch);
    return p;
}

inline size_t lds_bytes(int dtype, uint32_t batch) {
    const size_t s = dtype == R2S_F64 ? 8 : 4;
    return batch * (9 * s + 4);
}

template <typename S>
struct RasterArgs {
    const S* means2d; const S* conics; const S* opac; const S* mus; const S* betas; const S* unc;
    const int32_t* offsets; const int32_t* flatten; uint32_t n_isects, C, N, W, H, T, ntx, nty;
};

// Decodes block -> (camera, tile) and returns the tile's [start, end) range.
template <typename S>
__device__ __forceinline__ void tile_range(const RasterArgs<S>& A, uint32_t blk, uint32_t& cam,
                                           uint32_t& ty, uint32_t& tx, int32_t& start, int32_t& end) {
    const uint32_t nt = A.ntx * A.nty;
    cam = blk / nt;
    const uint32_t tile = blk - cam * nt;
    ty = tile / A.ntx;
    tx = tile - ty * A.ntx;
    const uint64_t key = uint64_t(cam) * nt + tile;
    start = A.offsets[key];
    end = (key + 1 == uint64_t(A.C) * nt) ? int32_t(A.n_isects) : A.offsets[key + 1];
    start = max(0, min(start, int32_t(A.n_isects)));
    end = max(start, min(end, int32_t(A.n_isects)));
}

template <typename S, bool BETA, bool VAR>
__device__ __forceinline__ void stage_batch(const RasterArgs<S>& A, const PrimLDS<S>& L, int32_t b0,
                                            int32_t end, uint32_t batch) {
    const uint32_t t = threadIdx.x;
    if (t < batch && b0 + int32_t(t) < end) {
        int32_t g = A.flatten[b0 + t];
        const bool ok = g >= 0 && uint32_t(g) < A.C * A.N;
        if (!ok) g = 0;  // out-of-range ids contribute nothing
        L.id[t] = g;
        L.mx[t] = A.means2d[2 * size_t(g)];
        L.my[t] = A.means2d[2 * size_t(g) + 1];
        L.a[t] = A.conics[3 * size_t(g)];
        L.b[t] = A.conics[3 * size_t(g) + 1];
        L.c[t] = A.conics[3 * size_t(g) + 2];
        L.opac[t] = ok ? A.opac[g] : S(0);
        L.mu[t] = A.mus[g];
        if (BETA) L.beta[t] = A.betas[g];
        if (VAR) L.q[t] = A.unc[uint32_t(g) % A.N];
    }
}

template <typename S, bool BETA>
__device__ __forceinline__ Prim2D<S> lds_prim(const PrimLDS<S>& L, uint32_t t) {
    Prim2D<S> p;
    p.mx = L.mx[t]; p.my = L.my[t]; p.a = L.a[t]; p.b = L.b[t]; p.c = L.c[t];
    p.opac = L.opac[t]; p.mu = L.mu[t]; p.beta = BETA ? L.beta[t] : S(0);
    return p;
}

// ---------------------------------------------------------------------------
// Forward (mean, optional variance). Block = one tile, T*T threads.
// ---------------------------------------------------------------------------
template <typename S, bool BETA, bool VAR>
__global__ void raster_fwd_kernel(RasterArgs<S> A, S* __restrict__ out, S* __restrict__ out_var) {
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t batch = min(blockDim.x, kBatch);
    PrimLDS<S> L = carve_lds<S>(smem, batch);
    uint32_t cam, ty, tx;
    int32_t start, end;
    tile_range(A, blockIdx.x, cam, ty, tx, start, end);
    const uint32_t i = ty * A.T + threadIdx.x / A.T;
    const uint32_t j = tx * A.T + threadIdx.x % A.T;
    const bool inside = (threadIdx.x < A.T * A.T) && i < A.H && j < A.W;
    const S px = S(j) + S(0.5), py = S(i) + S(0.5);
    S acc = S(0), acc_var = S(0);
    for (int32_t b0 = start; b0 < end; b0 += int32_t(batch)) {
        __syncthreads();
        stage_batch<S, BETA, VAR>(A, L, b0, end, batch);
        __syncthreads();
        if (!inside) continue;
        const uint32_t cnt = uint32_t(min<int32_t>(int32_t(batch), end - b0));
        for (uint32_t t = 0; t < cnt; ++t) {
            const Prim2D<S> p = lds_prim<S, BETA>(L, t);
            S vis, alpha;
            if (!eval_profile<S, BETA>(p, px, py, vis, alpha)) continue;
            acc += alpha;
            if (VAR) acc_var += L.q[t] * alpha * alpha;
        }
    }
    if (inside) {
        const size_t o = (size_t(cam) * A.H + i) * A.W + j;
        out[o] = acc;
        if (VAR) out_var[o] = acc_var;
    }
}

// ---------------------------------------------------------------------------
// Tile-parallel VJPs. MODE 0: mean VJP (pixel mode); MODE 1: uncertainty VJP.
// ---------------------------------------------------------------------------
template <typename S, bool BETA, int MODE>
__global__ void raster_bwd_tile_kernel(RasterArgs<S> A, const S* __restrict__ v_render,
                                       S* __restrict__ v_abs, S* __restrict__ v_xy,
                                       S* __restrict__ v_conic, S* __restrict__ v_opac,
                                       S* __restrict__ v_mu, S* __restrict__ v_beta,
                                       S* __restrict__ v_q) {
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t batch = min(blockDim.x, kBatch);
    PrimLDS<S> L = carve_lds<S>(smem, batch);
    uint32_t cam, ty, tx;
    int32_t start, end;
    tile_range(A, blockIdx.x, cam, ty, tx, start, end);
    const uint32_t i = ty * A.T + threadIdx.x / A.T;
    const uint32_t j = tx * A.T + threadIdx.x % A.T;
    const bool inside = (threadIdx.x < A.T * A.T) && i < A.H && j < A.W;
    const S px = S(j) + S(0.5), py = S(i) + S(0.5);
    const S v = inside ? v_render[(size_t(cam) * A.H + i) * A.W + j] : S(0);
    const bool lane0 = lane_id() == 0;
    for (int32_t b0 = start; b0 < end; b0 += int32_t(batch)) {
        __syncthreads();
        stage_batch<S, BETA, false>(A, L, b0, end, batch);
        __syncthreads();
        const uint32_t cnt = uint32_t(min<int32_t>(int32_t(batch), end - b0));
        for (uint32_t t = 0; t < cnt; ++t) {
            const Prim2D<S> p = lds_prim<S, BETA>(L, t);
            S vis = S(0), alpha = S(0);
            const bool valid = inside && eval_profile<S, BETA>(p, px, py, vis, alpha);
            const int32_t g = L.id[t];
            if (MODE == 1) {
                const S s = wave_sum(valid ? v * alpha * alpha : S(0));
                if (lane0) atomic_add(v_q + uint32_t(g) % A.N, s);
                continue;
            }
            Grad2D<S> gr;
            if (valid) pixel_vjp<S, BETA>(p, px, py, vis, alpha, v, gr);
            gr.reduce_wave(v_abs != nullptr);
            if (lane0) gr.commit(g, v_abs, v_xy, v_conic, v_opac, v_mu, v_beta);
        }
    }
}

// ---------------------------------------------------------------------------
// Intersection-parallel VJP: one wave64 per intersection.
// ---------------------------------------------------------------------------
template <typename S, bool BETA>
__global__ void __launch_bounds__(256)
raster_bwd_isect_kernel(RasterArgs<S> A, const int64_t* __restrict__ isect_ids,
                        const S* __restrict__ v_render, const S* __restrict__ v_var,
                        const S* __restrict__ unc, S* __restrict__ v_abs, S* __restrict__ v_xy,
                        S* __restrict__ v_conic, S* __restrict__ v_opac, S* __restrict__ v_mu,
                        S* __restrict__ v_beta, S* __restrict__ v_q) {
    // grid-stride over intersections (one wave each): a launch covers at most
    // kIsectBlocks blocks, whatever the intersection count
    const uint32_t waves = blockDim.x / kWave;
    const uint64_t stride = uint64_t(gridDim.x) * waves;
    for (uint64_t e = uint64_t(blockIdx.x) * waves + threadIdx.x / kWave; e < A.n_isects; e += stride) {
        const uint32_t nt = A.ntx * A.nty;
        const int64_t key = isect_ids[e];
        const uint32_t cam = uint32_t(key / nt);
        if (cam >= A.C) continue;
        const uint32_t tile = uint32_t(key - int64_t(cam) * nt);
        const uint32_t ty = tile / A.ntx, tx = tile - (tile / A.ntx) * A.ntx;
        const int32_t g = A.flatten[e];
        if (g < 0 || uint32_t(g) >= A.C * A.N) continue;
        Prim2D<S> p;
        p.mx = A.means2d[2 * size_t(g)];
        p.my = A.means2d[2 * size_t(g) + 1];
        p.a = A.conics[3 * size_t(g)];
        p.b = A.conics[3 * size_t(g) + 1];
        p.c = A.conics[3 * size_t(g) + 2];
        p.opac = A.opac[g];
        p.mu = A.mus[g];
        p.beta = BETA ? A.betas[g] : S(0);
        const uint32_t n = uint32_t(g) % A.N;
        const S q = unc ? unc[n] : S(0);
        const size_t img = size_t(cam) * A.H * A.W;
        Grad2D<S> gr;
        S vq = S(0);
        const uint32_t npix = A.T * A.T;
        for (uint32_t k = lane_id(); k < npix; k += kWave) {
            const uint32_t ly = k / A.T, lx = k - ly * A.T;
            const uint32_t i = ty * A.T + ly, j = tx * A.T + lx;
            if (i >= A.H || j >= A.W) continue;
            const S px = S(j) + S(0.5), py = S(i) + S(0.5);
            S vis, alpha;
            if (!eval_profile<S, BETA>(p, px, py, vis, alpha)) continue;
            const size_t o = img + size_t(i) * A.W + j;
            S v = v_render[o];
            if (v_var) {
                const S vv = v_var[o];
                vq += vv * alpha * alpha;
                if (unc) v += S(2) * q * alpha * vv;
            }
            pixel_vjp<S, BETA>(p, px, py, vis, alpha, v, gr);
        }
        gr.reduce_wave(v_abs != nullptr);
        if (v_q) vq = wave_sum(vq);
        if (lane_id() == 0) {
            gr.commit(g, v_abs, v_xy, v_conic, v_opac, v_mu, v_beta);
            if (v_q) atomic_add(v_q + n, vq);
        }
    }
}

// ---------------------------------------------------------------------------
// Tiles of T = 8, 16 and 32 pixels: forward and per-intersection VJP that
// evaluate only the rows of a tile a primitive can reach. In double precision
// the exponential (and, for Beta primitives, the power) is most of a pair's
// cost, so rows outside the footprint are what there is to save: 20k Gaussians
// on 8 views of 128^2 touch 9.8 of 16 rows per tile. A pixel per thread over
// the whole list took 688 us there (four waves a tile, two a SIMD), a wave per
// intersection with its nine wave reductions 494 us; these take 144 and 157. What
// bounds them is double arithmetic in the few tiles that the object covers.
// ---------------------------------------------------------------------------
// Whether every parameter of a primitive is finite.
template <typename S, bool BETA>
__device__ __forceinline__ bool all_finite(const Prim2D<S>& p) {
    return isfinite(p.mx) && isfinite(p.my) && isfinite(p.a) && isfinite(p.b) && isfinite(p.c) && isfinite(p.opac) &&
           isfinite(p.mu) && (!BETA || isfinite(p.beta));
}

// Rows [lo, hi) of a T-row tile (first pixel centre at row y_base + 1/2) in which
// |alpha| can reach 1e-5: dy^2 <= 4 A S / (4 A C - B^2) for the form A dx^2 + B dx
// dy + C dy^2 <= S, widened by 1e-3 and 0.05 px (the bound is formed in float).
// Forms that are flat, not positive definite or not finite get every row, and so do
// means that are not finite: their NaN shows where their pairs pass the cut-off. Only
// a finite primitive whose weight is surely below it gets none.
template <typename S, bool BETA>
__device__ __forceinline__ void reached_rows(const Prim2D<S>& p, S y_base, int T, int& lo, int& hi) {
    lo = 0;
    hi = T;
    const float w = fabsf(float(p.opac * p.mu));
    if (w < 0.999e-5f) {
        hi = all_finite<S, BETA>(p) ? 0 : T;
        return;
    }
    float A, B, C, bound;
    if (BETA) {
        A = float(p.a);
        B = 2.f * float(p.b);
        C = float(p.c);
        const float D = 1.f - __builtin_amdgcn_exp2f(__log2f(1e-5f / w) / float(p.beta));
        bound = p.beta > S(0) ? fminf(1.f, 1.002f * D + 1e-4f) : 1.f;
    } else {
        A = 0.5f * float(p.a);
        B = float(p.b);
        C = 0.5f * float(p.c);
        bound = 1.001f * __logf(w * 1e5f) + 1e-4f;
    }
    const float ac4 = 4.f * A * C, den = ac4 - B * B;
    const float e2 = 4.f * A * bound * __builtin_amdgcn_rcpf(den);
    if (!(A > 0.f) || !(den > 1e-3f * ac4) || !(e2 >= 0.f) || !(e2 < 1e30f)) return;
    const float ext = __builtin_amdgcn_sqrtf(e2) * 1.001f + 0.05f;
    const float c = float(p.my - y_base) - 0.5f;
    if (!(fabsf(c) < 1e9f) || !(fabsf(float(p.mx)) < 1e30f)) return;
    lo = int(fminf(fmaxf(ceilf(c - ext), 0.f), float(T)));
    hi = max(lo, int(fminf(fmaxf(floorf(c + ext) + 1.f, 0.f), float(T))));
}

// Columns [lo, hi) in which |alpha| can reach 1e-5: reached_rows with x and y exchanged.
template <typename S, bool BETA>
__device__ __forceinline__ void reached_cols(const Prim2D<S>& p, S x_base, int T, int& lo, int& hi) {
    Prim2D<S> t = p;
    t.mx = p.my;
    t.my = p.mx;
    t.a = p.c;
    t.c = p.a;
    reached_rows<S, BETA>(t, x_base, T, lo, hi);
}

// The form at a pixel, from a dx, dx, b dx (twice that for Beta), c and dy, in the
// roundings eval_profile compiles to: a thin footprint's float32 terms cancel, and any other order would give
// such a primitive an exponent that differs from the general kernel's.
template <typename S, bool BETA>
__device__ __forceinline__ S pair_form(S adx, S dx, S bdx, S c, S dy) {
    if constexpr (BETA) return Math<S>::fma(c * dy, dy, Math<S>::fma(adx, dx, bdx * dy));
    return Math<S>::fma(bdx, dy, S(0.5) * Math<S>::fma(adx, dx, c * dy * dy));
}

// The Gaussian VJP's form. The general VJP rounds the other square first, and a thin
// footprint's gradient keeps that float32 exponent.
template <typename S>
__device__ __forceinline__ S vjp_sigma(S adx, S dx, S bdx, S c, S dy) {
    if constexpr (sizeof(S) == sizeof(double)) return pair_form<S, false>(adx, dx, bdx, c, dy);
    return Math<S>::fma(bdx, dy, S(0.5) * Math<S>::fma(c * dy, dy, adx * dx));
}

template <typename S>
__device__ __forceinline__ Prim2D<S> load_prim(const RasterArgs<S>& A, int32_t g, bool beta) {
    Prim2D<S> p;
    p.mx = A.means2d[2 * size_t(g)];
    p.my = A.means2d[2 * size_t(g) + 1];
    p.a = A.conics[3 * size_t(g)];
    p.b = A.conics[3 * size_t(g) + 1];
    p.c = A.conics[3 * size_t(g) + 2];
    p.opac = A.opac[g];
    p.mu = A.mus[g];
    p.beta = beta ? A.betas[g] : S(0);
    return p;
}

// Forward: WAVES waves share a tile, wave k taking batches k, k + WAVES, ... of 64
// records; each lane stages one record of a batch in the wave's LDS slot with
// the row groups it reaches, and the wave reads the records back by broadcast.
// Lane = column and row group (PX rows STEP apart); groups not reached are
// skipped by scalar branches. The waves' partial images are summed in wave order.
// SPLIT: a workgroup renders one row group of a tile (PX workgroups a tile), for
// launches of few tiles, whose lists are long where the object is: 20k Gaussians
// on 8 views of 128^2 have 128 tiles that matter, half the compute units. Row groups
// of 16-pixel tiles are four blocks of 4 x 4 pixels there, each with a list of the
// batch's records that reach it (206 -> 144 us there).
template <typename S>
struct OpRec {
    S mx, my, a, b, c, w, beta, q;
};

template <int T, bool SPLIT>
constexpr int op_waves() { return (T == 32 ? 4 : 8) * (SPLIT ? 2 : 1); }

// Tiles of a launch up to which they are split. Over 1600 launches that take the row
// kernels (300 to 100k primitives, 1 to 16 views of 48^2 to 512^2, each tile and type),
// whole tiles take 3.2x the split ones' time at 128 tiles in the middle, 2.2x at 256,
// 1.6x at 1024 and 1.4x at 4096 (from 0.7 to 2.7 there, by how unequal the lists are).
constexpr uint64_t kSplitTiles = 4096;

template <typename S, int T, bool BETA, bool VAR, bool SPLIT>
__global__ void __launch_bounds__((op_waves<T, SPLIT>() * kWave))
raster_fwd_rows_kernel(RasterArgs<S> A, S* __restrict__ out, S* __restrict__ out_var) {
    constexpr int WAVES = op_waves<T, SPLIT>(), STEP = kWave / T, GROUPS = T * T / kWave, PX = SPLIT ? 1 : GROUPS;
    constexpr uint32_t kPixels = PX * kWave;
    constexpr bool BLOCKS = SPLIT && T == 16;
    __shared__ OpRec<S> stage[WAVES][kWave + (BLOCKS ? 1 : 0)];
    __shared__ S part[WAVES][kPixels];
    __shared__ __align__(16) uint8_t lists[BLOCKS ? WAVES : 1][4][kWave];
    uint32_t cam, ty, tx;
    int32_t start, end;
    const uint32_t group = SPLIT ? blockIdx.x % GROUPS : 0u, y0 = group * STEP;  // the workgroup's first row
    tile_range(A, SPLIT ? blockIdx.x / GROUPS : blockIdx.x, cam, ty, tx, start, end);
    const uint32_t lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t col = lane % T, row0 = lane / T;
    const S px = S(tx * T + col) + S(0.5);
    S py[PX], acc[PX], acc_var[PX];
#pragma unroll
    for (int k = 0; k < PX; ++k) {
        py[k] = S(ty * T + y0 + row0 + STEP * k) + S(0.5);
        acc[k] = S(0);
        acc_var[k] = S(0);
    }
    OpRec<S>* slot = stage[wave];
    if (BLOCKS && lane == 0) slot[kWave] = OpRec<S>{};  // the record past a list's end: no weight
    for (int32_t base = start + int32_t(wave) * kWave; base < end; base += WAVES * kWave) {
        uint32_t groups = 0, blocks = 0;
        OpRec<S> r = {};
        if (base + int32_t(lane) < end) {
            const int32_t g = A.flatten[base + int32_t(lane)];
            if (g >= 0 && uint32_t(g) < A.C * A.N) {  // out-of-range ids contribute nothing
                const Prim2D<S> p = load_prim(A, g, BETA);
                int lo, hi;
                reached_rows<S, BETA>(p, S(ty * T), T, lo, hi);
                const int k_lo = lo / STEP, k_hi = (hi + STEP - 1) / STEP;
                if (lo < hi) groups = (((1u << k_hi) - 1u) & ~((1u << k_lo) - 1u)) >> group;
                if constexpr (SPLIT) groups &= 1u;
                if constexpr (BLOCKS) {
                    if (groups != 0u) {
                        int c_lo, c_hi;
                        reached_cols<S, BETA>(p, S(tx * T), T, c_lo, c_hi);
                        if (c_lo < c_hi) blocks = (0xfu >> (3 - ((c_hi - 1) >> 2))) & (0xfu << (c_lo >> 2));
                    }
                }
                r = OpRec<S>{p.mx, p.my, p.a, p.b, p.c, p.opac * p.mu, p.beta, VAR ? A.unc[uint32_t(g) % A.N] : S(0)};
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // every lane is done with the previous batch
        slot[lane] = r;
        if constexpr (BLOCKS) {
            constexpr uint32_t kFill = uint32_t(kWave) * 0x01010101u;
            reinterpret_cast<uint32_t*>(lists[wave])[lane] = kFill;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const auto splat = [&](const OpRec<S>& s, uint32_t rows) {
            const S dx = px - s.mx, adx = s.a * dx, bdx = (BETA ? S(2) : S(1)) * s.b * dx;
#pragma unroll
            for (int k = 0; k < PX; ++k) {
                if (PX > 1 && !((rows >> k) & 1u)) continue;
                const S dy = py[k] - s.my;
                S alpha;
                bool keep;
                if constexpr (BETA) {
                    const S q = pair_form<S, BETA>(adx, dx, bdx, s.c, dy);
                    keep = !(q < S(0) || q >= S(1));
                    alpha = s.w * (keep ? Math<S>::pow(S(1) - q, s.beta) : S(0));
                } else {
                    const S sigma = pair_form<S, BETA>(adx, dx, bdx, s.c, dy);
                    alpha = s.w * Math<S>::exp(-sigma);
                    keep = !(sigma < S(0));
                }
                keep = keep && !(fabs(alpha) < S(1e-5));
                if (!keep) alpha = S(0);
                acc[k] += alpha;
                if constexpr (VAR) acc_var[k] += (keep ? s.q : S(0)) * alpha * alpha;
            }
        };
        if constexpr (BLOCKS) {
            // each 4 x 4 block of the row group (16 lanes) walks the records that reach it
            uint32_t longest = 0;
#pragma unroll
            for (uint32_t b = 0; b < 4; ++b) {
                const uint64_t members = __ballot((blocks >> b) & 1u);
                const uint32_t at = __builtin_amdgcn_mbcnt_hi(uint32_t(members >> 32),
                                                              __builtin_amdgcn_mbcnt_lo(uint32_t(members), 0u));
                if ((blocks >> b) & 1u) lists[wave][b][at] = uint8_t(lane);
                longest = max(longest, uint32_t(__popcll(members)));
            }
            wave_lds_sync();
            const uint8_t* list = lists[wave][(lane % 16u) / 4u];
            OpRec<S> next = slot[list[0]];
            for (uint32_t k = 0; k < longest; ++k) {
                const OpRec<S> now = next;
                next = slot[list[min(k + 1u, uint32_t(kWave) - 1u)]];  // read while this one is evaluated
                splat(now, 1u);
            }
            continue;
        }
        // the batch's records that reach a group, the next one read from LDS while
        // this one is evaluated (two registers that alternate roles)
        uint64_t todo = __ballot(groups != 0u);
        if (todo == 0ull) continue;
        const auto pop = [&]() -> int {
            const int j = __builtin_ctzll(todo);
            todo &= todo - 1ull;
            return j;
        };
        int ja = pop();
        OpRec<S> a = slot[ja];
        for (;;) {
            const bool more_b = todo != 0ull;
            const int jb = more_b ? pop() : ja;
            const OpRec<S> b = slot[jb];
            splat(a, __builtin_amdgcn_readlane(groups, ja));
            if (!more_b) break;
            const bool more_a = todo != 0ull;
            ja = more_a ? pop() : jb;
            a = slot[ja];
            splat(b, __builtin_amdgcn_readlane(groups, jb));
            if (!more_a) break;
        }
    }
#pragma unroll
    for (int o = 0; o < (VAR ? 2 : 1); ++o) {
#pragma unroll
        for (int k = 0; k < PX; ++k) part[wave][(row0 + STEP * k) * T + col] = o ? acc_var[k] : acc[k];
        __syncthreads();
        for (uint32_t p = threadIdx.x; p < kPixels; p += WAVES * kWave) {
            S v = S(0);
#pragma unroll
            for (int k = 0; k < WAVES; ++k) v += part[k][p];
            const uint32_t x = tx * T + p % T, y = ty * T + y0 + p / T;
            if (x < A.W && y < A.H) (o ? out_var : out)[(size_t(cam) * A.H + y) * A.W + x] = v;
        }
        if (VAR && o == 0) __syncthreads();  // the mean's partial images are consumed
    }
}

// VJP: one lane per intersection (sorted_chunk: a chunk's tiles staged together,
// most rows first), summing its moments over the rows it reaches:
//   Gaussian, delta = pixel - mean, g = v alpha: v_mean = (a Mx + b My, b Mx + c My),
//     v_conic = -(Mxx / 2, Mxy, Myy / 2), v_opac = mu sum v vis, v_mu = opac sum v vis;
//   Beta, delta = mean - pixel, G = v vis / h, k = -opac mu beta: v_mean = 2k (a Mx +
//     b My, b Mx + c My), v_conic = k (Mxx, 2 Mxy, Myy), v_beta = sum v alpha log h.
template <int T>
constexpr uint32_t op_tiles() { return T == 8 ? 16 : T == 16 ? 8 : 2; }

template <typename S, int T, uint32_t CHUNK, bool BETA, bool VAR>
__global__ void __launch_bounds__(kChunkThreads) __attribute__((amdgpu_waves_per_eu(3)))
raster_bwd_rows_kernel(RasterArgs<S> A, const int64_t* __restrict__ isect_ids, const S* __restrict__ v_render,
                       const S* __restrict__ v_var, const S* __restrict__ unc, S* __restrict__ v_xy,
                       S* __restrict__ v_conic, S* __restrict__ v_opac, S* __restrict__ v_mu,
                       S* __restrict__ v_beta, S* __restrict__ v_q) {
    constexpr uint32_t kPixels = T * T, kRun = std::is_same<S, float>::value ? 8 : T;  // columns of a row sum
    __shared__ __align__(16) S sv[op_tiles<T>() * kPixels];
    __shared__ __align__(16) S svv[VAR ? op_tiles<T>() * kPixels : 2];
    const uint32_t nt = A.ntx * A.nty;
    sorted_chunk<CHUNK, op_tiles<T>(), kPixels, false>(
        isect_ids, A.n_isects, int64_t(A.C) * nt,
        [&](uint32_t slot, uint32_t key, uint32_t p) {
            const uint32_t cam = key / nt, t = key - cam * nt, ty = t / A.ntx, tx = t - ty * A.ntx;
            const uint32_t x = tx * T + p % T, y = ty * T + p / T;
            const bool in = x < A.W && y < A.H;
            const size_t o = (size_t(cam) * A.H + y) * A.W + x;
            sv[slot * kPixels + p] = in ? v_render[o] : S(0);
            if constexpr (VAR) svv[slot * kPixels + p] = in ? v_var[o] : S(0);
        },
        [&](uint32_t e, uint32_t key, uint64_t& mask, double&) {
            const int32_t g = A.flatten[e];
            if (g < 0 || uint32_t(g) >= A.C * A.N) return false;
            int lo, hi;
            const uint32_t y0 = ((key % nt) / A.ntx) * T;
            reached_rows<S, BETA>(load_prim(A, g, BETA), S(y0), T, lo, hi);
            hi = max(lo, min(hi, int(A.H) - int(y0)));  // (a pair past the image is none)
            mask = ((1ull << hi) - 1ull) & ~((1ull << lo) - 1ull);
            return hi > lo;
        },
        [&](uint32_t e, uint32_t key, uint32_t slot, uint64_t rows, double, bool active) {
            const uint32_t t = key % nt, ty = t / A.ntx, tx = t - ty * A.ntx;
            const int32_t g = A.flatten[e];
            const Prim2D<S> p = load_prim(A, g, BETA);
            const uint32_t n = uint32_t(g) % A.N;
            const S w = p.opac * p.mu, q2 = VAR && unc ? S(2) * unc[n] : S(0);
            double m0 = 0.0, mx = 0.0, my = 0.0, mxx = 0.0, mxy = 0.0, myy = 0.0, sl = 0.0, vq = 0.0;
            while (rows) {
                const uint32_t r = uint32_t(__builtin_ctzll(rows));
                rows &= rows - 1ull;
                const S py = S(ty * T + r) + S(0.5), dy = BETA ? p.my - py : py - p.my;
                const S* row = sv + slot * kPixels + r * T;
                const S* rowv = svv + (VAR ? slot * kPixels + r * T : 0);
#pragma unroll 1
                for (uint32_t j0 = 0; j0 < uint32_t(T); j0 += kRun) {
                    S r0 = S(0), r1 = S(0), r2 = S(0), rm = S(0), rl = S(0), rq = S(0);
#pragma unroll 2
                    for (uint32_t j = j0; j < j0 + kRun; ++j) {
                        const S px = S(tx * T + j) + S(0.5), dx = BETA ? p.mx - px : px - p.mx;
                        S v = row[j];
                        const S vv = VAR ? rowv[VAR ? j : 0] : S(0);
                        if constexpr (BETA) {
                            const S q = pair_form<S, BETA>(p.a * dx, dx, S(2) * p.b * dx, p.c, dy);
                            if (q < S(0) || q >= S(1)) continue;
                            const S h = S(1) - q, vis = Math<S>::pow(h, p.beta), alpha = w * vis;
                            if (fabs(alpha) < S(1e-5)) continue;
                            if constexpr (VAR) {
                                row_sum(rq, vq, vv * alpha * alpha);
                                v += q2 * alpha * vv;
                            }
                            const S gv = v * (vis / h);
                            row_sum(rm, m0, v * vis);
                            row_sum(rl, sl, v * alpha * Math<S>::log(h));
                            r0 += gv;
                            r1 += gv * dx;
                            r2 += gv * dx * dx;
                        } else {
                            const S sigma = vjp_sigma(p.a * dx, dx, p.b * dx, p.c, dy);
                            const S vis = Math<S>::exp(-sigma), alpha = w * vis;
                            const bool keep = !(sigma < S(0) || fabs(alpha) < S(1e-5));
                            if constexpr (VAR) {
                                row_sum(rq, vq, keep ? vv * alpha * alpha : S(0));
                                v += q2 * alpha * vv;
                            }
                            const S gv = keep ? v * alpha : S(0);
                            row_sum(rm, m0, keep ? v * vis : S(0));
                            r0 += gv;
                            r1 += gv * dx;
                            r2 += gv * dx * dx;
                        }
                    }
                    mx += r1;
                    mxx += r2;
                    my += double(dy) * r0;
                    mxy += double(dy) * r1;
                    myy += double(dy) * dy * r0;
                    m0 += rm;
                    sl += rl;
                    vq += rq;
                }
            }
            if (!active) return;
            // no pair: an infinite parameter times an empty sum would be a NaN
            if (m0 == 0.0 && vq == 0.0 && !all_finite<S, BETA>(p)) return;
            const size_t G = size_t(g);
            if constexpr (BETA) {
                const double k = -w * p.beta;
                atomic_add(v_xy + 2 * G, S(2.0 * k * (p.a * mx + p.b * my)));
                atomic_add(v_xy + 2 * G + 1, S(2.0 * k * (p.b * mx + p.c * my)));
                atomic_add(v_conic + 3 * G, S(k * mxx));
                atomic_add(v_conic + 3 * G + 1, S(2.0 * k * mxy));
                atomic_add(v_conic + 3 * G + 2, S(k * myy));
                atomic_add(v_beta + G, S(sl));
            } else {
                atomic_add(v_xy + 2 * G, S(p.a * mx + p.b * my));
                atomic_add(v_xy + 2 * G + 1, S(p.b * mx + p.c * my));
                atomic_add(v_conic + 3 * G, S(-0.5 * mxx));
                atomic_add(v_conic + 3 * G + 1, S(-mxy));
                atomic_add(v_conic + 3 * G + 2, S(-0.5 * myy));
            }
            atomic_add(v_opac + G, S(p.mu * m0));
            atomic_add(v_mu + G, S(p.opac * m0));
            if constexpr (VAR)
                if (v_q) atomic_add(v_q + n, S(vq));
        });
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
inline int check_tile(uint32_t T, uint32_t ntx, uint32_t nty, uint32_t W, uint32_t H) {
    R2S_REQUIRE(T >= 1 && T * T <= 1024, "tile_size %u must satisfy 1 <= tile_size^2 <= 1024", T);
    R2S_REQUIRE(uint64_t(ntx) * T >= W && uint64_t(nty) * T >= H,
                "tile grid %ux%u of size %u does not cover the %ux%u image", ntx, nty, T, W, H);
    return R2S_OK;
}

inline uint32_t block_threads(uint32_t T) { return ((T * T + kWave - 1) / kWave) * kWave; }

template <typename S>
RasterArgs<S> make_args(const void* means2d, const void* conics, const void* opac, const void* mus,
                        const void* betas, const void* unc, const int32_t* offsets,
                        const int32_t* flatten, uint32_t n_isects, uint32_t C, uint32_t N,
                        uint32_t W, uint32_t H, uint32_t T, uint32_t ntx, uint32_t nty) {
    return RasterArgs<S>{(const S*)means2d, (const S*)conics, (const S*)opac, (const S*)mus,
                         (const S*)betas, (const S*)unc, offsets, flatten, n_isects, C, N, W, H, T,
                         ntx, nty};
}

// Whether a forward takes the row kernel. It gives a tile several waves, so it wins
// where tiles are few (float32, 137k intersections on 9 16-pixel tiles: 119 us, one
// wave per pixel group 7113) or their lists long, the longer the more tiles there
// are to fill the chip without it; it loses on short lists of many tiles (4096 tiles,
// 2778 intersections: 51 us against 10; 65536 8-pixel tiles of 11 each: 164 against 43).
inline bool fwd_by_rows(uint32_t n_isects, uint64_t prims, uint64_t tiles) {
    const double list = std::min(80.0, 4.0 + double(tiles) / 40.0) * (0.5 + 2.0 * tile_overhang(n_isects, prims, 2));
    return tiles <= 64 || double(n_isects) >= list * double(tiles);
}

// Whether a per-primitive VJP takes the row kernel, a lane per intersection: it needs
// intersections enough to fill the chip, more where each fills its tile (a lane then
// walks all T^2 pixels alone), and lists long enough that a chunk meets few tiles. On
// the other side the general kernel has a wave per intersection. float64 Beta, 32-pixel
// tiles: 1.9M intersections on 64 tiles 228 us against 3361; 545 on 256 tiles 5325
// against 25. float32, 16-pixel tiles: 2.2M on 144 tiles 343 against 1068; 718 on 1024
// 267 against 13.
template <typename S>
inline bool vjp_by_rows(uint32_t n_isects, uint64_t prims, uint64_t tiles, uint32_t T, bool beta) {
    constexpr bool kDouble = std::is_same<S, double>::value;
    const double over = tile_overhang(n_isects, prims, 2);
    double few, few_wide, list, list_wide;  // intersections and mean list at no overhang, and what a whole tile adds
    if (T == 8) few = 0, few_wide = 16e3, list = 8, list_wide = 0;
    else if (T == 16) few = 0, few_wide = kDouble && beta ? 128e3 : 32e3, list = 24, list_wide = kDouble && !beta ? 32 : 128;
    else if (T == 32) few = 8e3, few_wide = beta ? 256e3 : 160e3, list = 48, list_wide = kDouble && beta ? 512 : 96;
    else return false;
    return n_isects >= few + few_wide * over && double(n_isects) >= (list + list_wide * over) * double(tiles);
}

int launch_fwd(int dtype, bool beta, bool var, const void* means2d, const void* conics,
               const void* opac, const void* mus, const void* betas, const void* unc,
               const int32_t* offsets, const int32_t* flatten, uint32_t n_isects, uint32_t C,
               uint32_t N, uint32_t W, uint32_t H, uint32_t T, uint32_t ntx, uint32_t nty,
               void* out, void* out_var, hipStream_t stream) {
    if (int rc = check_tile(T, ntx, nty, W, H)) return rc;
    const uint64_t blocks = uint64_t(C) * ntx * nty;
    if (blocks == 0 || W == 0 || H == 0) return R2S_OK;
    const uint32_t threads = block_threads(T);
    const size_t shm = lds_bytes(dtype, std::min(threads, kBatch));
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        auto A = make_args<S>(means2d, conics, opac, mus, betas, unc, offsets, flatten, n_isects, C,
                              N, W, H, T, ntx, nty);
        const auto rows = [&](auto tile) {
            constexpr int TILE = decltype(tile)::value;
            const auto launch = [&](auto split) {
                constexpr bool SPLIT = decltype(split)::value;
                auto k = beta ? (var ? raster_fwd_rows_kernel<S, TILE, true, true, SPLIT>
                                     : raster_fwd_rows_kernel<S, TILE, true, false, SPLIT>)
                              : (var ? raster_fwd_rows_kernel<S, TILE, false, true, SPLIT>
                                     : raster_fwd_rows_kernel<S, TILE, false, false, SPLIT>);
                k<<<uint32_t(blocks) * (SPLIT ? TILE * TILE / kWave : 1), op_waves<TILE, SPLIT>() * kWave, 0, stream>>>(
                    A, (S*)out, (S*)out_var);
                return check_launch("rasterize_to_pixels_fwd");
            };
            return blocks <= kSplitTiles ? launch(std::true_type{}) : launch(std::false_type{});
        };
        if (fwd_by_rows(n_isects, uint64_t(C) * N, blocks)) {
            if (T == 8) return rows(std::integral_constant<int, 8>{});
            if (T == 16) return rows(std::integral_constant<int, 16>{});
            if (T == 32) return rows(std::integral_constant<int, 32>{});
        }
        auto k = beta ? (var ? raster_fwd_kernel<S, true, true> : raster_fwd_kernel<S, true, false>)
                      : (var ? raster_fwd_kernel<S, false, true> : raster_fwd_kernel<S, false, false>);
        k<<<uint32_t(blocks), threads, shm, stream>>>(A, (S*)out, (S*)out_var);
        return check_launch("rasterize_to_pixels_fwd");
    });
}

}  // namespace r2s

using namespace r2s;

extern "C" int r2s_rasterize_to_pixels_fwd(int dtype, const void* means2d, const void* conics,
                                           const void* opacities, const void* mus,
                                           const int32_t* tile_offsets, const int32_t* flatten_ids,
                                           uint32_t n_isects, uint32_t C, uint32_t N,
                                           uint32_t width, uint32_t height, uint32_t tile_size,
                                           uint32_t n_tiles_x, uint32_t n_tiles_y, void* render,
                                           r2s_stream_t stream) {
    return launch_fwd(dtype, false, false, means2d, conics, opacities, mus, nullptr, nullptr,
                      tile_offsets, flatten_ids, n_isects, C, N, width, height, tile_size,
                      n_tiles_x, n_tiles_y, render, nullptr, stream);
}

extern "C" int r2s_rasterize_to_pixels_mean_var_fwd(
    int dtype, const void* means2d, const void* conics, const void* opacities, const void* mus,
    const void* uncertainties, const int32_t* tile_offsets, const int32_t* flatten_ids,
    uint32_t n_isects, uint32_t C, uint32_t N, uint32_t width, uint32_t height, uint32_t tile_size,
    uint32_t n_tiles_x, uint32_t n_tiles_y, void* render, void* render_var, r2s_stream_t stream) {
    return launch_fwd(dtype, false, true, means2d, conics, opacities, mus, nullptr, uncertainties,
                      tile_offsets, flatten_ids, n_isects, C, N, width, height, tile_size,
                      n_tiles_x, n_tiles_y, render, render_var, stream);
}

extern "C" int r2s_beta_rasterize_to_pixels_fwd(int dtype, const void* means2d, const void* conics,
                                                const void* opacities, const void* mus,
                                                const void* betas, const int32_t* tile_offsets,
                                                const int32_t* flatten_ids, uint32_t n_isects,
                                                uint32_t C, uint32_t N, uint32_t width,
                                                uint32_t height, uint32_t tile_size,
                                                uint32_t n_tiles_x, uint32_t n_tiles_y,
                                                void* render, r2s_stream_t stream) {
    return launch_fwd(dtype, true, false, means2d, conics, opacities, mus, betas, nullptr,
                      tile_offsets, flatten_ids, n_isects, C, N, width, height, tile_size,
                      n_tiles_x, n_tiles_y, render, nullptr, stream);
}

extern "C" int r2s_beta_rasterize_to_pixels_mean_var_fwd(
    int dtype, const void* means2d, const void* conics, const void* opacities, const void* mus,
    const void* betas, const void* uncertainties, const int32_t* tile_offsets,
    const int32_t* flatten_ids, uint32_t n_isects, uint32_t C, uint32_t N, uint32_t width,
    uint32_t height, uint32_t tile_size, uint32_t n_tiles_x, uint32_t n_tiles_y, void* render,
    void* render_var, r2s_stream_t stream) {
    return launch_fwd(dtype, true, true, means2d, conics, opacities, mus, betas, uncertainties,
                      tile_offsets, flatten_ids, n_isects, C, N, width, height, tile_size,
                      n_tiles_x, n_tiles_y, render, render_var, stream);
}

extern "C" int r2s_rasterize_to_pixels_uncertainty_bwd(
    int dtype, const void* means2d, const void* conics, const void* opacities, const void* mus,
    const void* betas, const int32_t* tile_offsets, const int32_t* flatten_ids, uint32_t n_isects,
    uint32_t C, uint32_t N, uint32_t width, uint32_t height, uint32_t tile_size,
    uint32_t n_tiles_x, uint32_t n_tiles_y, const void* v_render_var, void* v_uncertainties,
    r2s_stream_t stream) {
    if (int rc = check_tile(tile_size, n_tiles_x, n_tiles_y, width, height)) return rc;
    const bool beta = betas != nullptr;
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        if (int rc = fill_zero<S>((S*)v_uncertainties, N, stream)) return rc;
        const uint64_t blocks = uint64_t(C) * n_tiles_x * n_tiles_y;
        if (blocks == 0 || n_isects == 0) return R2S_OK;
        const uint32_t threads = block_threads(tile_size);
        const size_t shm = lds_bytes(dtype, std::min(threads, kBatch));
        auto A = make_args<S>(means2d, conics, opacities, mus, betas, nullptr, tile_offsets,
                              flatten_ids, n_isects, C, N, width, height, tile_size, n_tiles_x,
                              n_tiles_y);
        auto k = beta ? raster_bwd_tile_kernel<S, true, 1> : raster_bwd_tile_kernel<S, false, 1>;
        k<<<uint32_t(blocks), threads, shm, stream>>>(A, (const S*)v_render_var, nullptr, nullptr,
                                                      nullptr, nullptr, nullptr, nullptr,
                                                      (S*)v_uncertainties);
        return check_launch("rasterize_to_pixels_uncertainty_bwd");
    });
}

extern "C" int r2s_rasterize_to_pixels_bwd(
    int dtype, const void* means2d, const void* conics, const void* opacities, const void* mus,
    const void* betas, const int32_t* tile_offsets, const int32_t* flatten_ids, uint32_t n_isects,
    uint32_t C, uint32_t N, uint32_t width, uint32_t height, uint32_t tile_size,
    uint32_t n_tiles_x, uint32_t n_tiles_y, const void* v_render, void* v_means2d_abs,
    void* v_means2d, void* v_conics, void* v_opacities, void* v_mus, void* v_betas,
    r2s_stream_t stream) {
    if (int rc = check_tile(tile_size, n_tiles_x, n_tiles_y, width, height)) return rc;
    const bool beta = betas != nullptr;
    R2S_REQUIRE(!beta || v_betas != nullptr, "v_betas is required with betas");
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        const size_t CN = size_t(C) * N;
        if (int rc = zero_grads_2d<S>(CN, v_means2d_abs, v_means2d, v_conics, v_opacities, v_mus,
                                      beta ? v_betas : nullptr, stream))
            return rc;
        const uint64_t blocks = uint64_t(C) * n_tiles_x * n_tiles_y;
        if (blocks == 0 || n_isects == 0 || CN == 0) return R2S_OK;
        const uint32_t threads = block_threads(tile_size);
        const size_t shm = lds_bytes(dtype, std::min(threads, kBatch));
        auto A = make_args<S>(means2d, conics, opacities, mus, betas, nullptr, tile_offsets,
                              flatten_ids, n_isects, C, N, width, height, tile_size, n_tiles_x,
                              n_tiles_y);
        auto k = beta ? raster_bwd_tile_kernel<S, true, 0> : raster_bwd_tile_kernel<S, false, 0>;
        k<<<uint32_t(blocks), threads, shm, stream>>>(A, (const S*)v_render, (S*)v_means2d_abs,
                                                      (S*)v_means2d, (S*)v_conics, (S*)v_opacities,
                                                      (S*)v_mus, (S*)v_betas, nullptr);
        return check_launch("rasterize_to_pixels_bwd");
    });
}

extern "C" int r2s_rasterize_to_pixels_bwd_per_gaussian(
    int dtype, const void* means2d, const void* conics, const void* opacities, const void* mus,
    const void* betas, const int64_t* isect_ids, const int32_t* flatten_ids, uint32_t n_isects,
    uint32_t C, uint32_t N, uint32_t width, uint32_t height, uint32_t tile_size,
    uint32_t n_tiles_x, uint32_t n_tiles_y, const void* v_render, const void* v_render_var,
    const void* uncertainties, void* v_means2d_abs, void* v_means2d, void* v_conics,
    void* v_opacities, void* v_mus, void* v_betas, void* v_uncertainties, r2s_stream_t stream) {
    if (int rc = check_tile(tile_size, n_tiles_x, n_tiles_y, width, height)) return rc;
    const bool beta = betas != nullptr;
    R2S_REQUIRE(!beta || v_betas != nullptr, "v_betas is required with betas");
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        const size_t CN = size_t(C) * N;
        if (int rc = zero_grads_2d<S>(CN, v_means2d_abs, v_means2d, v_conics, v_opacities, v_mus,
                                      beta ? v_betas : nullptr, stream, v_uncertainties, N))
            return rc;
        if (n_isects == 0 || CN == 0) return R2S_OK;
        auto A = make_args<S>(means2d, conics, opacities, mus, betas, nullptr, nullptr, flatten_ids,
                              n_isects, C, N, width, height, tile_size, n_tiles_x, n_tiles_y);
        const bool var = v_render_var != nullptr;
        const auto rows = [&](auto tile) {
            constexpr int TILE = decltype(tile)::value;
            const bool few = n_isects <= kFewIsects;
            const auto launch = [&](auto chunk) {
                constexpr uint32_t CHUNK = decltype(chunk)::value;
                auto k = beta ? (var ? raster_bwd_rows_kernel<S, TILE, CHUNK, true, true>
                                     : raster_bwd_rows_kernel<S, TILE, CHUNK, true, false>)
                              : (var ? raster_bwd_rows_kernel<S, TILE, CHUNK, false, true>
                                     : raster_bwd_rows_kernel<S, TILE, CHUNK, false, false>);
                k<<<ceil_div(n_isects, CHUNK), kChunkThreads, 0, stream>>>(
                    A, isect_ids, (const S*)v_render, (const S*)v_render_var, (const S*)uncertainties, (S*)v_means2d,
                    (S*)v_conics, (S*)v_opacities, (S*)v_mus, (S*)v_betas, (S*)v_uncertainties);
            };
            if (few) launch(std::integral_constant<uint32_t, 256>{});
            else launch(std::integral_constant<uint32_t, 512>{});
            return check_launch("rasterize_to_pixels_bwd_per_gaussian");
        };
        const uint64_t tiles = uint64_t(C) * n_tiles_x * n_tiles_y;
        if (!v_means2d_abs && tiles < (1ull << 32) - 1 && vjp_by_rows<S>(n_isects, CN, tiles, tile_size, beta)) {
            if (tile_size == 8) return rows(std::integral_constant<int, 8>{});
            if (tile_size == 16) return rows(std::integral_constant<int, 16>{});
            if (tile_size == 32) return rows(std::integral_constant<int, 32>{});
        }
        constexpr uint32_t waves = 4;
        auto k = beta ? raster_bwd_isect_kernel<S, true> : raster_bwd_isect_kernel<S, false>;
        k<<<std::min<uint32_t>(ceil_div(n_isects, waves), kIsectBlocks), waves * kWave, 0, stream>>>(
            A, isect_ids, (const S*)v_render, (const S*)v_render_var,
            v_render_var ? (const S*)uncertainties : nullptr, (S*)v_means2d_abs, (S*)v_means2d,
            (S*)v_conics, (S*)v_opacities, (S*)v_mus, (S*)v_betas,
            v_render_var ? (S*)v_uncertainties : nullptr);
        return check_launch("rasterize_to_pixels_bwd_per_gaussian");
    });
}
