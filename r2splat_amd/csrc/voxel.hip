// 3D voxelization: each voxel sums opacity * profile over the primitives binned
// to its 3D tile. Tile-parallel forward / VJP (LDS-staged batches) and the
// intersection-parallel VJP (one wave64 per intersection), for any tile size
// with tile_size^3 <= 1024 and both float/double; 8^3 tiles have forms that skip
// what a primitive does not reach (octants in the forward, rows in the VJP).
// Profiles follow r2splat/cuda/csrc/VoxelizeToVoxelsFwd.cu:181-219 (Gaussian,
// threshold 1e-6) and the Beta kernels (threshold 1e-5); the VJPs follow
// VoxelizeToVoxelsBwd.cu:387-434 and the Beta per-primitive kernel.
#include <type_traits>

#include "common.hpp"
#include "binning.hpp"
#include "geometry_common.hpp"
#include "raster_common.hpp"
#include "sorted_chunk.hpp"

namespace r2s {

constexpr uint32_t kVoxBatch = 256;

template <typename S>
struct Prim3D {
    S x, y, z, c[6], opac, beta;
};

template <typename S, bool BETA>
__device__ __forceinline__ bool eval_profile3(const Prim3D<S>& p, S px, S py, S pz, S& vis, S& alpha) {
    if (!BETA) {
        const S dx = px - p.x, dy = py - p.y, dz = pz - p.z;
        const S sigma = S(0.5) * (p.c[0] * dx * dx + p.c[3] * dy * dy + p.c[5] * dz * dz) +
                        p.c[1] * dx * dy + p.c[2] * dx * dz + p.c[4] * dy * dz;
        vis = Math<S>::exp(-sigma);
        alpha = p.opac * vis;
        return !(sigma < S(0) || fabs(alpha) < S(1e-6));
    } else {
        const S dx = p.x - px, dy = p.y - py, dz = p.z - pz;
        const S q = p.c[0] * dx * dx + p.c[3] * dy * dy + p.c[5] * dz * dz +
                    S(2) * (p.c[1] * dx * dy + p.c[2] * dx * dz + p.c[4] * dy * dz);
        if (q < S(0) || q >= S(1)) return false;
        const S h = S(1) - q;
        vis = Math<S>::pow(h, p.beta);
        alpha = p.opac * vis;
        return !(fabs(alpha) < S(1e-5));
    }
}

template <typename S>
struct Grad3D {
    S xyz[3] = {S(0), S(0), S(0)};
    S c[6] = {S(0), S(0), S(0), S(0), S(0), S(0)};
    S opac = S(0), beta = S(0);

    __device__ __forceinline__ void reduce_wave() {
#pragma unroll
        for (int k = 0; k < 3; ++k) xyz[k] = wave_sum(xyz[k]);
#pragma unroll
        for (int k = 0; k < 6; ++k) c[k] = wave_sum(c[k]);
        opac = wave_sum(opac);
        beta = wave_sum(beta);
    }
    __device__ __forceinline__ void commit(int32_t g, S* v_xyz, S* v_c, S* v_opac, S* v_beta) const {
        const size_t G = size_t(g);
#pragma unroll
        for (int k = 0; k < 3; ++k) atomic_add(v_xyz + 3 * G + k, xyz[k]);
#pragma unroll
        for (int k = 0; k < 6; ++k) atomic_add(v_c + 6 * G + k, c[k]);
        atomic_add(v_opac + G, opac);
        if (v_beta) atomic_add(v_beta + G, beta);
    }
};

template <typename S, bool BETA>
__device__ __forceinline__ void voxel_vjp(const Prim3D<S>& p, S px, S py, S pz, S vis, S alpha, S v,
                                          Grad3D<S>& g) {
    if (!BETA) {
        const S dx = px - p.x, dy = py - p.y, dz = pz - p.z;
        const S vs = -v * alpha;  // d/d sigma
        g.c[0] += vs * S(0.5) * dx * dx;
        g.c[1] += vs * dx * dy;
        g.c[2] += vs * dx * dz;
        g.c[3] += vs * S(0.5) * dy * dy;
        g.c[4] += vs * dy * dz;
        g.c[5] += vs * S(0.5) * dz * dz;
        const S va = v * alpha;  // d sigma / d mean = -P delta
        g.xyz[0] += va * (p.c[0] * dx + p.c[1] * dy + p.c[2] * dz);
        g.xyz[1] += va * (p.c[1] * dx + p.c[3] * dy + p.c[4] * dz);
        g.xyz[2] += va * (p.c[2] * dx + p.c[4] * dy + p.c[5] * dz);
    } else {
        const S dx = p.x - px, dy = p.y - py, dz = p.z - pz;
        const S q = p.c[0] * dx * dx + p.c[3] * dy * dy + p.c[5] * dz * dz +
                    S(2) * (p.c[1] * dx * dy + p.c[2] * dx * dz + p.c[4] * dy * dz);
        const S h = S(1) - q;
        const S vq = -p.opac * p.beta * (vis / h) * v;  // d/d q
        g.c[0] += vq * dx * dx;
        g.c[1] += S(2) * vq * dx * dy;
        g.c[2] += S(2) * vq * dx * dz;
        g.c[3] += vq * dy * dy;
        g.c[4] += S(2) * vq * dy * dz;
        g.c[5] += vq * dz * dz;
        g.xyz[0] += S(2) * vq * (p.c[0] * dx + p.c[1] * dy + p.c[2] * dz);
        g.xyz[1] += S(2) * vq * (p.c[1] * dx + p.c[3] * dy + p.c[4] * dz);
        g.xyz[2] += S(2) * vq * (p.c[2] * dx + p.c[4] * dy + p.c[5] * dz);
        g.beta += v * alpha * Math<S>::log(h);
    }
    g.opac += v * vis;
}

template <typename S>
struct VoxArgs {
    const S* means3d; const S* conics; const S* opac; const S* betas; const S* unc;
    const int32_t* offsets; const int32_t* flatten; uint32_t n_isects, N, dx, dy, dz, T, ntx, nty, ntz;
    // fused float32 kernels: each primitive's voxel-frame mean and inverse
    // covariance in double precision (kFrame doubles per primitive)
    const double* frame = nullptr;
};

template <typename S>
struct VoxLDS {
    S* f;  // [11][batch]: x y z c0..c5 opac beta
    S* q;
    int32_t* id;
    uint32_t batch;
    __device__ __forceinline__ Prim3D<S> prim(uint32_t t, bool beta) const {
        Prim3D<S> p;
        p.x = f[t]; p.y = f[batch + t]; p.z = f[2 * batch + t];
#pragma unroll
        for (int k = 0; k < 6; ++k) p.c[k] = f[(3 + k) * batch + t];
        p.opac = f[9 * batch + t];
        p.beta = beta ? f[10 * batch + t] : S(0);
        return p;
    }
};

inline size_t vox_lds_bytes(int dtype, uint32_t batch) {
    const size_t s = dtype == R2S_F64 ? 8 : 4;
    return batch * (12 * s + 4);
}

template <typename S>
__device__ __forceinline__ VoxLDS<S> vox_carve(unsigned char* smem, uint32_t batch) {
    VoxLDS<S> L;
    L.f = reinterpret_cast<S*>(smem);
    L.q = L.f + 11 * batch;
    L.id = reinterpret_cast<int32_t*>(L.f + 12 * batch);
    L.batch = batch;
    return L;
}

template <typename S, bool BETA, bool VAR>
__device__ __forceinline__ void vox_stage(const VoxArgs<S>& A, const VoxLDS<S>& L, int32_t b0, int32_t end) {
    const uint32_t t = threadIdx.x;
    if (t < L.batch && b0 + int32_t(t) < end) {
        int32_t g = A.flatten[b0 + t];
        const bool ok = g >= 0 && uint32_t(g) < A.N;
        if (!ok) g = 0;  // out-of-range ids contribute nothing
        const size_t G = size_t(g);
        L.id[t] = g;
        L.f[t] = A.means3d[3 * G];
        L.f[L.batch + t] = A.means3d[3 * G + 1];
        L.f[2 * L.batch + t] = A.means3d[3 * G + 2];
#pragma unroll
        for (int k = 0; k < 6; ++k) L.f[(3 + k) * L.batch + t] = A.conics[6 * G + k];
        L.f[9 * L.batch + t] = ok ? A.opac[g] : S(0);
        if (BETA) L.f[10 * L.batch + t] = A.betas[g];
        if (VAR) L.q[t] = A.unc[g];
    }
}

template <typename S>
__device__ __forceinline__ void vox_tile(const VoxArgs<S>& A, uint32_t blk, uint32_t& i, uint32_t& j,
                                         uint32_t& k, bool& inside, int32_t& start, int32_t& end) {
    const uint32_t tx = blk % A.ntx, rest = blk / A.ntx;
    const uint32_t ty = rest % A.nty, tz = rest / A.nty;
    const uint32_t t = threadIdx.x, T = A.T;
    const uint32_t lx = t % T, ly = (t / T) % T, lz = t / (T * T);
    k = tx * T + lx;
    j = ty * T + ly;
    i = tz * T + lz;
    inside = t < T * T * T && i < A.dz && j < A.dy && k < A.dx;
    start = A.offsets[blk];
    const uint32_t nt = A.ntx * A.nty * A.ntz;
    end = (blk + 1 == nt) ? int32_t(A.n_isects) : A.offsets[blk + 1];
    start = max(0, min(start, int32_t(A.n_isects)));
    end = max(start, min(end, int32_t(A.n_isects)));
}

template <typename S, bool BETA, bool VAR>
__global__ void vox_fwd_kernel(VoxArgs<S> A, S* __restrict__ out, S* __restrict__ out_var) {
    extern __shared__ __align__(16) unsigned char smem[];
    VoxLDS<S> L = vox_carve<S>(smem, min(blockDim.x, kVoxBatch));
    uint32_t i, j, k;
    bool inside;
    int32_t start, end;
    vox_tile(A, blockIdx.x, i, j, k, inside, start, end);
    const S px = S(k) + S(0.5), py = S(j) + S(0.5), pz = S(i) + S(0.5);
    S acc = S(0), acc_var = S(0);
    for (int32_t b0 = start; b0 < end; b0 += int32_t(L.batch)) {
        __syncthreads();
        vox_stage<S, BETA, VAR>(A, L, b0, end);
        __syncthreads();
        if (!inside) continue;
        const uint32_t cnt = uint32_t(min<int32_t>(int32_t(L.batch), end - b0));
        for (uint32_t t = 0; t < cnt; ++t) {
            const Prim3D<S> p = L.prim(t, BETA);
            S vis, alpha;
            if (!eval_profile3<S, BETA>(p, px, py, pz, vis, alpha)) continue;
            acc += alpha;
            if (VAR) acc_var += L.q[t] * alpha * alpha;
        }
    }
    if (inside) {
        const size_t o = (size_t(i) * A.dy + j) * A.dx + k;
        out[o] = acc;
        if (VAR) out_var[o] = acc_var;
    }
}

template <typename S, bool BETA>
__global__ void vox_bwd_tile_kernel(VoxArgs<S> A, const S* __restrict__ v_render, S* __restrict__ v_xyz,
                                    S* __restrict__ v_c, S* __restrict__ v_opac, S* __restrict__ v_beta) {
    extern __shared__ __align__(16) unsigned char smem[];
    VoxLDS<S> L = vox_carve<S>(smem, min(blockDim.x, kVoxBatch));
    uint32_t i, j, k;
    bool inside;
    int32_t start, end;
    vox_tile(A, blockIdx.x, i, j, k, inside, start, end);
    const S px = S(k) + S(0.5), py = S(j) + S(0.5), pz = S(i) + S(0.5);
    const S v = inside ? v_render[(size_t(i) * A.dy + j) * A.dx + k] : S(0);
    for (int32_t b0 = start; b0 < end; b0 += int32_t(L.batch)) {
        __syncthreads();
        vox_stage<S, BETA, false>(A, L, b0, end);
        __syncthreads();
        const uint32_t cnt = uint32_t(min<int32_t>(int32_t(L.batch), end - b0));
        for (uint32_t t = 0; t < cnt; ++t) {
            const Prim3D<S> p = L.prim(t, BETA);
            S vis = S(0), alpha = S(0);
            Grad3D<S> g;
            if (inside && eval_profile3<S, BETA>(p, px, py, pz, vis, alpha))
                voxel_vjp<S, BETA>(p, px, py, pz, vis, alpha, v, g);
            g.reduce_wave();
            if (lane_id() == 0) g.commit(L.id[t], v_xyz, v_c, v_opac, BETA ? v_beta : nullptr);
        }
    }
}

template <typename S, bool BETA>
__global__ void __launch_bounds__(256)
vox_bwd_isect_kernel(VoxArgs<S> A, const int64_t* __restrict__ isect_ids, const S* __restrict__ v_render,
                     const S* __restrict__ v_var, const S* __restrict__ unc, S* __restrict__ v_xyz,
                     S* __restrict__ v_c, S* __restrict__ v_opac, S* __restrict__ v_beta,
                     S* __restrict__ v_q) {
    // grid-stride over intersections (one wave each), at most kIsectBlocks blocks
    const uint32_t waves = blockDim.x / kWave;
    const uint64_t stride = uint64_t(gridDim.x) * waves;
    for (uint64_t e = uint64_t(blockIdx.x) * waves + threadIdx.x / kWave; e < A.n_isects; e += stride) {
        const uint32_t nt = A.ntx * A.nty * A.ntz;
        const int64_t key = isect_ids[e];
        if (key < 0 || key >= int64_t(nt)) continue;
        const uint32_t tile = uint32_t(key);
        const uint32_t tx = tile % A.ntx, ty = (tile / A.ntx) % A.nty, tz = tile / (A.ntx * A.nty);
        const int32_t g = A.flatten[e];
        if (g < 0 || uint32_t(g) >= A.N) continue;
        const size_t G = size_t(g);
        Prim3D<S> p;
        p.x = A.means3d[3 * G];
        p.y = A.means3d[3 * G + 1];
        p.z = A.means3d[3 * G + 2];
#pragma unroll
        for (int k = 0; k < 6; ++k) p.c[k] = A.conics[6 * G + k];
        p.opac = A.opac[g];
        p.beta = BETA ? A.betas[g] : S(0);
        const S q = unc ? unc[g] : S(0);
        Grad3D<S> gr;
        S vq = S(0);
        const uint32_t T = A.T, nvox = T * T * T;
        for (uint32_t t = lane_id(); t < nvox; t += kWave) {
            const uint32_t lx = t % T, ly = (t / T) % T, lz = t / (T * T);
            const uint32_t k = tx * T + lx, j = ty * T + ly, i = tz * T + lz;
            if (i >= A.dz || j >= A.dy || k >= A.dx) continue;
            const S px = S(k) + S(0.5), py = S(j) + S(0.5), pz = S(i) + S(0.5);
            S vis, alpha;
            if (!eval_profile3<S, BETA>(p, px, py, pz, vis, alpha)) continue;
            const size_t o = (size_t(i) * A.dy + j) * A.dx + k;
            S v = v_render[o];
            if (v_var) {
                const S vv = v_var[o];
                vq += vv * alpha * alpha;
                if (unc) v += S(2) * q * alpha * vv;
            }
            voxel_vjp<S, BETA>(p, px, py, pz, vis, alpha, v, gr);
        }
        gr.reduce_wave();
        if (v_q) vq = wave_sum(vq);
        if (lane_id() == 0) {
            gr.commit(g, v_xyz, v_c, v_opac, BETA ? v_beta : nullptr);
            if (v_q) atomic_add(v_q + G, vq);
        }
    }
}

// ---------------------------------------------------------------------------
// Moments form of the per-primitive VJP (float32, 8^3 tiles): a workgroup takes
// a fixed chunk of the tile-sorted intersections (equal work per workgroup,
// whatever the tile populations), with the adjoints of its tiles staged in LDS
// kMomTiles at a time; a lane sums one intersection's moments over the rows of
// 8 voxels that its primitive reaches, without cross-lane reduction:
//   Gaussian, delta = voxel - mean, G = v e^-sigma (terms that pass the cut-off):
//     M0 = sum G, M_k = sum G delta_k, M_kl = sum G delta_k delta_l,
//     v_mean = opac P M, v_conic = -opac (M_xx/2, M_xy, M_xz, M_yy/2, M_yz, M_zz/2),
//     v_opac = M0;
//   Beta, h = 1 - q, G = v h^(beta - 1): v_mean = 2 opac beta P M,
//     v_conic = -opac beta (M_xx, 2M_xy, 2M_xz, M_yy, 2M_yz, M_zz),
//     v_opac = sum v h^beta, v_beta = opac ln2 sum v h^beta log2 h;
// the same VJP as voxel_vjp summed over the tile. sigma is evaluated in log2
// units (P scaled by log2 e) and the cut-off "sigma >= 0 and |opac e^-sigma| >=
// 1e-6" (Beta: "0 <= q < 1 and |opac h^beta| >= 1e-5") is one unsigned compare
// of the bits of q against qlim.
//
// Vector issue bounds it, so lanes must neither walk rows their primitive does
// not reach nor wait for lanes that walk more: the reached rows are a 64-bit
// mask per intersection (vox_row_mask), the chunk's intersections are sorted by
// its population (a counting sort in LDS), and the waves take 64 at a time, most
// rows first. Walking all 64 rows with only the lanes of one tile at a time
// active took 3.40 ms for 500k Beta primitives with a variance in 256^3 (4% of
// the pairs contribute), now 0.77, and 0.60 ms for 100k Gaussians in 128^3 (three
// quarters of the rows are reached), now 0.48 at the full issue rate. The
// register target is four waves a SIMD: the double-precision form at two (209
// registers) took 0.92 ms.
// ---------------------------------------------------------------------------
constexpr uint32_t kMomT = 8;

// The fused float32 kernels read each primitive's voxel-frame mean and
// inverse covariance from a double-precision frame, kFrame doubles per
// primitive (mean x y z, then the conic xx xy xz yy yz zz), computed from the
// world-frame parameters in double (vox_frame_kernel: the operator chain
// parameter transform -> volume mapping, in double). Gaussian offsets are
// formed as (v - hi) - lo with hi + lo the mean split into two floats, so the
// float32 rounding of a voxel coordinate (up to 1.5e-5 voxels at 256) never
// enters the profile. The Beta profile (1 - d^2)^beta is steep at its support
// edge when beta < 1 (there a change of 1e-7 in d^2 moves a term by up to
// ~3e-4), so Beta kernels form d^2 and 1 - d^2 in double from the frame.
constexpr int kFrame = 9;

__global__ void __launch_bounds__(256)
vox_frame_kernel(const float* __restrict__ means, const float* __restrict__ quats, const float* __restrict__ scales,
                 const double* __restrict__ ranges, const double* __restrict__ centers, uint32_t dx, uint32_t dy,
                 uint32_t dz, double eps, uint32_t N, double* __restrict__ frame) {
    const uint32_t n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    voxel_frame(means + 3 * size_t(n), quats + 4 * size_t(n), scales + 3 * size_t(n), ranges, centers, dx, dy, dz, eps,
                frame + kFrame * size_t(n));
}

// Mean of primitive G split into float hi + lo (lo = 0 without a frame).
__device__ __forceinline__ void vox_mean_split(const VoxArgs<float>& A, size_t G, float hi[3], float lo[3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (A.frame) {
            const double m = A.frame[kFrame * G + k];
            hi[k] = float(m);
            lo[k] = float(m - double(hi[k]));
        } else {
            hi[k] = A.means3d[3 * G + k];
            lo[k] = 0.f;
        }
    }
}

// Conic of primitive G (from the frame when there is one).
__device__ __forceinline__ void vox_conic(const VoxArgs<float>& A, size_t G, float P[6]) {
#pragma unroll
    for (int k = 0; k < 6; ++k) P[k] = A.frame ? float(A.frame[kFrame * G + 3 + k]) : A.conics[6 * G + k];
}

// Largest Beta d^2 whose term passes the cut-off, in double: |alpha| =
// |w| (1 - d^2)^beta >= 1e-5 for 0 <= d^2 <= qmax; negative when none does.
__device__ __forceinline__ double beta_qmax(float w, float beta) {
    const double aw = fabs(double(w));
    if (!(aw >= 1e-5) || !(beta > 0.f)) return -1.0;
    return 1.0 - exp2(log2(1e-5 / aw) / double(beta));
}

constexpr uint32_t kVoxPartial = 12;  // floats per intersection partial (11, or 12 with a variance)
constexpr uint32_t kMomThreads = kChunkThreads;
constexpr float kL2E = 1.4426950408889634f;

__device__ __forceinline__ uint32_t vox_qlim(float opac, float beta, bool is_beta) {
    if (!is_beta) {
        const float S = __log2f(fabsf(opac)) + 19.931568569324174f;  // log2(|opac| / 1e-6)
        return (opac != 0.f && S >= 0.f) ? __float_as_uint(S) + 1u : 0u;
    }
    const float S = __log2f(fabsf(opac)) + 16.609640474436812f;      // log2(|opac| / 1e-5)
    const float D = 1.f - __builtin_amdgcn_exp2f(-S / beta);
    if (!(opac != 0.f && S >= 0.f && D >= 0.f)) return 0u;
    return __float_as_uint(fminf(D, 0.99999994f)) + 1u;
}

// One intersection's quadratic form q = a dx^2 + bxy dx dy + bxz dx dz + cyy
// dy^2 + cyz dy dz + czz dz^2 (Gaussian: sigma in log2 units) and its mean.
struct VoxForm {
    float hi[3], lo[3], P[6];  // mean as hi + lo, conic
    float a, bxy, bxz, cyy, cyz, czz;
    float opac, beta;
    uint32_t qlim;  // float cut-off, or (WIDE) 1 when some term passes
    double qmax;    // WIDE: the cut-off on d^2
};

template <bool BETA, bool WIDE>
__device__ __forceinline__ VoxForm vox_form(const VoxArgs<float>& A, size_t G, const double* bound = nullptr) {
    VoxForm f;
    vox_mean_split(A, G, f.hi, f.lo);
    vox_conic(A, G, f.P);
    const float s = BETA ? 1.f : 0.5f * kL2E, t2 = BETA ? 2.f : kL2E;
    f.a = s * f.P[0];
    f.bxy = t2 * f.P[1];
    f.bxz = t2 * f.P[2];
    f.cyy = s * f.P[3];
    f.cyz = t2 * f.P[4];
    f.czz = s * f.P[5];
    f.opac = A.opac[G];
    f.beta = BETA ? A.betas[G] : 0.f;
    f.qmax = -1.0;
    if constexpr (WIDE) {
        f.qmax = bound ? *bound : beta_qmax(f.opac, f.beta);  // (given where it was computed before)
        f.qlim = f.qmax >= 0.0 ? 1u : 0u;
    } else {
        f.qlim = vox_qlim(f.opac, f.beta, BETA);
    }
    return f;
}

// Rows of 8 voxels (bit 8 z + y) of the tile whose first voxel centre is (x0, y0,
// z0) that can hold a voxel with q <= S. In the plane dz the ellipsoid is an
// ellipse in (x, y) of bound S - k dz^2 (k the Schur complement of czz) about
// the mean shifted by (xs, ys) dz; its extent in y over the row's eight columns
// is that of its upper and lower branches y(x) = (+-sqrt(4 cyy S - den x^2) - bxy
// x) / 2 cyy, den = 4 a cyy - bxy^2, at their extremes clamped to the columns. S
// is widened by 2e-3 and the columns and rows by 0.05 voxels. That covers the
// float32 rounding of q and of this bound while the determinant k den of the form
// is at least 1e-3 of the product of its diagonal: k is formed with den's error,
// so two cancellations of 1e-3 each, as in a thin disc's form, leave an error of
// a few percent of k. Forms that cancel further get every row, and a form no term
// of which passes none.
__device__ __forceinline__ uint64_t vox_row_mask(const VoxForm& f, float S, float x0, float y0, float z0) {
    if (!(fabsf(f.hi[0]) + fabsf(f.hi[1]) + fabsf(f.hi[2]) < 1e30f)) return ~0ull;  // (a NaN reaches every row)
    if (f.qlim == 0u) return 0ull;
    const float ac4 = 4.f * f.a * f.cyy, den = ac4 - f.bxy * f.bxy, inv = __builtin_amdgcn_rcpf(den);
    const float xs = (f.bxy * f.cyz - 2.f * f.cyy * f.bxz) * inv, ys = (f.bxy * f.bxz - 2.f * f.a * f.cyz) * inv;
    const float k = f.czz + 0.5f * (f.bxz * xs + f.cyz * ys);
    const float wide = S * 1.002f;
    if (!(f.a > 0.f) || !(f.cyy > 0.f) || !(den > 1e-3f * ac4) || !(k * den > 1e-3f * f.czz * ac4) ||
        !(wide * inv < 1e30f))
        return ~0ull;
    const float reach_x = __builtin_amdgcn_sqrtf(4.f * f.cyy * inv) * 1.001f;      // per sqrt of the plane's bound
    const float top = -0.5f * f.bxy * __builtin_amdgcn_rcpf(f.a) * __builtin_amdgcn_sqrtf(4.f * f.a * inv);
    const float half_c = 0.5f * __builtin_amdgcn_rcpf(f.cyy), c4 = 4.f * f.cyy;
    const float mx = f.hi[0] - x0, my = f.hi[1] - y0, mz = f.hi[2] - z0;  // the mean in voxels of this tile
    uint32_t half[2] = {0u, 0u};
#pragma unroll
    for (int z = 0; z < int(kMomT); ++z) {
        const float dz = float(z) - mz, Sz = fmaf(-k * dz, dz, wide);
        const float r = __builtin_amdgcn_sqrtf(fmaxf(Sz, 0.f)), rx = reach_x * r;
        const float cx = fmaf(xs, dz, mx), cy = fmaf(ys, dz, my);
        const float u0 = -0.05f - cx, u1 = float(kMomT - 1) + 0.05f - cx;
        const float xt = fminf(fmaxf(top * r, u0), u1), xb = fminf(fmaxf(-top * r, u0), u1);
        const float yt = (__builtin_amdgcn_sqrtf(fmaxf(c4 * Sz - den * xt * xt, 0.f)) - f.bxy * xt) * half_c;
        const float yb = -(__builtin_amdgcn_sqrtf(fmaxf(c4 * Sz - den * xb * xb, 0.f)) + f.bxy * xb) * half_c;
        const uint32_t lo = uint32_t(fminf(fmaxf(ceilf(cy + yb - 0.05f), 0.f), float(kMomT)));
        const uint32_t hi = uint32_t(fminf(fmaxf(floorf(cy + yt + 0.05f) + 1.f, 0.f), float(kMomT)));
        const bool hit = Sz >= 0.f && u0 <= rx && u1 >= -rx && hi > lo;
        half[z / 4] |= hit ? ((1u << hi) - (1u << lo)) << (8 * (z % 4)) : 0u;
    }
    return (uint64_t(half[1]) << 32) | half[0];
}

// VAR: the voxel adjoint becomes v + var_scale q alpha v_var (var_scale 2, or
// 0 when the variance is detached) and the partial's twelfth slot carries
// v_q = sum v_var alpha^2 (variance = sum q alpha^2). WIDE (Beta with a
// frame): q and h = 1 - q are formed in double from the frame, with the
// cut-off 0 <= q <= qmax decided in double, exactly as the fused forward does.
// With `partials` an intersection's gradient goes to its emission index, else
// it is added to the outputs with one atomic per field.
constexpr uint32_t kMomTiles = 8;  // tiles whose adjoints are staged together

template <uint32_t kMomChunk, bool BETA, bool VAR, bool WIDE>
__global__ void __launch_bounds__(kMomThreads) __attribute__((amdgpu_waves_per_eu(4)))
vox_bwd_moments_kernel(VoxArgs<float> A, const int64_t* __restrict__ isect_ids, const float* __restrict__ v_render,
                       const float* __restrict__ v_render_var, float var_scale,
                       float* __restrict__ v_xyz, float* __restrict__ v_c, float* __restrict__ v_opac,
                       float* __restrict__ v_beta, const int32_t* __restrict__ radii,
                       const uint32_t* __restrict__ cum, float* __restrict__ partials) {
    constexpr uint32_t T = kMomT, T3 = T * T * T;
    static_assert(!WIDE || BETA, "the double-precision form is for Beta profiles");
    __shared__ __align__(16) float sv[kMomTiles * T3];
    __shared__ __align__(16) float svv[VAR ? kMomTiles * T3 : 4];
    sorted_chunk<kMomChunk, kMomTiles, T3, WIDE>(
        isect_ids, A.n_isects, int64_t(A.ntx) * A.nty * A.ntz,
        [&](uint32_t slot, uint32_t tile, uint32_t p) {
            const uint32_t tx = tile % A.ntx, rest = tile / A.ntx, ty = rest % A.nty, tz = rest / A.nty;
            const uint32_t x = tx * T + p % T, j = ty * T + (p / T) % T, i = tz * T + p / (T * T);
            const bool in = i < A.dz && j < A.dy && x < A.dx;
            const size_t o = (size_t(i) * A.dy + j) * A.dx + x;
            sv[slot * T3 + p] = in ? v_render[o] : 0.f;
            if constexpr (VAR) svv[slot * T3 + p] = in ? v_render_var[o] : 0.f;
        },
        [&](uint32_t e, uint32_t tile, uint64_t& mask, double& bound) {
            const int32_t g = A.flatten[e];
            if (g < 0 || uint32_t(g) >= A.N) return false;
            const VoxForm f = vox_form<BETA, WIDE>(A, size_t(g));
            const uint32_t tx = tile % A.ntx, rest = tile / A.ntx;
            const float S = WIDE ? float(f.qmax) : __uint_as_float(f.qlim - 1u);
            bound = f.qmax;
            mask = vox_row_mask(f, S, float(tx * T) + 0.5f, float((rest % A.nty) * T) + 0.5f,
                                float((rest / A.nty) * T) + 0.5f);
            return true;
        },
        [&](uint32_t e, uint32_t tile, uint32_t slot, uint64_t rows, double bound, bool active) {
            const uint32_t staged = slot * T3;
            const uint32_t tx = tile % A.ntx, rest = tile / A.ntx, ty = rest % A.nty, tz = rest / A.nty;
            const float x0 = float(tx * T) + 0.5f, y0 = float(ty * T) + 0.5f, z0 = float(tz * T) + 0.5f;
            const int32_t g = A.flatten[e];
            const size_t G = size_t(g);
            const VoxForm f = vox_form<BETA, WIDE>(A, G, &bound);
            const float* P = f.P;
            const float opac = f.opac, beta = f.beta;
            double md[3] = {0.0, 0.0, 0.0}, Pd[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            if constexpr (WIDE) {
#pragma unroll
                for (int k = 0; k < 3; ++k) md[k] = A.frame[kFrame * G + k];
#pragma unroll
                for (int k = 0; k < 6; ++k) Pd[k] = A.frame[kFrame * G + 3 + k];
            }
            const double ad = Pd[0], bxyd = 2.0 * Pd[1], bxzd = 2.0 * Pd[2], cyyd = Pd[3], cyzd = 2.0 * Pd[4],
                         czzd = Pd[5];
            const double dx0d = double(x0) - md[0];
            const float kvar = VAR ? var_scale * A.unc[g] * opac : 0.f;  // d variance / d (alpha / w) factor
            const float bm1 = beta - 1.f;
            float m0 = 0.f, m_x = 0.f, m_y = 0.f, m_z = 0.f, mxx = 0.f, myy = 0.f, mzz = 0.f, mxy = 0.f, mxz = 0.f,
                  myz = 0.f, se = 0.f, sl = 0.f, vq = 0.f;
            const float dx0 = (x0 - f.hi[0]) - f.lo[0];
            float dxc[T];  // the columns' offsets, the same in every row
#pragma unroll
            for (uint32_t x = 0; x < T; ++x) dxc[x] = dx0 + float(x);
            while (rows) {
                const uint32_t bit = uint32_t(__builtin_ctzll(rows)), z = bit / T, y = bit % T;
                rows &= rows - 1ull;
                const double dzd = double(z0 + float(z)) - md[2], dyd = double(y0 + float(y)) - md[1];
                const float dz = WIDE ? float(dzd) : ((z0 + float(z)) - f.hi[2]) - f.lo[2];
                const float dy = WIDE ? float(dyd) : ((y0 + float(y)) - f.hi[1]) - f.lo[1];
                const float c1 = fmaf(f.bxy, dy, f.bxz * dz);
                const float c0 = fmaf(dy, fmaf(f.cyy, dy, f.cyz * dz), f.czz * dz * dz);
                const double c1d = fma(bxyd, dyd, bxzd * dzd);
                const double c0d = fma(dyd, fma(cyyd, dyd, cyzd * dzd), czzd * dzd * dzd);
                float r0 = 0.f, r1 = 0.f, r2 = 0.f, re = 0.f, rl = 0.f;
                // four voxels at a time: with the double-precision form all eight at once
                // take 209 registers (two waves a SIMD)
                constexpr int kStep = WIDE ? 4 : 8;
#pragma unroll 1
                for (int h4 = 0; h4 < 8; h4 += kStep) {
                    float v[kStep], vv[kStep];
#pragma unroll
                    for (int j = 0; j < kStep; j += 4) {
                        const float4 w = *reinterpret_cast<const float4*>(sv + staged + bit * T + h4 + j);
                        v[j] = w.x; v[j + 1] = w.y; v[j + 2] = w.z; v[j + 3] = w.w;
                        if constexpr (VAR) {
                            const float4 u = *reinterpret_cast<const float4*>(svv + staged + bit * T + h4 + j);
                            vv[j] = u.x; vv[j + 1] = u.y; vv[j + 2] = u.z; vv[j + 3] = u.w;
                        }
                    }
                    const double dx4 = dx0d + double(h4);
#pragma unroll
                    for (int x = 0; x < kStep; ++x) {
                        float dx, q, h;
                        bool in;
                        if constexpr (WIDE) {
                            const double dxd = dx4 + double(x);
                            const double qd = fma(dxd, fma(ad, dxd, c1d), c0d);
                            in = qd >= 0.0 && qd <= f.qmax;
                            h = float(1.0 - qd);
                            q = 0.f;
                            dx = float(dxd);
                        } else {
                            dx = dxc[x];
                            q = fmaf(dx, fmaf(f.a, dx, c1), c0);
                            in = __float_as_uint(q) < f.qlim;
                            h = 1.f - q;
                        }
                        float gv;
                        if constexpr (BETA) {
                            const float lg = __log2f(h);
                            const float hb = in ? __builtin_amdgcn_exp2f(bm1 * lg) : 0.f;  // h^(beta - 1)
                            float ve;
                            if constexpr (VAR) {
                                const float he = hb * h;  // h^beta = alpha / w
                                const float vj = fmaf(kvar * he, vv[x], v[x]);
                                gv = vj * hb;
                                ve = vj * he;
                                vq = fmaf(vv[x] * he, he, vq);
                            } else {
                                gv = v[x] * hb;
                                ve = gv * h;
                            }
                            re += ve;
                            rl = fmaf(ve, in ? lg : 0.f, rl);
                        } else {
                            const float e = in ? __builtin_amdgcn_exp2f(-q) : 0.f;
                            if constexpr (VAR) {
                                const float vj = fmaf(kvar * e, vv[x], v[x]);
                                gv = vj * e;
                                vq = fmaf(vv[x] * e, e, vq);
                            } else {
                                gv = v[x] * e;
                            }
                        }
                        r0 += gv;
                        const float gx = gv * dx;
                        r1 += gx;
                        r2 = fmaf(gx, dx, r2);
                    }
                }
                m0 += r0;
                m_x += r1;
                mxx += r2;
                m_y = fmaf(dy, r0, m_y);
                m_z = fmaf(dz, r0, m_z);
                myy = fmaf(dy * dy, r0, myy);
                mzz = fmaf(dz * dz, r0, mzz);
                myz = fmaf(dy * dz, r0, myz);
                mxy = fmaf(dy, r1, mxy);
                mxz = fmaf(dz, r1, mxz);
                if constexpr (BETA) {
                    se += re;
                    sl += rl;
                }
            }
            const float k = BETA ? 2.f * opac * beta : opac;
            const float gm[3] = {k * (P[0] * m_x + P[1] * m_y + P[2] * m_z), k * (P[1] * m_x + P[3] * m_y + P[4] * m_z),
                                 k * (P[2] * m_x + P[4] * m_y + P[5] * m_z)};
            float gc[6];
            if constexpr (BETA) {
                const float kb = -opac * beta;
                gc[0] = kb * mxx; gc[1] = 2.f * kb * mxy; gc[2] = 2.f * kb * mxz;
                gc[3] = kb * myy; gc[4] = 2.f * kb * myz; gc[5] = kb * mzz;
            } else {
                gc[0] = -0.5f * opac * mxx; gc[1] = -opac * mxy; gc[2] = -opac * mxz;
                gc[3] = -0.5f * opac * myy; gc[4] = -opac * myz; gc[5] = -0.5f * opac * mzz;
            }
            const float go = BETA ? se : m0, gb = BETA ? opac * 0.6931471805599453f * sl : 0.f;
            if (!active) {
            } else if (partials) {
                // the partial of this intersection at its emission index: the binning wrote
                // the primitive's tiles from cum[n] on, in z, y, x order over its tile box
                uint32_t lo[3], hi[3];
                if (box_3d(A.means3d, radii, G, T, A.ntx, A.nty, A.ntz, lo, hi) && tx >= lo[0] && tx < hi[0] &&
                    ty >= lo[1] && ty < hi[1] && tz >= lo[2] && tz < hi[2]) {
                    const uint32_t w = cum[G] + ((tz - lo[2]) * (hi[1] - lo[1]) + (ty - lo[1])) * (hi[0] - lo[0]) +
                                       (tx - lo[0]);
                    if (w < A.n_isects) {
                        float4* out = reinterpret_cast<float4*>(partials + kVoxPartial * size_t(w));
                        out[0] = make_float4(gm[0], gm[1], gm[2], gc[0]);
                        out[1] = make_float4(gc[1], gc[2], gc[3], gc[4]);
                        out[2] = make_float4(gc[5], go, gb, VAR ? opac * opac * vq : 0.f);
                    }
                }
            } else {
#pragma unroll
                for (int q = 0; q < 3; ++q) atomic_add(v_xyz + 3 * G + q, gm[q]);
#pragma unroll
                for (int q = 0; q < 6; ++q) atomic_add(v_c + 6 * G + q, gc[q]);
                atomic_add(v_opac + G, go);
                if constexpr (BETA) atomic_add(v_beta + G, gb);
            }
        });
}

// ---------------------------------------------------------------------------
// Fused float32 forward (8^3 tiles): kVoxFwdWaves waves per tile, wave k summing
// the k-th contiguous slice of the tile's list. Records (the mean and the
// quadratic form, the cut-off, opacity, beta) are built from the primitive
// arrays a batch of 64 ahead by the lanes and read back from LDS by broadcast.
// Gaussians (log2 units), which reach most of the tiles they are binned to: lane
// = one (y, z) row of 8 voxels, a lane forms the row terms once and evaluates q
// = a dx^2 + (bxy dy + bxz dz) dx + c(dy, dz) for its 8 voxels. Beta primitives,
// whose support fills 4% of the voxels of its tiles at 500k primitives in
// 256^3: lane = one voxel of each 4^3 octant, and octants that the support's
// bounding box does not reach are skipped by scalar branches (0.97 -> 0.52 ms
// there; 100k Gaussians in 128^3 take 0.38 ms). The slices' partial volumes are summed in LDS in wave order, so the result does
// not depend on scheduling.
// ---------------------------------------------------------------------------
constexpr int kVoxFwdWaves = 4;

// Gaussian record: the quadratic form in log2 units, the mean as hi + lo floats.
struct __align__(16) VoxRec {
    float mx, my, mz, a, bxy, bxz, cyy, cyz, czz, w, beta;
    uint32_t qlim;
    float lx, ly, lz, pad;  // the mean's float32 remainder (vox_mean_split)
};
static_assert(sizeof(VoxRec) == 64, "voxel record must be 64 bytes");

// Beta record: the mean and the conic (off-diagonals doubled) in double; a
// term passes the cut-off when 0 <= d^2 <= qmax; the octants it can reach.
struct __align__(16) VoxRecB {
    double mx, my, mz, a, bxy, bxz, cyy, cyz, czz, qmax;
    float w, beta;
    uint32_t octants, pad;  // bit 4 oz + 2 oy + ox
};
static_assert(sizeof(VoxRecB) == 96, "Beta voxel record must be 96 bytes");

template <bool BETA>
using VoxRecOf = typename std::conditional<BETA, VoxRecB, VoxRec>::type;

__device__ __forceinline__ VoxRec load_gauss_rec(const VoxArgs<float>& A, int32_t i, int32_t hi) {
    VoxRec r = {};
    if (i >= hi) return r;
    const int32_t g = A.flatten[i];
    if (g < 0 || uint32_t(g) >= A.N) return r;
    const size_t G = size_t(g);
    float h3[3], l3[3], P[6];
    vox_mean_split(A, G, h3, l3);
    vox_conic(A, G, P);
    constexpr float s = 0.5f * kL2E, t2 = kL2E;
    r.mx = h3[0];
    r.my = h3[1];
    r.mz = h3[2];
    r.lx = l3[0];
    r.ly = l3[1];
    r.lz = l3[2];
    r.a = s * P[0];
    r.bxy = t2 * P[1];
    r.bxz = t2 * P[2];
    r.cyy = s * P[3];
    r.cyz = t2 * P[4];
    r.czz = s * P[5];
    r.w = A.opac[g];
    r.qlim = vox_qlim(r.w, 0.f, false);
    return r;
}

// Octants of the tile at voxel (x0, y0, z0) that the ellipsoid d^2 <= qmax of a
// record can reach: its bounding box (half-extents sqrt(qmax C_kk), C the
// inverse of the conic), widened by 1e-3 and 0.05 voxels; every octant where
// the conic's determinant cancels.
__device__ __forceinline__ uint32_t vox_octants(const VoxRecB& r, float x0, float y0, float z0) {
    if (!(r.qmax >= 0.0)) return 0u;
    const float xx = float(r.a), yy = float(r.cyy), zz = float(r.czz), xy = 0.5f * float(r.bxy),
                xz = 0.5f * float(r.bxz), yz = 0.5f * float(r.cyz), S = float(r.qmax);
    const float c[3] = {yy * zz - yz * yz, xx * zz - xz * xz, xx * yy - xy * xy};
    const float det = xx * c[0] - xy * (xy * zz - xz * yz) + xz * (xy * yz - xz * yy);
    if (!(det > 1e-3f * xx * yy * zz)) return 0xffu;
    const float m[3] = {float(r.mx - double(x0)), float(r.my - double(y0)), float(r.mz - double(z0))};
    uint32_t part[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float e = __builtin_amdgcn_sqrtf(fmaxf(S * c[k] * __builtin_amdgcn_rcpf(det), 0.f)) * 1.001f + 0.05f;
        const float lo = m[k] - e, hi = m[k] + e;  // voxel centres of the tile at 0.5 .. 7.5
        part[k] = (lo <= 3.5f && hi >= 0.5f ? 1u : 0u) | (lo <= 7.5f && hi >= 4.5f ? 2u : 0u);
        if (!(e < 1e30f)) part[k] = 3u;
    }
    const uint32_t row = part[0], plane = (part[1] & 1u ? row : 0u) | (part[1] & 2u ? row << 2 : 0u);
    return (part[2] & 1u ? plane : 0u) | (part[2] & 2u ? plane << 4 : 0u);
}

// Needs the frame (the fused entry points require it).
__device__ __forceinline__ VoxRecB load_beta_rec(const VoxArgs<float>& A, int32_t i, int32_t hi, float x0, float y0,
                                                 float z0) {
    VoxRecB r = {};
    if (i >= hi) return r;
    const int32_t g = A.flatten[i];
    if (g < 0 || uint32_t(g) >= A.N) return r;
    const double* f = A.frame + kFrame * size_t(g);
    r.mx = f[0];
    r.my = f[1];
    r.mz = f[2];
    r.a = f[3];
    r.bxy = 2.0 * f[4];
    r.bxz = 2.0 * f[5];
    r.cyy = f[6];
    r.cyz = 2.0 * f[7];
    r.czz = f[8];
    r.w = A.opac[g];
    r.beta = A.betas[g];
    r.qmax = beta_qmax(r.w, r.beta);
    r.octants = vox_octants(r, x0, y0, z0);
    return r;
}

// Entry i's record for the tile whose corner is (x0, y0, z0).
template <bool BETA>
__device__ __forceinline__ VoxRecOf<BETA> load_vox_rec(const VoxArgs<float>& A, int32_t i, int32_t hi, float x0,
                                                       float y0, float z0) {
    if constexpr (BETA)
        return load_beta_rec(A, i, hi, x0, y0, z0);
    else
        return load_gauss_rec(A, i, hi);
}

// The uncertainty of the primitive a list entry names (0 past the list).
__device__ __forceinline__ float load_vox_unc(const VoxArgs<float>& A, int32_t i, int32_t hi) {
    if (i >= hi) return 0.f;
    const int32_t g = A.flatten[i];
    return (g < 0 || uint32_t(g) >= A.N) ? 0.f : A.unc[g];
}

// VAR also accumulates the variance sum q alpha^2 (q the primitive's
// uncertainty, staged beside the record) and sums it in a second LDS phase.
// Beta terms form d^2 and 1 - d^2 in double (the record's mean and conic),
// decide the cut-off on d^2 in double and take the power in float32.
template <bool BETA, bool VAR>
__global__ void __launch_bounds__(kVoxFwdWaves * kWave) __attribute__((amdgpu_waves_per_eu(4)))
vox_fwd_fused_kernel(VoxArgs<float> A, float* __restrict__ out, float* __restrict__ out_var) {
    constexpr uint32_t T = kMomT;
    using R = VoxRecOf<BETA>;
    __shared__ R stage[kVoxFwdWaves][kWave];
    __shared__ float stage_q[VAR ? kVoxFwdWaves : 1][kWave];
    __shared__ float part[kVoxFwdWaves][T * T * T];
    const uint32_t blk = blockIdx.x;
    const uint32_t nt = A.ntx * A.nty * A.ntz;
    int32_t start = A.offsets[blk];
    int32_t end = (blk + 1 == nt) ? int32_t(A.n_isects) : A.offsets[blk + 1];
    start = max(0, min(start, int32_t(A.n_isects)));
    end = max(start, min(end, int32_t(A.n_isects)));
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int32_t per = (end - start + kVoxFwdWaves - 1) / kVoxFwdWaves;
    const int32_t lo = min(end, start + int32_t(wave) * per), hi = min(end, lo + per);
    const uint32_t tx = blk % A.ntx, rest = blk / A.ntx, ty = rest % A.nty, tz = rest / A.nty;
    // a lane's voxels: Gaussian row (0 .. 7, ly, lz); Beta (lx + 4 ox, ly + 4 oy, lz + 4 oz) for octant 4 oz + 2 oy + ox
    constexpr uint32_t kEdge = BETA ? 4 : T;
    const uint32_t lx = BETA ? lane % 4 : 0u, ly = BETA ? (lane / 4) % 4 : lane % T, lz = BETA ? lane / 16 : lane / T;
    const float x0 = float(tx * T), y0 = float(ty * T), z0 = float(tz * T);
    const float px = x0 + float(lx) + 0.5f, py = y0 + float(ly) + 0.5f, pz = z0 + float(lz) + 0.5f;
    auto place = [&](uint32_t k) -> uint32_t {  // the tile voxel of accumulator k
        if constexpr (BETA)
            return ((lz + kEdge * (k >> 2)) * T + ly + kEdge * ((k >> 1) & 1u)) * T + lx + kEdge * (k & 1u);
        else
            return (lz * T + ly) * T + k;
    };
    float acc[T], acc_var[T];
#pragma unroll
    for (uint32_t x = 0; x < T; ++x) {
        acc[x] = 0.f;
        acc_var[x] = 0.f;
    }
    R* slot = stage[wave];
    R next = load_vox_rec<BETA>(A, lo + int32_t(lane), hi, x0, y0, z0);
    float next_q = VAR ? load_vox_unc(A, lo + int32_t(lane), hi) : 0.f;
    for (int32_t base = lo; base < hi; base += kWave) {
        wave_lds_sync();
        slot[lane] = next;
        if constexpr (VAR) stage_q[wave][lane] = next_q;
        wave_lds_sync();
        next = load_vox_rec<BETA>(A, base + kWave + int32_t(lane), hi, x0, y0, z0);
        if constexpr (VAR) next_q = load_vox_unc(A, base + kWave + int32_t(lane), hi);
        const int32_t n = min(int32_t(kWave), hi - base);
        for (int32_t j = 0; j < n; ++j) {
            const R r = slot[j];
            const float unc = VAR ? stage_q[VAR ? wave : 0][j] : 0.f;
            auto add = [&](uint32_t k, float e) {
                if constexpr (VAR) {
                    const float alpha = e * r.w;
                    acc[k] += alpha;
                    acc_var[k] = fmaf(unc * alpha, alpha, acc_var[k]);
                } else {
                    acc[k] = fmaf(e, r.w, acc[k]);
                }
            };
            if constexpr (BETA) {
                const uint32_t octants = __builtin_amdgcn_readfirstlane(r.octants);  // every lane reads the same record
                if (octants == 0u) continue;
                const double dx0 = double(px) - r.mx, dy0 = double(py) - r.my, dz0 = double(pz) - r.mz;
#pragma unroll
                for (uint32_t o = 0; o < 8; o += 2) {
                    if (((octants >> o) & 3u) == 0u) continue;
                    const double dy = (o & 2u) ? dy0 + 4.0 : dy0, dz = (o & 4u) ? dz0 + 4.0 : dz0;
                    const double c1 = fma(r.bxy, dy, r.bxz * dz);
                    const double c0 = fma(dy, fma(r.cyy, dy, r.cyz * dz), r.czz * dz * dz);
#pragma unroll
                    for (uint32_t ox = 0; ox < 2; ++ox) {
                        if (!((octants >> (o + ox)) & 1u)) continue;
                        const double dx = ox ? dx0 + 4.0 : dx0;
                        const double q = fma(dx, fma(r.a, dx, c1), c0);
                        const float e = __builtin_amdgcn_exp2f(r.beta * __log2f(float(1.0 - q)));
                        add(o + ox, (q >= 0.0 && q <= r.qmax) ? e : 0.f);
                    }
                }
            } else {
                if (r.qlim == 0u) continue;  // wave-uniform
                const float dy = (py - r.my) - r.ly, dz = (pz - r.mz) - r.lz, dx0 = (px - r.mx) - r.lx;
                const float c1 = fmaf(r.bxy, dy, r.bxz * dz);
                const float c0 = fmaf(dy, fmaf(r.cyy, dy, r.cyz * dz), r.czz * dz * dz);
#pragma unroll
                for (uint32_t x = 0; x < T; ++x) {
                    const float dx = dx0 + float(x);
                    const float q = fmaf(dx, fmaf(r.a, dx, c1), c0);
                    const float e = __builtin_amdgcn_exp2f(-q);
                    add(x, __float_as_uint(q) < r.qlim ? e : 0.f);
                }
            }
        }
    }
#pragma unroll
    for (uint32_t x = 0; x < T; ++x) part[wave][place(x)] = acc[x];
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < T * T * T; p += blockDim.x) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < kVoxFwdWaves; ++k) v += part[k][p];
        const uint32_t k = tx * T + p % T, j = ty * T + (p / T) % T, i = tz * T + p / (T * T);
        if (i < A.dz && j < A.dy && k < A.dx) out[(size_t(i) * A.dy + j) * A.dx + k] = v;
    }
    if constexpr (VAR) {
        __syncthreads();  // the mean's partial volumes are consumed
#pragma unroll
        for (uint32_t x = 0; x < T; ++x) part[wave][place(x)] = acc_var[x];
        __syncthreads();
        for (uint32_t p = threadIdx.x; p < T * T * T; p += blockDim.x) {
            float v = 0.f;
#pragma unroll
            for (int k = 0; k < kVoxFwdWaves; ++k) v += part[k][p];
            const uint32_t k = tx * T + p % T, j = ty * T + (p / T) % T, i = tz * T + p / (T * T);
            if (i < A.dz && j < A.dy && k < A.dx) out_var[(size_t(i) * A.dy + j) * A.dx + k] = v;
        }
    }
}

// Per-primitive sums of the intersection partials [cum[n], cum[n+1]) in emission
// order (deterministic; no atomics): four lanes per primitive, lane c adding float4
// c (of three) of its partials one after another, kBatch loads ahead of the sums.
// (One lane per primitive, a partial's three loads at a time: 65 us for 2.9M
// partials of 100k primitives, now 31, and 21 us for 285k of 3k, now 6.)
constexpr uint32_t kReduceLanes = 4, kReduceThreads = 256;

__global__ void __launch_bounds__(kReduceThreads)
vox_partials_reduce_kernel(const uint32_t* __restrict__ cum, const float* __restrict__ partials, uint32_t N,
                           uint32_t n_isects, float* __restrict__ v_xyz, float* __restrict__ v_c,
                           float* __restrict__ v_opac, float* __restrict__ v_beta, float* __restrict__ v_unc) {
    constexpr uint32_t kBatch = 16, kGroups = kReduceThreads / kReduceLanes;  // loads in flight; primitives per round
    const uint32_t column = threadIdx.x % kReduceLanes;
    const float4* part = reinterpret_cast<const float4*>(partials);
    static_assert(kVoxPartial == 12, "a partial is three float4");
    if (column == 3) return;
    for (uint32_t n = blockIdx.x * kGroups + threadIdx.x / kReduceLanes; n < N; n += gridDim.x * kGroups) {
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        const uint32_t lo = min(cum[n], n_isects), hi = min(cum[n + 1], n_isects);
        for (uint32_t j = lo; j < hi; j += kBatch) {
            float4 p[kBatch];
#pragma unroll
            for (uint32_t k = 0; k < kBatch; ++k)
                p[k] = j + k < hi ? part[3 * size_t(j + k) + column] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (uint32_t k = 0; k < kBatch; ++k) {
                acc.x += p[k].x;
                acc.y += p[k].y;
                acc.z += p[k].z;
                acc.w += p[k].w;
            }
        }
        if (column == 0) {  // v_mean, v_conic xx
            v_xyz[3 * size_t(n)] = acc.x;
            v_xyz[3 * size_t(n) + 1] = acc.y;
            v_xyz[3 * size_t(n) + 2] = acc.z;
            v_c[6 * size_t(n)] = acc.w;
        } else if (column == 1) {  // v_conic xy, xz, yy, yz
            v_c[6 * size_t(n) + 1] = acc.x;
            v_c[6 * size_t(n) + 2] = acc.y;
            v_c[6 * size_t(n) + 3] = acc.z;
            v_c[6 * size_t(n) + 4] = acc.w;
        } else {  // v_conic zz, v_opac, v_beta, v_q
            v_c[6 * size_t(n) + 5] = acc.x;
            v_opac[n] = acc.y;
            if (v_beta) v_beta[n] = acc.z;
            if (v_unc) v_unc[n] = acc.w;
        }
    }
}

// ---------------------------------------------------------------------------
// Operator kernels for 8^3 tiles that skip what a primitive does not reach (the
// exponential or power in double is most of a pair's cost; 20k Gaussians in 72 x
// 64 x 56 contribute to a sixth of the voxels of their tiles). One voxel per
// thread over the whole list took 210 us there and a wave per intersection 373 us;
// these take 166 and 160.
// ---------------------------------------------------------------------------
// Whether every parameter of a primitive is finite.
template <typename S, bool BETA>
__device__ __forceinline__ bool all_finite(const Prim3D<S>& p) {
    bool ok = isfinite(p.x) && isfinite(p.y) && isfinite(p.z) && isfinite(p.opac) && (!BETA || isfinite(p.beta));
#pragma unroll
    for (int k = 0; k < 6; ++k) ok = ok && isfinite(p.c[k]);
    return ok;
}

// The float form of a primitive and the bound S on its q (Gaussian: q = sigma)
// beyond which no term passes the cut-off; false when none can (a finite primitive
// whose weight is surely below it). The bounds by rows and octants give a primitive
// with a NaN or an infinity every voxel, so that it shows where its pairs pass.
template <typename S, bool BETA>
__device__ __forceinline__ bool op_form(const Prim3D<S>& p, VoxForm& f, float& bound) {
    const float w = fabsf(float(p.opac)), cut = BETA ? 1e-5f : 1e-6f;
    if (w < 0.999f * cut && all_finite<S, BETA>(p)) return false;
    const float s = BETA ? 1.f : 0.5f, t2 = BETA ? 2.f : 1.f;
    f.hi[0] = float(p.x);
    f.hi[1] = float(p.y);
    f.hi[2] = float(p.z);
    f.a = s * float(p.c[0]);
    f.bxy = t2 * float(p.c[1]);
    f.bxz = t2 * float(p.c[2]);
    f.cyy = s * float(p.c[3]);
    f.cyz = t2 * float(p.c[4]);
    f.czz = s * float(p.c[5]);
    f.qlim = 1u;
    if (BETA) {
        const float D = 1.f - __builtin_amdgcn_exp2f(__log2f(cut / w) / float(p.beta));
        bound = p.beta > S(0) ? fminf(1.f, 1.002f * D + 1e-4f) : 1.f;
    } else {
        bound = 1.001f * __logf(w / cut) + 1e-4f;
    }
    return true;
}

// Octants (bit 4 oz + 2 oy + ox) of the tile whose first voxel is (x0, y0, z0) that
// the ellipsoid q <= S can reach, by its bounding box; every octant of forms
// that cancel or are not finite.
__device__ __forceinline__ uint32_t form_octants(const VoxForm& f, float S, float x0, float y0, float z0) {
    const float xy = 0.5f * f.bxy, xz = 0.5f * f.bxz, yz = 0.5f * f.cyz;
    const float c[3] = {f.cyy * f.czz - yz * yz, f.a * f.czz - xz * xz, f.a * f.cyy - xy * xy};
    const float det = f.a * c[0] - xy * (xy * f.czz - xz * yz) + xz * (xy * yz - xz * f.cyy);
    if (!(f.a > 0.f) || !(det > 1e-3f * f.a * f.cyy * f.czz) || !(S >= 0.f)) return 0xffu;
    const float m[3] = {f.hi[0] - x0, f.hi[1] - y0, f.hi[2] - z0};
    uint32_t part[3];
    bool far = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float e = __builtin_amdgcn_sqrtf(S * c[k] * __builtin_amdgcn_rcpf(det)) * 1.002f + 0.05f;
        const float lo = m[k] - e, hi = m[k] + e;  // voxel centres of the tile at 0.5 .. 7.5
        part[k] = (lo <= 3.5f && hi >= 0.5f ? 1u : 0u) | (lo <= 7.5f && hi >= 4.5f ? 2u : 0u);
        if (!(e < 1e9f)) part[k] = 3u;
        far = far || !(fabsf(m[k]) < 1e9f);
    }
    if (far) return 0xffu;
    const uint32_t row = part[0], plane = (part[1] & 1u ? row : 0u) | (part[1] & 2u ? row << 2 : 0u);
    return (part[2] & 1u ? plane : 0u) | (part[2] & 2u ? plane << 4 : 0u);
}

template <typename S>
__device__ __forceinline__ Prim3D<S> load_prim3(const VoxArgs<S>& A, int32_t g, bool beta) {
    Prim3D<S> p;
    const size_t G = size_t(g);
    p.x = A.means3d[3 * G];
    p.y = A.means3d[3 * G + 1];
    p.z = A.means3d[3 * G + 2];
#pragma unroll
    for (int k = 0; k < 6; ++k) p.c[k] = A.conics[6 * G + k];
    p.opac = A.opac[g];
    p.beta = beta ? A.betas[g] : S(0);
    return p;
}

// Forward: kVoxFwdWaves waves share a tile's list as in the fused forward; lane =
// one voxel of each 4^3 octant, octants not reached skipped by scalar branches.
template <typename S, bool BETA, bool VAR>
__global__ void __launch_bounds__(kVoxFwdWaves * kWave) __attribute__((amdgpu_waves_per_eu(3)))
vox_fwd_octants_kernel(VoxArgs<S> A, S* __restrict__ out, S* __restrict__ out_var) {
    constexpr uint32_t T = kMomT;
    __shared__ Prim3D<S> stage[kVoxFwdWaves][kWave];
    __shared__ S stage_q[VAR ? kVoxFwdWaves : 1][kWave];
    __shared__ S part[kVoxFwdWaves][T * T * T];
    const uint32_t blk = blockIdx.x, nt = A.ntx * A.nty * A.ntz;
    int32_t start = A.offsets[blk];
    int32_t end = (blk + 1 == nt) ? int32_t(A.n_isects) : A.offsets[blk + 1];
    start = max(0, min(start, int32_t(A.n_isects)));
    end = max(start, min(end, int32_t(A.n_isects)));
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const uint32_t tx = blk % A.ntx, rest = blk / A.ntx, ty = rest % A.nty, tz = rest / A.nty;
    const uint32_t lx = lane % 4, ly = (lane / 4) % 4, lz = lane / 16;
    const S px = S(tx * T + lx) + S(0.5), py = S(ty * T + ly) + S(0.5), pz = S(tz * T + lz) + S(0.5);
    S acc[8], acc_var[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) acc[o] = acc_var[o] = S(0);
    for (int32_t base = start + int32_t(wave) * kWave; base < end; base += kVoxFwdWaves * kWave) {
        uint32_t octants = 0;
        Prim3D<S> r = {};
        S q = S(0);
        if (base + int32_t(lane) < end) {
            const int32_t g = A.flatten[base + int32_t(lane)];
            if (g >= 0 && uint32_t(g) < A.N) {  // out-of-range ids contribute nothing
                r = load_prim3(A, g, BETA);
                if constexpr (VAR) q = A.unc[g];
                VoxForm f;
                float bound;
                if (op_form<S, BETA>(r, f, bound))
                    octants = form_octants(f, bound, float(tx * T), float(ty * T), float(tz * T));
            }
        }
        wave_lds_sync();
        stage[wave][lane] = r;
        if constexpr (VAR) stage_q[wave][lane] = q;
        wave_lds_sync();
        const int32_t n = min(int32_t(kWave), end - base);
        for (int32_t j = 0; j < n; ++j) {
            const uint32_t reach = __builtin_amdgcn_readlane(octants, j);
            if (reach == 0u) continue;
            const Prim3D<S> p = stage[wave][j];
            const S unc = VAR ? stage_q[VAR ? wave : 0][j] : S(0);
#pragma unroll
            for (uint32_t o = 0; o < 8; ++o) {
                if (!((reach >> o) & 1u)) continue;
                S vis, alpha;
                const bool keep =
                    eval_profile3<S, BETA>(p, px + S(4 * (o & 1u)), py + S(2 * (o & 2u)), pz + S(o & 4u), vis, alpha);
                if (!keep) alpha = S(0);
                acc[o] += alpha;
                if constexpr (VAR) acc_var[o] += (keep ? unc : S(0)) * alpha * alpha;
            }
        }
    }
#pragma unroll
    for (int v = 0; v < (VAR ? 2 : 1); ++v) {
#pragma unroll
        for (uint32_t o = 0; o < 8; ++o)
            part[wave][((lz + (o & 4u)) * T + ly + 2 * (o & 2u)) * T + lx + 4 * (o & 1u)] = v ? acc_var[o] : acc[o];
        __syncthreads();
        for (uint32_t p = threadIdx.x; p < T * T * T; p += kVoxFwdWaves * kWave) {
            S sum = S(0);
#pragma unroll
            for (int k = 0; k < kVoxFwdWaves; ++k) sum += part[k][p];
            const uint32_t k = tx * T + p % T, j = ty * T + (p / T) % T, i = tz * T + p / (T * T);
            if (i < A.dz && j < A.dy && k < A.dx) (v ? out_var : out)[(size_t(i) * A.dy + j) * A.dx + k] = sum;
        }
        if (VAR && v == 0) __syncthreads();  // the mean's partial volumes are consumed
    }
}

// Gaussian: sigma, Beta: q, in the roundings eval_profile3 compiles to: the float32
// terms of a thin primitive cancel, and another order would give it another exponent.
template <typename S, bool BETA>
__device__ __forceinline__ S triple_form(const Prim3D<S>& p, S dx, S dy, S dz) {
    const S sq = Math<S>::fma(p.c[5] * dz, dz, Math<S>::fma(p.c[0] * dx, dx, p.c[3] * dy * dy));
    const S xy = p.c[1] * dx, xz = p.c[2] * dx, yz = p.c[4] * dy;
    if constexpr (BETA) return sq + S(2) * Math<S>::fma(yz, dz, Math<S>::fma(xy, dy, xz * dz));
    return Math<S>::fma(yz, dz, Math<S>::fma(xz, dz, Math<S>::fma(xy, dy, S(0.5) * sq)));
}

// VJP: one lane per intersection over the rows it reaches (sorted_chunk), the
// moments of vox_bwd_moments_kernel in S, one atomic per field.
constexpr uint32_t kOpTiles = 4;

template <typename S, uint32_t CHUNK, bool BETA, bool VAR>
__global__ void __launch_bounds__(kChunkThreads) __attribute__((amdgpu_waves_per_eu(3)))
vox_bwd_rows_kernel(VoxArgs<S> A, const int64_t* __restrict__ isect_ids, const S* __restrict__ v_render,
                    const S* __restrict__ v_var, const S* __restrict__ unc, S* __restrict__ v_xyz,
                    S* __restrict__ v_c, S* __restrict__ v_opac, S* __restrict__ v_beta, S* __restrict__ v_q) {
    constexpr uint32_t T = kMomT, T3 = T * T * T;
    __shared__ __align__(16) S sv[kOpTiles * T3];
    __shared__ __align__(16) S svv[VAR ? kOpTiles * T3 : 2];
    sorted_chunk<CHUNK, kOpTiles, T3, false>(
        isect_ids, A.n_isects, int64_t(A.ntx) * A.nty * A.ntz,
        [&](uint32_t slot, uint32_t tile, uint32_t p) {
            const uint32_t tx = tile % A.ntx, rest = tile / A.ntx, ty = rest % A.nty, tz = rest / A.nty;
            const uint32_t x = tx * T + p % T, j = ty * T + (p / T) % T, i = tz * T + p / (T * T);
            const bool in = i < A.dz && j < A.dy && x < A.dx;
            const size_t o = (size_t(i) * A.dy + j) * A.dx + x;
            sv[slot * T3 + p] = in ? v_render[o] : S(0);
            if constexpr (VAR) svv[slot * T3 + p] = in ? v_var[o] : S(0);
        },
        [&](uint32_t e, uint32_t tile, uint64_t& mask, double&) {
            const int32_t g = A.flatten[e];
            if (g < 0 || uint32_t(g) >= A.N) return false;
            VoxForm f;
            float bound;
            if (!op_form<S, BETA>(load_prim3(A, g, BETA), f, bound)) return false;
            const uint32_t tx = tile % A.ntx, rest = tile / A.ntx, ty = rest % A.nty, tz = rest / A.nty;
            mask = vox_row_mask(f, bound, float(tx * T) + 0.5f, float(ty * T) + 0.5f, float(tz * T) + 0.5f);
            // the rows of the volume (a pair past it is none)
            const uint32_t ny = ty * T < A.dy ? min(T, A.dy - ty * T) : 0u, nz = tz * T < A.dz ? min(T, A.dz - tz * T) : 0u;
            mask &= nz == 0u ? 0ull : (0x0101010101010101ull * ((1u << ny) - 1u)) & (~0ull >> (8u * (T - nz)));
            return mask != 0ull;
        },
        [&](uint32_t e, uint32_t tile, uint32_t slot, uint64_t rows, double, bool active) {
            const uint32_t tx = tile % A.ntx, rest = tile / A.ntx, ty = rest % A.nty, tz = rest / A.nty;
            const int32_t g = A.flatten[e];
            const Prim3D<S> p = load_prim3(A, g, BETA);
            const S q2 = VAR && unc ? S(2) * unc[g] : S(0);
            double m0 = 0.0, m_x = 0.0, m_y = 0.0, m_z = 0.0, mxx = 0.0, myy = 0.0, mzz = 0.0, mxy = 0.0, mxz = 0.0,
                   myz = 0.0, sl = 0.0, vq = 0.0;
            while (rows) {
                const uint32_t bit = uint32_t(__builtin_ctzll(rows)), z = bit / T, y = bit % T;
                rows &= rows - 1ull;
                const S dy = (S(ty * T + y) + S(0.5)) - p.y, dz = (S(tz * T + z) + S(0.5)) - p.z;
                S r0 = S(0), r1 = S(0), r2 = S(0), rm = S(0), rl = S(0), rq = S(0);
                const S* row = sv + slot * T3 + bit * T;
                const S* rowv = svv + (VAR ? slot * T3 + bit * T : 0);
#pragma unroll 2
                for (uint32_t j = 0; j < T; ++j) {
                    const S dx = (S(tx * T + j) + S(0.5)) - p.x;
                    const S q = triple_form<S, BETA>(p, dx, dy, dz);
                    S v = row[j];
                    const S vv = VAR ? rowv[VAR ? j : 0] : S(0);
                    if constexpr (BETA) {
                        if (q < S(0) || q >= S(1)) continue;
                        const S h = S(1) - q, vis = Math<S>::pow(h, p.beta), alpha = p.opac * vis;
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
                        const S vis = Math<S>::exp(-q), alpha = p.opac * vis;
                        const bool keep = !(q < S(0) || fabs(alpha) < S(1e-6));
                        if constexpr (VAR) {
                            row_sum(rq, vq, keep ? vv * alpha * alpha : S(0));
                            v += q2 * alpha * vv;
                        }
                        const S gv = keep ? v * vis : S(0);
                        r0 += gv;
                        r1 += gv * dx;
                        r2 += gv * dx * dx;
                    }
                }
                m0 += BETA ? rm : r0;
                m_x += r1;
                mxx += r2;
                const double ey = dy, ez = dz;
                m_y += ey * r0;
                m_z += ez * r0;
                myy += ey * ey * r0;
                mzz += ez * ez * r0;
                myz += ey * ez * r0;
                mxy += ey * r1;
                mxz += ez * r1;
                sl += rl;
                vq += rq;
            }
            if (!active) return;
            // no pair: an infinite parameter times an empty sum would be a NaN
            if (m0 == 0.0 && vq == 0.0 && !all_finite<S, BETA>(p)) return;
            const size_t G = size_t(g);
            const double k = BETA ? S(2) * p.opac * p.beta : p.opac, kc = BETA ? -p.opac * p.beta : S(-0.5) * p.opac;
            atomic_add(v_xyz + 3 * G, S(k * (p.c[0] * m_x + p.c[1] * m_y + p.c[2] * m_z)));
            atomic_add(v_xyz + 3 * G + 1, S(k * (p.c[1] * m_x + p.c[3] * m_y + p.c[4] * m_z)));
            atomic_add(v_xyz + 3 * G + 2, S(k * (p.c[2] * m_x + p.c[4] * m_y + p.c[5] * m_z)));
            atomic_add(v_c + 6 * G, S(kc * mxx));
            atomic_add(v_c + 6 * G + 1, S(2.0 * kc * mxy));
            atomic_add(v_c + 6 * G + 2, S(2.0 * kc * mxz));
            atomic_add(v_c + 6 * G + 3, S(kc * myy));
            atomic_add(v_c + 6 * G + 4, S(2.0 * kc * myz));
            atomic_add(v_c + 6 * G + 5, S(kc * mzz));
            atomic_add(v_opac + G, S(m0));
            if constexpr (BETA) atomic_add(v_beta + G, S(sl));
            if constexpr (VAR)
                if (v_q) atomic_add(v_q + G, S(vq));
        });
}

inline int check_vox_tile(uint32_t T, uint32_t ntx, uint32_t nty, uint32_t ntz, uint32_t dx,
                          uint32_t dy, uint32_t dz) {
    R2S_REQUIRE(T >= 1 && T * T * T <= 1024, "tile_size %u must satisfy 1 <= tile_size^3 <= 1024", T);
    R2S_REQUIRE(uint64_t(ntx) * T >= dx && uint64_t(nty) * T >= dy && uint64_t(ntz) * T >= dz,
                "tile grid does not cover the volume");
    return R2S_OK;
}

inline uint32_t vox_threads(uint32_t T) { return ((T * T * T + kWave - 1) / kWave) * kWave; }

template <typename S>
VoxArgs<S> make_vox_args(const void* means3d, const void* conics, const void* opac, const void* betas,
                         const void* unc, const int32_t* offsets, const int32_t* flatten,
                         uint32_t n_isects, uint32_t N, uint32_t dx, uint32_t dy, uint32_t dz,
                         uint32_t T, uint32_t ntx, uint32_t nty, uint32_t ntz) {
    return VoxArgs<S>{(const S*)means3d, (const S*)conics, (const S*)opac, (const S*)betas,
                      (const S*)unc, offsets, flatten, n_isects, N, dx, dy, dz, T, ntx, nty, ntz};
}

// Whether an operator forward of 8^3 tiles takes the octant kernel, whose waves share
// a tile's list and skip the octants a primitive does not reach. It wins on long lists
// (142k intersections on 8 tiles, Beta: float32 609 us against 2674, float64 684 against
// 3050) and loses where lists are short for what a primitive covers: float32, 18.7k
// intersections on 512 tiles, primitives reaching into the next tile, 31 us against 23.
// Launches of up to 600 tiles need longer lists for it (float64, 3604 intersections on
// 125 tiles: 51 us against 21).
template <typename S>
inline bool fwd_by_octants(uint32_t n_isects, uint64_t prims, uint64_t tiles) {
    const double wide = std::is_same<S, double>::value ? 64.0 : 24.0;
    double list = 4.0 + wide * tile_overhang(n_isects, prims, 3);
    if (tiles <= 600) list = 2.0 * list + 32.0;
    return double(n_isects) >= list * double(tiles);
}

// Whether an operator VJP of 8^3 tiles takes the kernel with a lane per intersection:
// it needs intersections enough to fill the chip, more where a lane walks its whole
// tile of 512 voxels, and lists long enough that a chunk meets few tiles; the general
// kernel has a wave per intersection. float64 Beta: 142k intersections on 8 tiles 20 us
// against 280, 1895 on 4096 tiles 8698 against 26.
template <typename S>
inline bool vjp_by_rows(uint32_t n_isects, uint64_t prims, uint64_t tiles, bool beta) {
    const double over = tile_overhang(n_isects, prims, 3);
    const double wide = std::is_same<S, double>::value && !beta ? 32.0 : 64.0;
    return n_isects >= 4e3 + 48e3 * over && double(n_isects) >= (4.0 + wide * over) * double(tiles);
}

}  // namespace r2s

using namespace r2s;

extern "C" int r2s_voxelize_to_voxels_fwd(int dtype, const void* means3d, const void* conics,
                                          const void* opacities, const void* betas,
                                          const void* uncertainties, const int32_t* tile_offsets,
                                          const int32_t* flatten_ids, uint32_t n_isects, uint32_t N,
                                          uint32_t dim_x, uint32_t dim_y, uint32_t dim_z,
                                          uint32_t tile_size, uint32_t n_tiles_x,
                                          uint32_t n_tiles_y, uint32_t n_tiles_z, void* render,
                                          void* render_var, r2s_stream_t stream) {
    if (int rc = check_vox_tile(tile_size, n_tiles_x, n_tiles_y, n_tiles_z, dim_x, dim_y, dim_z))
        return rc;
    const uint64_t blocks = uint64_t(n_tiles_x) * n_tiles_y * n_tiles_z;
    if (blocks == 0) return R2S_OK;
    const bool beta = betas != nullptr, var = render_var != nullptr;
    R2S_REQUIRE(!var || uncertainties != nullptr, "render_var requires uncertainties");
    const uint32_t threads = vox_threads(tile_size);
    const size_t shm = vox_lds_bytes(dtype, std::min(threads, kVoxBatch));
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        auto A = make_vox_args<S>(means3d, conics, opacities, betas, uncertainties, tile_offsets,
                                  flatten_ids, n_isects, N, dim_x, dim_y, dim_z, tile_size,
                                  n_tiles_x, n_tiles_y, n_tiles_z);
        if (tile_size == kMomT && fwd_by_octants<S>(n_isects, N, blocks)) {
            auto k = beta ? (var ? vox_fwd_octants_kernel<S, true, true> : vox_fwd_octants_kernel<S, true, false>)
                          : (var ? vox_fwd_octants_kernel<S, false, true> : vox_fwd_octants_kernel<S, false, false>);
            k<<<uint32_t(blocks), kVoxFwdWaves * kWave, 0, stream>>>(A, (S*)render, (S*)render_var);
            return check_launch("voxelize_to_voxels_fwd");
        }
        auto k = beta ? (var ? vox_fwd_kernel<S, true, true> : vox_fwd_kernel<S, true, false>)
                      : (var ? vox_fwd_kernel<S, false, true> : vox_fwd_kernel<S, false, false>);
        k<<<uint32_t(blocks), threads, shm, stream>>>(A, (S*)render, (S*)render_var);
        return check_launch("voxelize_to_voxels_fwd");
    });
}

extern "C" int r2s_voxelize_to_voxels_bwd(int dtype, const void* means3d, const void* conics,
                                          const void* opacities, const void* betas,
                                          const int32_t* tile_offsets, const int32_t* flatten_ids,
                                          uint32_t n_isects, uint32_t N, uint32_t dim_x,
                                          uint32_t dim_y, uint32_t dim_z, uint32_t tile_size,
                                          uint32_t n_tiles_x, uint32_t n_tiles_y,
                                          uint32_t n_tiles_z, const void* v_render, void* v_means3d,
                                          void* v_conics, void* v_opacities, void* v_betas,
                                          r2s_stream_t stream) {
    if (int rc = check_vox_tile(tile_size, n_tiles_x, n_tiles_y, n_tiles_z, dim_x, dim_y, dim_z))
        return rc;
    const bool beta = betas != nullptr;
    R2S_REQUIRE(!beta || v_betas != nullptr, "v_betas is required with betas");
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        if (int rc = fill_zeros<S>({{v_means3d, 3 * size_t(N)}, {v_conics, 6 * size_t(N)}, {v_opacities, N},
                                    {beta ? v_betas : nullptr, N}}, stream))
            return rc;
        const uint64_t blocks = uint64_t(n_tiles_x) * n_tiles_y * n_tiles_z;
        if (blocks == 0 || n_isects == 0 || N == 0) return R2S_OK;
        const uint32_t threads = vox_threads(tile_size);
        const size_t shm = vox_lds_bytes(dtype, std::min(threads, kVoxBatch));
        auto A = make_vox_args<S>(means3d, conics, opacities, betas, nullptr, tile_offsets,
                                  flatten_ids, n_isects, N, dim_x, dim_y, dim_z, tile_size,
                                  n_tiles_x, n_tiles_y, n_tiles_z);
        auto k = beta ? vox_bwd_tile_kernel<S, true> : vox_bwd_tile_kernel<S, false>;
        k<<<uint32_t(blocks), threads, shm, stream>>>(A, (const S*)v_render, (S*)v_means3d,
                                                      (S*)v_conics, (S*)v_opacities, (S*)v_betas);
        return check_launch("voxelize_to_voxels_bwd");
    });
}

extern "C" int r2s_voxelize_to_voxels_bwd_per_gaussian(
    int dtype, const void* means3d, const void* conics, const void* opacities, const void* betas,
    const int64_t* isect_ids, const int32_t* flatten_ids, uint32_t n_isects, uint32_t N,
    uint32_t dim_x, uint32_t dim_y, uint32_t dim_z, uint32_t tile_size, uint32_t n_tiles_x,
    uint32_t n_tiles_y, uint32_t n_tiles_z, const void* v_render, const void* v_render_var,
    const void* uncertainties, void* v_means3d, void* v_conics, void* v_opacities, void* v_betas,
    void* v_uncertainties, r2s_stream_t stream) {
    if (int rc = check_vox_tile(tile_size, n_tiles_x, n_tiles_y, n_tiles_z, dim_x, dim_y, dim_z))
        return rc;
    const bool beta = betas != nullptr;
    R2S_REQUIRE(!beta || v_betas != nullptr, "v_betas is required with betas");
    return dispatch_dtype(dtype, [&](auto tag) {
        using S = decltype(tag);
        if (int rc = fill_zeros<S>({{v_means3d, 3 * size_t(N)}, {v_conics, 6 * size_t(N)}, {v_opacities, N},
                                    {beta ? v_betas : nullptr, N}, {v_uncertainties, N}}, stream))
            return rc;
        if (n_isects == 0 || N == 0) return R2S_OK;
        auto A = make_vox_args<S>(means3d, conics, opacities, betas, nullptr, nullptr, flatten_ids,
                                  n_isects, N, dim_x, dim_y, dim_z, tile_size, n_tiles_x,
                                  n_tiles_y, n_tiles_z);
        if constexpr (std::is_same<S, float>::value) {
            const uint64_t n_tiles = uint64_t(n_tiles_x) * n_tiles_y * n_tiles_z;
            if (tile_size == kMomT && !v_render_var && n_tiles < (1ull << 31)) {  // moments form
                const bool few = n_isects <= kFewIsects;
                auto km = beta ? (few ? vox_bwd_moments_kernel<256, true, false, false>
                                      : vox_bwd_moments_kernel<512, true, false, false>)
                               : (few ? vox_bwd_moments_kernel<256, false, false, false>
                                      : vox_bwd_moments_kernel<512, false, false, false>);
                km<<<ceil_div(n_isects, few ? 256 : 512), kMomThreads, 0, stream>>>(
                    A, isect_ids, (const float*)v_render, nullptr, 0.f, (float*)v_means3d, (float*)v_conics,
                    (float*)v_opacities, (float*)v_betas, nullptr, nullptr, nullptr);
                return check_launch("voxelize_to_voxels_bwd_per_gaussian");
            }
        }
        const uint64_t tiles = uint64_t(n_tiles_x) * n_tiles_y * n_tiles_z;
        if (tile_size == kMomT && tiles < (1ull << 31) && vjp_by_rows<S>(n_isects, N, tiles, beta)) {
            const bool var = v_render_var != nullptr;
            const auto launch = [&](auto chunk) {
                constexpr uint32_t CHUNK = decltype(chunk)::value;
                auto k = beta ? (var ? vox_bwd_rows_kernel<S, CHUNK, true, true> : vox_bwd_rows_kernel<S, CHUNK, true, false>)
                              : (var ? vox_bwd_rows_kernel<S, CHUNK, false, true>
                                     : vox_bwd_rows_kernel<S, CHUNK, false, false>);
                k<<<ceil_div(n_isects, CHUNK), kChunkThreads, 0, stream>>>(
                    A, isect_ids, (const S*)v_render, (const S*)v_render_var, (const S*)uncertainties, (S*)v_means3d,
                    (S*)v_conics, (S*)v_opacities, (S*)v_betas, (S*)v_uncertainties);
            };
            if (n_isects <= kFewIsects) launch(std::integral_constant<uint32_t, 256>{});
            else launch(std::integral_constant<uint32_t, 512>{});
            return check_launch("voxelize_to_voxels_bwd_per_gaussian");
        }
        constexpr uint32_t waves = 4;
        auto k = beta ? vox_bwd_isect_kernel<S, true> : vox_bwd_isect_kernel<S, false>;
        k<<<std::min<uint32_t>(ceil_div(n_isects, waves), kIsectBlocks), waves * kWave, 0, stream>>>(
            A, isect_ids, (const S*)v_render, (const S*)v_render_var,
            v_render_var ? (const S*)uncertainties : nullptr, (S*)v_means3d, (S*)v_conics,
            (S*)v_opacities, (S*)v_betas, v_render_var ? (S*)v_uncertainties : nullptr);
        return check_launch("voxelize_to_voxels_bwd_per_gaussian");
    });
}

extern "C" size_t r2s_voxel_partials_bytes(uint32_t n_isects) {
    return size_t(n_isects) * kVoxPartial * sizeof(float);
}

extern "C" int r2s_voxel_frame(const float* means, const float* quats, const float* scales, const double* ranges,
                               const double* centers, uint32_t dim_x, uint32_t dim_y, uint32_t dim_z, double eps,
                               uint32_t N, double* frame, r2s_stream_t stream) {
    if (N == 0) return R2S_OK;
    R2S_REQUIRE(means && quats && scales && ranges && centers && frame, "voxel_frame: null argument");
    vox_frame_kernel<<<ceil_div(N, 256), 256, 0, stream>>>(means, quats, scales, ranges, centers, dim_x, dim_y,
                                                           dim_z, eps, N, frame);
    return check_launch("voxel_frame");
}

extern "C" int r2s_voxelize_fused_vjp(const float* means3d, const double* frame, const float* conics,
                                      const float* opacities,
                                      const float* betas, const float* uncertainties, const int32_t* radii,
                                      const uint32_t* tile_cum, const int64_t* isect_ids, const int32_t* flatten_ids,
                                      uint32_t n_isects, uint32_t N, uint32_t dim_x, uint32_t dim_y, uint32_t dim_z,
                                      uint32_t tile_size, uint32_t n_tiles_x, uint32_t n_tiles_y, uint32_t n_tiles_z,
                                      const float* v_render, const float* v_render_var, int detach, float* partials,
                                      size_t partials_bytes, float* v_means3d, float* v_conics, float* v_opacities,
                                      float* v_betas, float* v_uncertainties, r2s_stream_t stream) {
    if (int rc = check_vox_tile(tile_size, n_tiles_x, n_tiles_y, n_tiles_z, dim_x, dim_y, dim_z)) return rc;
    R2S_REQUIRE(tile_size == kMomT, "the fused voxel VJP takes %u^3 tiles (got %u)", kMomT, tile_size);
    R2S_REQUIRE(uint64_t(n_tiles_x) * n_tiles_y * n_tiles_z < (1ull << 31), "too many tiles");
    R2S_REQUIRE(partials_bytes >= r2s_voxel_partials_bytes(n_isects), "partials buffer too small: %zu < %zu",
                partials_bytes, r2s_voxel_partials_bytes(n_isects));
    const bool beta = betas != nullptr, var = v_render_var != nullptr;
    R2S_REQUIRE(!beta || v_betas != nullptr, "v_betas is required with betas");
    R2S_REQUIRE(!var || (uncertainties != nullptr && v_uncertainties != nullptr),
                "a variance adjoint needs uncertainties and v_uncertainties");
    R2S_REQUIRE(frame != nullptr, "voxelize_fused_vjp: the double-precision frame is required");
    if (N == 0) return R2S_OK;
    if (n_isects > 0) {
        auto A = make_vox_args<float>(means3d, conics, opacities, betas, uncertainties, nullptr, flatten_ids,
                                      n_isects, N, dim_x, dim_y, dim_z, tile_size, n_tiles_x, n_tiles_y, n_tiles_z);
        A.frame = frame;
        const bool few = n_isects <= kFewIsects;
        auto km = beta ? (var ? (few ? vox_bwd_moments_kernel<256, true, true, true>
                                     : vox_bwd_moments_kernel<512, true, true, true>)
                              : (few ? vox_bwd_moments_kernel<256, true, false, true>
                                     : vox_bwd_moments_kernel<512, true, false, true>))
                       : (var ? (few ? vox_bwd_moments_kernel<256, false, true, false>
                                     : vox_bwd_moments_kernel<512, false, true, false>)
                              : (few ? vox_bwd_moments_kernel<256, false, false, false>
                                     : vox_bwd_moments_kernel<512, false, false, false>));
        km<<<ceil_div(n_isects, few ? 256 : 512), kMomThreads, 0, stream>>>(
            A, isect_ids, v_render, v_render_var, detach ? 0.f : 2.f, nullptr, nullptr, nullptr, nullptr, radii,
            tile_cum, partials);
        if (int rc = check_launch("voxelize_fused_vjp")) return rc;
    }
    vox_partials_reduce_kernel<<<std::min(ceil_div(N, kReduceThreads / kReduceLanes), 1u << 22), kReduceThreads, 0,
                                 stream>>>(tile_cum, partials, N, n_isects, v_means3d, v_conics, v_opacities,
                                           beta ? v_betas : nullptr, var ? v_uncertainties : nullptr);
    return check_launch("voxelize_fused_vjp_reduce");
}

extern "C" int r2s_voxelize_fused_fwd(const float* means3d, const double* frame, const float* conics,
                                      const float* opacities,
                                      const float* betas, const float* uncertainties, const int32_t* tile_offsets,
                                      const int32_t* flatten_ids, uint32_t n_isects, uint32_t N, uint32_t dim_x,
                                      uint32_t dim_y, uint32_t dim_z, uint32_t tile_size, uint32_t n_tiles_x,
                                      uint32_t n_tiles_y, uint32_t n_tiles_z, float* render, float* render_var,
                                      r2s_stream_t stream) {
    if (int rc = check_vox_tile(tile_size, n_tiles_x, n_tiles_y, n_tiles_z, dim_x, dim_y, dim_z)) return rc;
    R2S_REQUIRE(tile_size == kMomT, "the fused voxel forward takes %u^3 tiles (got %u)", kMomT, tile_size);
    const bool var = render_var != nullptr;
    R2S_REQUIRE(!var || uncertainties != nullptr, "render_var requires uncertainties");
    const uint64_t n_tiles = uint64_t(n_tiles_x) * n_tiles_y * n_tiles_z;
    R2S_REQUIRE(n_tiles < (1ull << 31), "too many tiles");
    if (n_tiles == 0) return R2S_OK;
    R2S_REQUIRE(frame != nullptr, "voxelize_fused_fwd: the double-precision frame is required");
    auto A = make_vox_args<float>(means3d, conics, opacities, betas, uncertainties, tile_offsets, flatten_ids,
                                  n_isects, N, dim_x, dim_y, dim_z, tile_size, n_tiles_x, n_tiles_y, n_tiles_z);
    A.frame = frame;
    auto k = betas ? (var ? vox_fwd_fused_kernel<true, true> : vox_fwd_fused_kernel<true, false>)
                   : (var ? vox_fwd_fused_kernel<false, true> : vox_fwd_fused_kernel<false, false>);
    k<<<uint32_t(n_tiles), kVoxFwdWaves * kWave, 0, stream>>>(A, render, render_var);
    return check_launch("voxelize_fused_fwd");
}
