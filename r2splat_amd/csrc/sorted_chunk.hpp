// A workgroup's chunk of tile-sorted intersections, its tiles staged together
// and its intersections worked on in order of how many rows of their tile they
// reach: the frame of the lane-per-intersection backward kernels.
#pragma once

#include "common.hpp"

namespace r2s {

constexpr uint32_t kChunkThreads = 256;
constexpr uint32_t kNoTile = 0xffffffffu;
// Chunks hold 512 intersections, or 256 where those would leave most compute
// units with a single workgroup; a shorter chunk's rows are sorted less finely.
// VJPs of 30k to 13M intersections, 512 against 256 in each: float64 32-pixel tiles
// 588 us against 432 at 92k and 1115 against 1315 at 1.5M, 8^3 voxels 176 against 130
// at 151k, 196 against 243 at 456k (the widest miss of this line) and 496 against 600
// at 1.5M; the others are within 12% of one another above the line.
constexpr uint32_t kFewIsects = 1u << 19;

// How far the mean primitive reaches beyond one tile along an axis, in tiles, at
// most one, from n_isects intersections of `prims` primitives on tiles of `axes`
// dimensions. The operator kernels that work row by row are chosen by it and by
// the lengths of the lists: a primitive that fills its tiles has no rows to skip.
inline double tile_overhang(uint32_t n_isects, uint64_t prims, int axes) {
    const double tiles = prims ? double(n_isects) / double(prims) : 0.0;
    return std::min(1.0, std::max(0.0, (axes == 2 ? std::sqrt(tiles) : std::cbrt(tiles)) - 1.0));
}

// Takes intersections [e0, e0 + CHUNK) of the list (ids: their tile ids,
// ascending; those outside [0, n_tiles) are skipped), for at most TILES distinct
// tiles at a time:
//   stage(slot, tile, p)  every thread, p = 0 .. PER_TILE - 1 over the threads:
//                         stages element p of a tile into its slot (0 .. TILES - 1);
//   rows(i, tile, mask, extra) -> bool  the rows of the tile that intersection i
//                         reaches, as a mask of up to 64 (false: nothing to do),
//                         and with EXTRA a value that work() needs again;
//   work(i, tile, slot, mask, extra, active)  one lane per intersection, whole
//                         waves (inactive lanes repeat an active one's
//                         intersection with no rows and must not write).
// The intersections are counted by row count in LDS (a counting sort; ties in
// any order, so work() must not depend on the order) and the waves take 64 at a
// time, most rows first: a wave runs as long as its longest lane.
template <uint32_t CHUNK, uint32_t TILES, uint32_t PER_TILE, bool EXTRA, typename Stage, typename Rows, typename Work>
__device__ __forceinline__ void sorted_chunk(const int64_t* __restrict__ ids, uint32_t n_isects, int64_t tile_count,
                                             Stage&& stage, Rows&& rows_of, Work&& work) {
    constexpr uint32_t kPer = CHUNK / kChunkThreads, kWaves = kChunkThreads / kWave;
    static_assert(CHUNK % kChunkThreads == 0 && CHUNK <= 65536, "whole rounds, 16-bit chunk entries");
    __shared__ uint64_t masks[CHUNK];
    __shared__ double extras[EXTRA ? CHUNK : 1];
    __shared__ uint32_t tile_of[CHUNK], sorted[CHUNK];  // sorted: chunk entry | slot << 16
    __shared__ uint32_t first_of[CHUNK + 1];            // first entry of the chunk's k-th tile
    __shared__ uint32_t hist[kWave + 1], first[kWave + 1], wave_tiles[kPer * kWaves], n_items, next_item;
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t e0 = blockIdx.x * CHUNK, n_here = min(CHUNK, n_isects - e0);
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t i = k * kChunkThreads + threadIdx.x;
        int64_t id = -1;
        if (i < n_here) id = ids[e0 + i];
        tile_of[i] = id >= 0 && id < tile_count ? uint32_t(id) : kNoTile;
    }
    __syncthreads();
    uint64_t starts[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t i = k * kChunkThreads + threadIdx.x;
        starts[k] = __ballot(i < n_here && (i == 0 || tile_of[i] != tile_of[i - 1]));
        if (lane == 0) wave_tiles[k * kWaves + wave] = uint32_t(__popcll(starts[k]));
    }
    __syncthreads();
    uint32_t place[kPer], n_tiles = 0;  // place: which of the chunk's tiles an entry belongs to
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        uint32_t before = 0;
        for (uint32_t w = 0; w < k * kWaves + wave; ++w) before += wave_tiles[w];
        place[k] = before + uint32_t(__popcll(starts[k] & (~0ull >> (kWave - 1 - lane)))) - 1u;
        if ((starts[k] >> lane) & 1ull) first_of[place[k]] = k * kChunkThreads + threadIdx.x;
    }
    for (uint32_t w = 0; w < kPer * kWaves; ++w) n_tiles += wave_tiles[w];
    for (uint32_t t0 = 0; t0 < n_tiles; t0 += TILES) {
        __syncthreads();  // first_of is written; the previous tiles are consumed
        const uint32_t n_staged = min(TILES, n_tiles - t0);
        for (uint32_t p = threadIdx.x; p < n_staged * PER_TILE; p += kChunkThreads) {
            const uint32_t slot = p / PER_TILE, tile = tile_of[first_of[t0 + slot]];
            if (tile != kNoTile) stage(slot, tile, p % PER_TILE);
        }
        if (threadIdx.x <= kWave) hist[threadIdx.x] = 0u;
        __syncthreads();
        uint64_t mask[kPer];
        double extra[kPer];
        uint32_t rank[kPer];
        bool mine[kPer];
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k) {
            const uint32_t i = k * kChunkThreads + threadIdx.x;
            mask[k] = 0ull;
            extra[k] = 0.0;
            rank[k] = 0u;
            mine[k] = i < n_here && place[k] >= t0 && place[k] < t0 + n_staged && tile_of[i] != kNoTile &&
                      rows_of(e0 + i, tile_of[i], mask[k], extra[k]);
            if (mine[k]) rank[k] = atomicAdd(&hist[kWave - uint32_t(__popcll(mask[k]))], 1u);
        }
        __syncthreads();
        if (wave == 0) {  // starts of the row counts 64 .. 0
            const uint32_t c = hist[lane], incl = wave_scan(c);
            first[lane] = incl - c;
            if (lane == kWave - 1) {
                first[kWave] = incl;
                n_items = incl + hist[kWave];
                next_item = 0u;
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kPer; ++k)
            if (mine[k]) {
                const uint32_t at = first[kWave - uint32_t(__popcll(mask[k]))] + rank[k];
                masks[at] = mask[k];
                if constexpr (EXTRA) extras[at] = extra[k];
                sorted[at] = (k * kChunkThreads + threadIdx.x) | ((place[k] - t0) << 16);
            }
        __syncthreads();
        for (;;) {
            uint32_t c = 0;
            if (lane == 0) c = atomicAdd(&next_item, uint32_t(kWave));
            c = __builtin_amdgcn_readfirstlane(c);
            if (c >= n_items) break;
            const bool active = c + lane < n_items;
            const uint32_t at = active ? c + lane : c, it = sorted[at], i = it & 0xffffu;
            work(e0 + i, tile_of[i], it >> 16, active ? masks[at] : 0ull, EXTRA ? extras[EXTRA ? at : 0] : 0.0, active);
        }
    }
}

// The sums of work(): a lane adds a whole tile's terms by itself, so float terms are
// summed over eight columns of a row and those sums in double (one float sum over a
// 16- or 32-pixel tile was 2.5 to 6 times as far from 64 bits as a wave's tree of
// sums, these are as near). Double terms go straight to the total.
template <typename S>
__device__ __forceinline__ void row_sum(S& row, double& total, S term) {
    if constexpr (sizeof(S) == sizeof(double)) total += term;
    else row += term;
}

}  // namespace r2s
