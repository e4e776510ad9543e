// search.hip - compact-grid neighbour search with a Morton-ordered structure-of-arrays reorder.
//
// Reference: ParticleSearch::FindNeighbors (VFD/Source/Simulation/DFSPH/ParticleSearch/ParticleSearch.cu:29-195,
// ParticleSearchKernels.cu:4-193). Same grid (cell = support radius, origin two cells below the particles' minimum
// cell, 8^3 Morton meta blocks), same strict test 0 < d^2 < R^2, same cap of 70 and the same traversal order (27 cells
// z,y,x). Different from the reference by design:
//   - particles are physically reordered by (cell, original id) every step, so every later neighbour loop reads
//     contiguous cells; the reference keeps particles in input order and only sorts index arrays;
//   - the order inside a cell is ascending original id (deterministic) instead of atomicAdd order;
//   - lists hold slot indices, tile by tile in a transposed [j][i] layout with a fixed capacity of 70 per particle.
#include <algorithm>
#include <mutex>

#include "device.h"
#include "kernels.h"

namespace vfd {

__device__ __forceinline__ unsigned spread3(unsigned x) {  // low 10 bits of x to every third bit
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}
// cell (cx,cy,cz) -> meta-block linear index * 512 + Morton code inside the 8^3 block (ParticleSearchKernels.cu:24-38)
__device__ __forceinline__ uint32_t cell_key(const SceneGrid& g, uint32_t cx, uint32_t cy, uint32_t cz) {
    const uint32_t mx = cx >> 3, my = cy >> 3, mz = cz >> 3;
    const uint32_t lin = (mz * g.meta[1] + my) * g.meta[0] + mx;
    const uint32_t m = (spread3(cz & 7u) << 2) | (spread3(cy & 7u) << 1) | spread3(cx & 7u);
    return g.cellBase + lin * kMetaBlock + m;
}

// ComputeMinMaxKernel (ParticleSearchKernels.cu:40-62): integer cell bounds floor(x / R). Each tile writes its
// bounds to part[tile * 6 + a]; k_minmax_finish reduces a scene's tiles (no atomics on a single address).
__global__ void __launch_bounds__(kTile) k_minmax(const float4* __restrict__ pos, const SceneParams* __restrict__ P,
                                                  const uint32_t* __restrict__ tileScene, int* part,
                                                  long long* stamps) {
    note_time(stamps, kStampStart);
    __shared__ int sh[kTile / kWave][6];
    const TileCtx c = tile_ctx(tileScene, P);
    const float R = P[c.s].R;
    int v[6] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN};
    if (c.valid) {
        const float4 x = pos[c.i];
        v[0] = v[3] = (int)floorf(x.x / R);
        v[1] = v[4] = (int)floorf(x.y / R);
        v[2] = v[5] = (int)floorf(x.z / R);
    }
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        v[a] = wave_min_i(v[a]);
        v[3 + a] = wave_max_i(v[3 + a]);
    }
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < 6; ++a) sh[w][a] = v[a];
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        int m = sh[0][a];
        for (int j = 1; j < (int)(kTile / kWave); ++j) m = a < 3 ? min(m, sh[j][a]) : max(m, sh[j][a]);
        part[(size_t)blockIdx.x * 6 + a] = m;
    }
}

__global__ void __launch_bounds__(kTile) k_minmax_finish(const SceneParams* __restrict__ P,
                                                         const int* __restrict__ part, int* mm) {
    __shared__ int sh[kTile / kWave][6];
    const uint32_t s = blockIdx.x;
    const SceneParams& p = P[s];
    int v[6] = {INT_MAX, INT_MAX, INT_MAX, INT_MIN, INT_MIN, INT_MIN};
    for (uint32_t t = p.tileBegin + threadIdx.x; t < p.tileEnd; t += kTile)
#pragma unroll
        for (int a = 0; a < 6; ++a) v[a] = a < 3 ? min(v[a], part[(size_t)t * 6 + a]) : max(v[a], part[(size_t)t * 6 + a]);
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        v[a] = wave_min_i(v[a]);
        v[3 + a] = wave_max_i(v[3 + a]);
    }
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < 6; ++a) sh[w][a] = v[a];
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        int m = sh[0][a];
        for (int j = 1; j < (int)(kTile / kWave); ++j) m = a < 3 ? min(m, sh[j][a]) : max(m, sh[j][a]);
        mm[6 * s + a] = m;
    }
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__device__ __forceinline__ uint32_t clampu(int v, uint32_t hi) { return v < 0 ? 0u : ((uint32_t)v >= hi ? hi - 1u : (uint32_t)v); }

// InsertParticlesMortonKernel (ParticleSearchKernels.cu:64-78): cell key and arbitrary rank inside the cell.
// Coordinates are clamped into the grid so that a non-finite position cannot index outside the cell arrays.
__global__ void __launch_bounds__(kTile) k_insert(const float4* __restrict__ pos, const SceneParams* __restrict__ P,
                                                  const SceneGrid* __restrict__ G,
                                                  const uint32_t* __restrict__ tileScene, uint32_t* cellOf,
                                                  uint32_t* rank, uint32_t* cellCount) {
    const TileCtx c = tile_ctx(tileScene, P);
    if (!c.valid) return;
    const SceneGrid& g = G[c.s];
    const float4 x = pos[c.i];
    const float fx = (x.x - g.gridMin[0]) * g.gridDelta[0];
    const float fy = (x.y - g.gridMin[1]) * g.gridDelta[1];
    const float fz = (x.z - g.gridMin[2]) * g.gridDelta[2];
    const uint32_t key = cell_key(g, clampu((int)fx, g.dims[0]), clampu((int)fy, g.dims[1]), clampu((int)fz, g.dims[2]));
    cellOf[c.i] = key;
    rank[c.i] = atomicAdd(&cellCount[key], 1u);
}

// Places every particle's original id at its provisional slot (CountingSortIndicesKernel, :80-91).
__global__ void __launch_bounds__(kTile) k_scatter_ids(const SceneParams* __restrict__ P,
                                                       const SceneGrid* __restrict__ G,
                                                       const uint32_t* __restrict__ tileScene,
                                                       const uint32_t* __restrict__ cellOf,
                                                       const uint32_t* __restrict__ rank,
                                                       const uint32_t* __restrict__ cellStart,
                                                       const uint32_t* __restrict__ idOld, uint32_t* tmpId) {
    const TileCtx c = tile_ctx(tileScene, P);
    if (!c.valid) return;
    const uint32_t key = cellOf[c.i];
    tmpId[(uint32_t)((int32_t)cellStart[key] + G[c.s].startCorr) + rank[c.i]] = idOld[c.i];
}

// Final slot = cell start + number of cell members with a smaller original id. Moves the persistent state there.
__global__ void __launch_bounds__(kTile) k_reorder(const SceneParams* __restrict__ P, const SceneGrid* __restrict__ G,
                                                   const uint32_t* __restrict__ tileScene,
                                                   const uint32_t* __restrict__ cellOf,
                                                   const uint32_t* __restrict__ cellStart,
                                                   const uint32_t* __restrict__ cellCount,
                                                   const uint32_t* __restrict__ tmpId, const float4* __restrict__ posIn,
                                                   const float4* __restrict__ velIn, const float4* __restrict__ dvIn,
                                                   const float* __restrict__ dkIn, const uint32_t* __restrict__ idIn,
                                                   float4* posOut, float4* velOut, float4* dvOut, float* dkOut,
                                                   uint32_t* idOut) {
    const TileCtx c = tile_ctx(tileScene, P);
    if (!c.valid) return;
    const uint32_t key = cellOf[c.i];
    const uint32_t start = (uint32_t)((int32_t)cellStart[key] + G[c.s].startCorr);
    const uint32_t n = cellCount[key];
    const uint32_t me = idIn[c.i];
    uint32_t r = 0;
    for (uint32_t t = 0; t < n; ++t) r += tmpId[start + t] < me ? 1u : 0u;
    const uint32_t dst = start + r;
    posOut[dst] = posIn[c.i];
    velOut[dst] = velIn[c.i];
    dvOut[dst] = dvIn[c.i];
    dkOut[dst] = dkIn[c.i];
    idOut[dst] = me;
}

#ifndef VFD_SEARCH_UNROLL
#define VFD_SEARCH_UNROLL 8
#endif
constexpr uint32_t kSearchUnroll = VFD_SEARCH_UNROLL;

// The block's neighbour total and longest list to stats[block], which the step's report sums up. (A 64-bit atomic add
// and maximum per wave on the scene's two counters were what the kernel waited for, about 14 ns a wave whatever the
// search did: 866 -> 659 us on 2 million particles, 92 -> 65 us on 123,000.)
__device__ __forceinline__ void note_neighbors(uint32_t cnt, uint32_t block, uint2* stats) {
    __shared__ uint2 sh[kTile / kWave];
    uint32_t tot = cnt, mx = cnt;
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        tot += (uint32_t)__shfl_xor((int)tot, o, kWave);
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, o, kWave));
    }
    if ((threadIdx.x & (kWave - 1)) == 0) sh[threadIdx.x / kWave] = make_uint2(tot, mx);
    __syncthreads();
    if (threadIdx.x == 0) {
        uint2 t = sh[0];
        for (uint32_t w = 1; w < kTile / kWave; ++w) t = make_uint2(t.x + sh[w].x, max(t.y, sh[w].y));
        stats[block] = t;
    }
}

// FindNeighbors (ParticleSearch.cu:95-195; kernels ParticleSearchKernels.cu:93-193) in one traversal per particle:
// the 27 cells in z, y, x order, each cell's particles in slot order (= ascending original id), strict
// 0 < d^2 < R^2, at most kMaxNeighbors; out(cnt, t) receives the cnt-th neighbour. The ranges of all 27 cells are
// requested before the first candidate is loaded. The three cells of a row (x - 1, x, x + 1 at fixed y, z) form one
// stream of candidates, loaded kSearchUnroll at a time from clamped positions (every load stays inside a range) with
// no branch around the loads; a candidate past the row's end or past the cap is simply not accepted, so the first
// kMaxNeighbors in the reference's order are kept. Cells whose box lies farther than the support radius from the
// particle (by a 0.1% margin: no candidate there can pass d^2 < R^2) are skipped: about a quarter of the 27 on
// average, corner and edge cells, without changing the list.
template <class Out>
__device__ __forceinline__ uint32_t neighbor_list(const TileCtx& c, const SceneParams* __restrict__ P,
                                                  const SceneGrid* __restrict__ G, const float4* __restrict__ pos,
                                                  const uint32_t* __restrict__ cellStart,
                                                  const uint32_t* __restrict__ cellCount, Out&& out) {
    const SceneGrid& g = G[c.s];
    const float R2 = P[c.s].R * P[c.s].R;
    const float4 xi = pos[c.i];
    const float ux = (xi.x - g.gridMin[0]) * g.gridDelta[0], uy = (xi.y - g.gridMin[1]) * g.gridDelta[1];
    const float uz = (xi.z - g.gridMin[2]) * g.gridDelta[2];
    const int gx = (int)floorf(ux), gy = (int)floorf(uy), gz = (int)floorf(uz);
    // squared distances (world units) from the particle to the slabs of the cells below / above along each axis
    const float csx = 1.0f / g.gridDelta[0], csy = 1.0f / g.gridDelta[1], csz = 1.0f / g.gridDelta[2];
    const float fx = ux - (float)gx, fy = uy - (float)gy, fz = uz - (float)gz;
    const float bx[3] = {fx * csx * fx * csx, 0.0f, (1.0f - fx) * csx * (1.0f - fx) * csx};
    const float by[3] = {fy * csy * fy * csy, 0.0f, (1.0f - fy) * csy * (1.0f - fy) * csy};
    const float bz[3] = {fz * csz * fz * csz, 0.0f, (1.0f - fz) * csz * (1.0f - fz) * csz};
    const float lim = R2 * 1.002f;
    uint32_t cs[27], cn[27];
#pragma unroll
    for (int k = 0; k < 27; ++k) {
        const int ox = k % 3, oy = (k / 3) % 3, oz = k / 9;
        const int cx = gx + ox - 1, cy = gy + oy - 1, cz = gz + oz - 1;
        const bool in = cx >= 0 && cx < (int)g.dims[0] && cy >= 0 && cy < (int)g.dims[1] && cz >= 0 &&
                        cz < (int)g.dims[2] && bx[ox] + by[oy] + bz[oz] <= lim;
        const uint32_t key = in ? cell_key(g, (uint32_t)cx, (uint32_t)cy, (uint32_t)cz) : 0u;
        cn[k] = in ? cellCount[key] : 0u;
        cs[k] = in ? (uint32_t)((int32_t)cellStart[key] + g.startCorr) : 0u;
    }
    uint32_t cnt = 0;
#pragma unroll
    for (int row = 0; row < 9; ++row) {
        const uint32_t sa = cs[3 * row], sb = cs[3 * row + 1], sc = cs[3 * row + 2];
        const uint32_t a = cn[3 * row], ab = a + cn[3 * row + 1], L = ab + cn[3 * row + 2];
        for (uint32_t q0 = 0; q0 < L; q0 += kSearchUnroll) {
            uint32_t t[kSearchUnroll];
            float4 xj[kSearchUnroll];
#pragma unroll
            for (uint32_t u = 0; u < kSearchUnroll; ++u) {
                const uint32_t q = min(q0 + u, L - 1u);
                t[u] = q < a ? sa + q : (q < ab ? sb + (q - a) : sc + (q - ab));
                xj[u] = pos[t[u]];
            }
#pragma unroll
            for (uint32_t u = 0; u < kSearchUnroll; ++u) {
                const float ddx = xj[u].x - xi.x, ddy = xj[u].y - xi.y, ddz = xj[u].z - xi.z;
                const float d2 = fmaf(ddz, ddz, fmaf(ddy, ddy, ddx * ddx));
                const bool acc = q0 + u < L && d2 < R2 && d2 > 0.0f && cnt < kMaxNeighbors;
                if (acc) out(cnt, t[u]);
                cnt += acc ? 1u : 0u;
            }
        }
    }
    return cnt;
}

// ---- the lists of few particles: a lane per row of cells -------------------------------------------------------------
// k_build_lists takes as long as its longest thread, 30 us of waiting on some 30 batches of candidates one after the
// other, however few particles there are. Where the chip is not full the nine rows of a particle (three cells each) are
// given to nine lanes of sixteen: a lane tests its row, the lanes' counts are summed up so that each knows where its
// neighbours begin in the list, and it stores them there. Same candidates, same tests, same order, same cap.
// us, a thread a particle -> a lane a row, on lattices of 2 and of 1.6 radii: 990 particles 33 -> 9 and 71 -> 24, 8,000
// 37 -> 9 and 81 -> 25, 32,768 37 -> 21 and 82 -> 51, 50,000 38 -> 31 and 84 -> 74, 65,536 39 -> 38 and 84 -> 90, 123,000
// 46 -> 65 and 97 -> 154: sixteen lanes a particle cost about 0.5 us per thousand, and the two meet at about 60,000. The
// line lies at half of that, 128 tiles, where a lane a row is far ahead on either lattice; up to 50,000 it would still be.
constexpr uint32_t kRowTiles = 128;
constexpr uint32_t kRowLanes = 16;                       // nine rows
constexpr uint32_t kRowParticles = kTile / kRowLanes;    // particles of a block
constexpr uint32_t kRowBlocks = kTile / kRowParticles;   // blocks of a tile
__global__ void __launch_bounds__(kTile) k_build_lists_rows(const float4* __restrict__ pos,
                                                            const SceneParams* __restrict__ P,
                                                            const SceneGrid* __restrict__ G,
                                                            const uint32_t* __restrict__ tileScene,
                                                            const uint32_t* __restrict__ cellStart,
                                                            const uint32_t* __restrict__ cellCount, uint32_t* nbrCount,
                                                            uint32_t* nbrList, uint2* blockStats) {
    const uint32_t s = tileScene[blockIdx.x / kRowBlocks];
    const SceneGrid& g = G[s];
    const uint32_t i = blockIdx.x * kRowParticles + threadIdx.x / kRowLanes, row = threadIdx.x % kRowLanes;
    const bool valid = i < P[s].base + P[s].count;
    const float R2 = P[s].R * P[s].R;
    const float4 xi = valid ? pos[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const int gx = (int)floorf((xi.x - g.gridMin[0]) * g.gridDelta[0]);
    const int gy = (int)floorf((xi.y - g.gridMin[1]) * g.gridDelta[1]) + (int)(row % 3u) - 1;
    const int gz = (int)floorf((xi.z - g.gridMin[2]) * g.gridDelta[2]) + (int)(row / 3u) - 1;
    uint32_t cs[3], cn[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int cx = gx + k - 1;
        const bool in = valid && row < 9u && cx >= 0 && cx < (int)g.dims[0] && gy >= 0 && gy < (int)g.dims[1] &&
                        gz >= 0 && gz < (int)g.dims[2];
        const uint32_t key = in ? cell_key(g, (uint32_t)cx, (uint32_t)gy, (uint32_t)gz) : 0u;
        cn[k] = in ? cellCount[key] : 0u;
        cs[k] = in ? (uint32_t)((int32_t)cellStart[key] + g.startCorr) : 0u;
    }
    const uint32_t a = cn[0], ab = a + cn[1], L = ab + cn[2];
    const auto slot = [&](uint32_t q) { return q < a ? cs[0] + q : (q < ab ? cs[1] + (q - a) : cs[2] + (q - ab)); };
    const auto accepted = [&](const float4& xj) {
        const float ddx = xj.x - xi.x, ddy = xj.y - xi.y, ddz = xj.z - xi.z;
        const float d2 = fmaf(ddz, ddz, fmaf(ddy, ddy, ddx * ddx));
        return d2 < R2 && d2 > 0.0f;
    };
    // the outcomes of the row's first 32 candidates are kept as bits, those of the rest only counted
    constexpr uint32_t kKept = 32;
    uint32_t kept = 0, found = 0;
    for (uint32_t q0 = 0; q0 < L; q0 += kSearchUnroll) {
        float4 xj[kSearchUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kSearchUnroll; ++u) xj[u] = pos[slot(min(q0 + u, L - 1u))];
#pragma unroll
        for (uint32_t u = 0; u < kSearchUnroll; ++u) {
            const uint32_t acc = q0 + u < L && accepted(xj[u]) ? 1u : 0u;
            found += acc;
            if (q0 + u < kKept) kept |= acc << (q0 + u);
        }
    }
    uint32_t incl = found;
#pragma unroll
    for (int o = 1; o < (int)kRowLanes; o <<= 1) {
        const uint32_t t = __shfl_up(incl, o, (int)kRowLanes);
        if ((int)row >= o) incl += t;
    }
    const uint32_t count = min((uint32_t)__shfl((int)incl, (int)kRowLanes - 1, (int)kRowLanes), kMaxNeighbors);
    uint32_t rank = incl - found;
    if (found) {
        uint32_t* out = nbrList + list_at(i, 0);
        const auto store = [&](uint32_t q) {
            if (rank < kMaxNeighbors) out[rank * kTile] = slot(q);
            ++rank;
        };
        for (; kept; kept &= kept - 1u) store((uint32_t)__ffs((int)kept) - 1u);
        for (uint32_t q = kKept; q < L; ++q)
            if (accepted(pos[slot(q)])) store(q);
    }
    if (valid && row == 0u) nbrCount[i] = count;
    note_neighbors(valid && row == 0u ? count : 0u, blockIdx.x, blockStats);
}

// One thread per particle, each entry stored as it is found; a tile's lists are one stretch of memory (list_at). An XCD
// takes a stretch of the Morton order, so that its L2 holds the cells that its tiles share: 652 -> 597 us on 2 million
// particles, 197 -> 178 on 500,000, 64 -> 60 on 123,000.
__global__ void __launch_bounds__(kTile) k_build_lists(const float4* __restrict__ pos, const SceneParams* __restrict__ P,
                                                       const SceneGrid* __restrict__ G,
                                                       const uint32_t* __restrict__ tileScene, uint32_t tiles,
                                                       uint32_t per, const uint32_t* __restrict__ cellStart,
                                                       const uint32_t* __restrict__ cellCount, uint32_t* nbrCount,
                                                       uint32_t* nbrList, uint2* tileStats) {
    const uint32_t tile = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (tile >= tiles) return;  // block-uniform
    const TileCtx c = tile_ctx(tile, tileScene, P);
    uint32_t cnt = 0;
    if (c.valid) {
        uint32_t* out = nbrList + list_at(c.i, 0);
        cnt = neighbor_list(c, P, G, pos, cellStart, cellCount, [&](uint32_t j, uint32_t t) { out[j * kTile] = t; });
        nbrCount[c.i] = cnt;
    }
    note_neighbors(cnt, tile, tileStats);
}

// ---- exclusive scan of uint32 (cell counts) --------------------------------------------------------------------
constexpr unsigned kScanThreads = 256, kScanItems = 8, kScanChunk = kScanThreads * kScanItems;
static_assert(kStaticScanWords >= (kStaticCells + kScanChunk - 1) / kScanChunk + 1,
              "static scratch must hold the chunk sums of kStaticCells cells");

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t& total) {
    __shared__ uint32_t wsum[kScanThreads / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    uint32_t incl = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t t = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += t;
    }
    if (lane == kWave - 1) wsum[w] = incl;
    __syncthreads();
    uint32_t before = 0, tot = 0;
    for (int j = 0; j < (int)(kScanThreads / kWave); ++j) {
        if (j < w) before += wsum[j];
        tot += wsum[j];
    }
    __syncthreads();
    total = tot;
    return before + incl - v;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_chunks(const uint32_t* __restrict__ in, uint32_t* out,
                                                              uint32_t* chunkSums, uint32_t n) {
    const uint32_t base = blockIdx.x * kScanChunk + threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t local = 0;
#pragma unroll
    for (unsigned k = 0; k < kScanItems; ++k) {
        v[k] = base + k < n ? in[base + k] : 0u;
        local += v[k];
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan(local, total);
#pragma unroll
    for (unsigned k = 0; k < kScanItems; ++k) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == 0) chunkSums[blockIdx.x] = total;
}

// single block: exclusive scan of the chunk sums in place (any count, sequential over blocks of kScanThreads)
__global__ void __launch_bounds__(kScanThreads) k_scan_sums(uint32_t* sums, uint32_t n) {
    uint32_t carry = 0;
    for (uint32_t b = 0; b < n; b += kScanThreads) {
        const uint32_t i = b + threadIdx.x;
        const uint32_t v = i < n ? sums[i] : 0u;
        uint32_t total;
        const uint32_t ex = block_exclusive_scan(v, total);
        if (i < n) sums[i] = carry + ex;
        carry += total;
    }
}

__global__ void __launch_bounds__(kScanThreads) k_scan_add(uint32_t* out, const uint32_t* __restrict__ chunkSums,
                                                           uint32_t n) {
    const uint32_t add = chunkSums[blockIdx.x];
    const uint32_t base = blockIdx.x * kScanChunk;
    for (unsigned k = threadIdx.x; k < kScanChunk; k += kScanThreads)
        if (base + k < n) out[base + k] += add;
}

uint32_t scan_scratch_words(uint32_t n) { return (n + kScanChunk - 1) / kScanChunk + 1; }

void exclusive_scan(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* scratch, hipStream_t st) {
    if (n == 0) return;
    const uint32_t chunks = (n + kScanChunk - 1) / kScanChunk;
    hipLaunchKernelGGL(k_scan_chunks, dim3(chunks), dim3(kScanThreads), 0, st, in, out, scratch, n);
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanThreads), 0, st, scratch, chunks);
    hipLaunchKernelGGL(k_scan_add, dim3(chunks), dim3(kScanThreads), 0, st, out, (const uint32_t*)scratch, n);
}

void launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t v, uint32_t n) {
    if (n) hipLaunchKernelGGL(k_fill_u32, dim3((n + 255) / 256), dim3(256), 0, st, p, v, n);
}

// ---- host launchers ---------------------------------------------------------------------------------------------
void launch_minmax(const Launch& L, const float4* pos, int* part, int* mm) {
    hipLaunchKernelGGL(k_minmax, dim3(L.tiles), dim3(kTile), 0, L.stream, pos, L.P, L.tileScene, part, L.stamps);
    hipLaunchKernelGGL(k_minmax_finish, dim3(L.sceneCount), dim3(kTile), 0, L.stream, L.P, (const int*)part, mm);
}

__global__ void __launch_bounds__(kTile) k_sort_begin(GridArgs args, SceneGrid* G, uint32_t scenes, uint32_t* cellCount,
                                                      uint32_t totalCells, uint32_t* haloStats, uint32_t* surface) {
    const uint32_t i = blockIdx.x * kTile + threadIdx.x;
    if (i < scenes) G[i] = args.g[i];
    if (i < 3u) haloStats[i] = 0u;
    if (i == 0u) surface[0] = 0u;
    for (uint32_t c = i; c < totalCells; c += gridDim.x * kTile) cellCount[c] = 0u;
}
void launch_sort_begin(const Launch& L, const GridArgs* args, SceneGrid* G, uint32_t* cellCount, uint32_t totalCells,
                       uint32_t* haloStats, uint32_t* surface) {
    hipLaunchKernelGGL(k_sort_begin, dim3(std::min((totalCells + kTile - 1) / kTile, 2048u)), dim3(kTile), 0, L.stream,
                       args ? *args : GridArgs{}, G, args ? L.sceneCount : 0u, cellCount, totalCells, haloStats, surface);
}

void launch_sort(const Launch& L, const SceneGrid* G, uint32_t totalCells, const float4* posIn, const float4* velIn,
                 const float4* dvIn, const float* dkIn, const uint32_t* idIn, float4* posOut, float4* velOut,
                 float4* dvOut, float* dkOut, uint32_t* idOut, uint32_t* cellOf, uint32_t* rank, uint32_t* tmpId,
                 uint32_t* cellCount, uint32_t* cellStart, uint32_t* scanScratch) {
    hipLaunchKernelGGL(k_insert, dim3(L.tiles), dim3(kTile), 0, L.stream, posIn, L.P, G, L.tileScene, cellOf, rank,
                       cellCount);
    exclusive_scan(cellCount, cellStart, totalCells, scanScratch, L.stream);
    hipLaunchKernelGGL(k_scatter_ids, dim3(L.tiles), dim3(kTile), 0, L.stream, L.P, G, L.tileScene,
                       (const uint32_t*)cellOf, (const uint32_t*)rank, (const uint32_t*)cellStart, idIn, tmpId);
    hipLaunchKernelGGL(k_reorder, dim3(L.tiles), dim3(kTile), 0, L.stream, L.P, G, L.tileScene,
                       (const uint32_t*)cellOf, (const uint32_t*)cellStart, (const uint32_t*)cellCount,
                       (const uint32_t*)tmpId, posIn, velIn, dvIn, dkIn, idIn, posOut, velOut, dvOut, dkOut, idOut);
}

// ---- halos of the neighbour groups ------------------------------------------------------------------------------
// One block per group of kTiles tiles. The distinct particle slots among the lists of its particles are collected in an
// LDS hash set of 32-slot buckets (bucket = slot >> 5, Fibonacci-hashed, linear probing) with a presence mask each;
// halo numbers are handed out bucket by bucket, ascending inside a bucket, so runs of consecutive particle slots stay
// consecutive in the halo. Every list entry is then rewritten as its halo number, packed with the pair's
// kernel-table code (gcode: the table index GetGradientW reads, or kGCodeZero beyond the cutoff) in the upper 16
// bits: positions do not change between here and the step's last neighbour loop, so the loops read the code instead
// of recomputing the distance, its square root and the index in every pass. A group with more than `limit` distinct
// neighbours (or more than kBucketLimit buckets) gets kHaloNone and is served by the global lists.
// haloStats = {groups staged, groups gathered, largest halo}.
constexpr uint32_t kBucketSlots = 2048;
constexpr uint32_t kBucketLimit = 896;  // + one bucket per thread in flight < kBucketSlots: probing always ends
constexpr uint32_t kHashEmpty = 0xFFFFFFFFu;
static_assert(kBucketLimit + 4 * kTile < kBucketSlots, "bucket table must never fill");

__device__ __forceinline__ uint32_t bucket_hash(uint32_t b) { return (b * 0x9E3779B1u) >> 21; }  // 11 bits
constexpr size_t kLdsHaloPos = (size_t)kHaloMax * 3 * sizeof(float);  // halo positions of k_build_halo

//
// Smaller groups (the resident solves') have fewer threads than a CU runs, and each entry is a chain of LDS reads: there
// kSplit threads share a particle's list, a batch of entries each in turn: 30.5 -> 15.4 us on 990 particles (groups of
// 256), 46.8 -> 34.9 us on 123,000 (groups of 512).
template <unsigned kTiles, unsigned kSplit = (kTiles < kGroupTiles ? kGroupTiles / kTiles : 1u)>
__global__ void __launch_bounds__(kTiles * kTile * kSplit) k_build_halo(const SceneParams* __restrict__ P,
                                                           const uint32_t* __restrict__ tileScene, uint32_t tiles,
                                                           const uint32_t* __restrict__ nbrCount,
                                                           const uint32_t* __restrict__ nbrList, uint32_t limit, uint32_t* haloCount, uint32_t* haloIds,
                                                           uint32_t* nbrLocal, uint32_t* haloStats,
                                                           const float4* __restrict__ pos, float R, float invStep) {
    constexpr uint32_t kOwn = kTiles * kTile, kThreads = kOwn * kSplit;
    constexpr uint32_t kFill = (halo_cap(kTiles) + kThreads - 1) / kThreads;
    __shared__ uint32_t bkey[kBucketSlots];
    __shared__ uint32_t bmask[kBucketSlots];
    __shared__ uint16_t bbase[kBucketSlots];
    __shared__ uint32_t waveTotal[kThreads / kWave];
    __shared__ uint32_t used, rows;
    extern __shared__ float hpos[];  // [kHaloMax * 3]: positions of the halo, by halo number
    const uint32_t g = blockIdx.x;
    const uint32_t i = g * kOwn + threadIdx.x % kOwn, tile = i / kTile;
    const uint32_t share = threadIdx.x / kOwn;  // which of the list's batches are this thread's
    uint32_t n = 0;
    if (tile < tiles) {
        const SceneParams& p = P[tileScene[tile]];
        if (i < p.base + p.count) n = nbrCount[i];
    }
    for (uint32_t k = threadIdx.x; k < kBucketSlots; k += blockDim.x) {
        bkey[k] = kHashEmpty;
        bmask[k] = 0u;
    }
    if (threadIdx.x == 0) {
        used = 0;
        rows = 0;
    }
    __syncthreads();
    if (n) atomicMax(&rows, n);
    __syncthreads();
    const uint32_t nr = rows;
    volatile uint32_t* vkey = bkey;
    volatile uint32_t* vmask = bmask;
    volatile uint32_t* vused = &used;
    // the list entries are loaded kHaloBatch at a time (their latencies overlap), then inserted in list order
    constexpr uint32_t kHaloBatch = 8;
    for (uint32_t j0 = share * kHaloBatch; j0 < nr; j0 += kSplit * kHaloBatch) {
        uint32_t tb[kHaloBatch];
#pragma unroll
        for (uint32_t u = 0; u < kHaloBatch; ++u) tb[u] = j0 + u < n ? nbrList[list_at(i, j0 + u)] : 0u;
#pragma unroll
        for (uint32_t u = 0; u < kHaloBatch; ++u) {
            if (j0 + u >= n || *vused > kBucketLimit) continue;
            const uint32_t t = tb[u];
            const uint32_t b = t >> 5, bit = 1u << (t & 31u);
            uint32_t h = bucket_hash(b);
            for (;;) {
                uint32_t cur = vkey[h];
                if (cur == kHashEmpty) {
                    cur = atomicCAS(&bkey[h], kHashEmpty, b);
                    if (cur == kHashEmpty) {
                        atomicAdd(&used, 1u);
                        cur = b;
                    }
                }
                if (cur == b) {
                    if (!(vmask[h] & bit)) atomicOr(&bmask[h], bit);
                    break;
                }
                h = (h + 1) & (kBucketSlots - 1);
            }
        }
    }
    __syncthreads();
    // halo numbers: thread t owns bucket slots [kPer * t, kPer * (t + 1))
    constexpr uint32_t kPer = kBucketSlots / kThreads;
    uint32_t own = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) own += __popc(bmask[kPer * threadIdx.x + k]);
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    uint32_t incl = own;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t v = __shfl_up(incl, o, kWave);
        if (lane >= o) incl += v;
    }
    if (lane == kWave - 1) waveTotal[w] = incl;
    __syncthreads();
    uint32_t m = 0;
    for (int k = 0; k < (int)(kThreads / kWave); ++k) m += waveTotal[k];
    if (used > kBucketLimit || m > limit) {  // block-uniform
        if (threadIdx.x == 0) {
            haloCount[g] = kHaloNone;
            atomicAdd(&haloStats[1], 1u);
        }
        return;
    }
    uint32_t base = incl - own;
    for (int k = 0; k < w; ++k) base += waveTotal[k];
    uint32_t* ids = haloIds + (size_t)g * kHaloMax;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t slot = kPer * threadIdx.x + k;
        uint32_t mask = bmask[slot];
        bbase[slot] = (uint16_t)base;
        const uint32_t b0 = bkey[slot] << 5;
        while (mask) {
            const uint32_t bit = (uint32_t)__ffs(mask) - 1u;
            ids[base++] = b0 + bit;
            mask &= mask - 1u;
        }
    }
    if (threadIdx.x == 0) {
        haloCount[g] = m;
        if (m) atomicAdd(&haloStats[0], 1u);
        atomicMax(&haloStats[2], m);
    }
    __syncthreads();
    // the halo's positions, by halo number (ids written above by the block, visible after the barrier)
    if (m) {  // up to kFill entries per thread: all id loads, then all gathers
        uint32_t t[kFill];
        float4 x[kFill];
#pragma unroll
        for (uint32_t u = 0; u < kFill; ++u) t[u] = ids[min(threadIdx.x + u * kThreads, m - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < kFill; ++u) x[u] = pos[t[u]];
#pragma unroll
        for (uint32_t u = 0; u < kFill; ++u) {
            const uint32_t k = threadIdx.x + u * kThreads;
            if (k < m) {
                hpos[3 * k] = x[u].x;
                hpos[3 * k + 1] = x[u].y;
                hpos[3 * k + 2] = x[u].z;
            }
        }
    }
    __syncthreads();
    // staged entries: the halo number of each neighbour | its table code << 16, in list order (the neighbour's
    // position from the halo's copy in LDS), rows in pairs (one 8-byte store per row pair; the entry
    // after a list's last one is 0 and never read)
    static_assert(kHaloBatch % 2 == 0 && kMaxNeighbors % 2 == 0, "staged rows are stored in pairs");
    const f3 xi = n ? ld3(pos[i]) : mk3(0.0f, 0.0f, 0.0f);
    for (uint32_t j0 = share * kHaloBatch; j0 < nr; j0 += kSplit * kHaloBatch) {
        uint32_t tb[kHaloBatch];
        // the list's last read in the step: non-temporal loads (it would only displace cached positions)
#pragma unroll
        for (uint32_t u = 0; u < kHaloBatch; ++u)
            tb[u] = j0 + u < n ? __builtin_nontemporal_load(nbrList + list_at(i, j0 + u)) : 0u;
        uint32_t en[kHaloBatch];
#pragma unroll
        for (uint32_t u = 0; u < kHaloBatch; ++u) {
            en[u] = 0u;
            if (j0 + u >= n) continue;
            const uint32_t t = tb[u];
            const uint32_t b = t >> 5, below = (1u << (t & 31u)) - 1u;
            uint32_t h = bucket_hash(b);
            while (bkey[h] != b) h = (h + 1) & (kBucketSlots - 1);
            const uint32_t s = bbase[h] + __popc(bmask[h] & below);
            const uint32_t code = gcode<false>(R, invStep, xi - mk3(hpos[3 * s], hpos[3 * s + 1], hpos[3 * s + 2]));
            en[u] = s | (code << 16);
        }
        uint2* out = reinterpret_cast<uint2*>(nbrLocal) + local_at(i, j0 >> 1);
#pragma unroll
        for (uint32_t u = 0; u < kHaloBatch; u += 2)
            if (j0 + u < n) out[(u >> 1) * kTile] = make_uint2(en[u], en[u + 1]);
    }
}

void launch_build_halo(const Launch& L, uint32_t groupTiles, const uint32_t* nbrCount, const uint32_t* nbrList,
                       uint32_t haloLimit, uint32_t* haloCount, uint32_t* haloIds, uint32_t* nbrLocal,
                       uint32_t* haloStats, const float4* pos, const KTabHost& kt) {
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(L.group_count(groupTiles)), dim3(std::max(groupTiles, kGroupTiles) * kTile),
                           kLdsHaloPos, L.stream, L.P, L.tileScene, L.tiles, nbrCount, nbrList,
                           std::min<uint32_t>(haloLimit, halo_cap(groupTiles)), haloCount, haloIds, nbrLocal,
                           haloStats, pos, kt.R, kt.invStep);
    };
    if (groupTiles == 1)
        run(k_build_halo<1>);
    else if (groupTiles == 2)
        run(k_build_halo<2>);
    else
        run(k_build_halo<4>);
}

uint32_t list_stats_per_tile(uint32_t tiles) { return tiles <= kRowTiles ? kRowBlocks : 1u; }
void launch_build_lists(const Launch& L, const SceneGrid* G, const float4* pos, const uint32_t* cellStart,
                        const uint32_t* cellCount, uint32_t* nbrCount, uint32_t* nbrList,
                        uint2* tileStats) {
    if (list_stats_per_tile(L.tiles) > 1u) {
        hipLaunchKernelGGL(k_build_lists_rows, dim3(L.tiles * kRowBlocks), dim3(kTile), 0, L.stream, pos, L.P, G,
                           L.tileScene, cellStart, cellCount, nbrCount, nbrList, tileStats);
        return;
    }
    hipLaunchKernelGGL(k_build_lists, dim3(L.gridAll), dim3(kTile), 0, L.stream, pos, L.P, G, L.tileScene, L.tiles,
                       L.tg.per, cellStart, cellCount, nbrCount, nbrList, tileStats);
}

int configure_search_kernels() {
    for (const void* fn : {(const void*)k_build_halo<1>, (const void*)k_build_halo<2>, (const void*)k_build_halo<4>})
        if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsHaloPos) != hipSuccess)
            return 1;
    return 0;
}

// ---- static scratch of the allocation-free step -------------------------------------------------------------------
// The grid cell arrays (counts, starts, scan partials) and the surface-tension curvature tables of vfd_step_no_alloc
// live here instead of in buffers the simulation allocates. Each device holds its own copy for the life of the
// process; every no-alloc step on a device shares it (overlapping calls on one device race). Its address is looked up
// once per device with that device current, and only that address is handed to kernels and copies: in host code
// `scratch` names a host-side stand-in, not device memory.
static __device__ __align__(256) uint32_t scratch[kStaticScratchWords];

namespace {
std::mutex g_scratchMu;
uint32_t* g_scratchPtr[kMaxStaticScratchDevices] = {};
}  // namespace

int static_scratch_address(int device, uint32_t** out) {
    *out = nullptr;
    if (device < 0 || device >= (int)kMaxStaticScratchDevices) return 1;
    std::lock_guard<std::mutex> lk(g_scratchMu);
    if (!g_scratchPtr[device]) {
        int cur = -1;
        if (hipGetDevice(&cur) != hipSuccess || cur != device) return 1;
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) {
            (void)hipGetLastError();
            return 1;
        }
        g_scratchPtr[device] = static_cast<uint32_t*>(p);
    }
    *out = g_scratchPtr[device];
    return 0;
}

}  // namespace vfd
