// solve.hip - resident solvers: a whole divergence, pressure or viscosity solve as one launch (no reference
// counterpart; the reference launches every iteration's kernels and synchronises after each,
// DFSPHImplementation.cu:443-808).
//
// For a simulation whose neighbour groups all fit the chip at once (one group of 256, 512 or 1024 particles per block,
// one block per CU: 262,144 particles on 256 CUs; resident.h has the rule) an iteration launched as separate kernels is bound by the launches:
// each pays about 4.5 us of start and end, 4-5 us to copy the kernel table into LDS and the latency of refilling the halo's
// positions, around 2-5 us of neighbour sums; iterations enqueued past convergence pay the launches too. Here a block
// keeps the table, its halo's positions and slots and its particles' own data for the whole solve, and the blocks
// meet at grid barriers: after every acceleration and every update, twice an iteration (Jacobi and CG alike). An
// iteration of the 8,000-particle dam break takes 9.2 us instead of 30 (21 with groups of 1024), and none runs past
// convergence; beyond 1024 particles per CU the launched kernels stay, bound by memory there (k_div_iter: 118 us at 2M
// particles).
//
// Memory. What blocks exchange (kappa, pressure accelerations, CG directions, tile partials) is written with
// write-through stores at agent scope, waited for before the barrier's arrival, and read with agent-scope loads that
// take no stale copy from an XCD's L2; everything else is read-only during the solve or private to its thread. A
// value is overwritten only after a barrier that follows its last read.
//
// Barriers (resident.h) are bounded. A block that waits longer than waitTicks - other work holds CUs that this launch
// needs - sets the abort bit in the arrival word, atomically with the arrivals and only while the barrier is open, so that
// either every block passes the solve's last barrier or none does; an aborted solve writes neither velocities nor
// positions, every later resident solve of the step returns at once, and the host takes the step again with launched
// iterations. Whether to return is decided by a block as a whole, so every wave leaves every launch.
//
// Results are the launched kernels' bits: the same sums in the same list order (terms.h), the same per-tile and
// per-scene FP64 trees, the same loop conditions.
#include <algorithm>
#include <type_traits>

#include "terms.h"

namespace vfd {

// ---- agent-scope exchange ---------------------------------------------------------------------------------------
__device__ __forceinline__ void put_agent(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float get_agent(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put_agent(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get_agent(const double* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// a float4 record as two 8-byte halves
__device__ __forceinline__ void put_agent(float4* p, f3 v) {
    unsigned long long* q = reinterpret_cast<unsigned long long*>(p);
    const unsigned long long a = ((unsigned long long)__float_as_uint(v.y) << 32) | __float_as_uint(v.x);
    const unsigned long long b = __float_as_uint(v.z);  // w = 0
    __hip_atomic_store(q, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 1, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ f3 get_agent(const float4* p) {
    const unsigned long long* q = reinterpret_cast<const unsigned long long*>(p);
    const unsigned long long a = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long b = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return mk3(__uint_as_float((uint32_t)a), __uint_as_float((uint32_t)(a >> 32)), __uint_as_float((uint32_t)b));
}

// ---- the blocks' meeting (resident.h) on the device -----------------------------------------------------------------
struct DeviceOps {
    static __device__ __forceinline__ uint32_t load(const uint32_t* p) {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ void store(uint32_t* p, uint32_t v) {
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ uint32_t add(uint32_t* p, uint32_t v) {
        return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + v;
    }
    static __device__ __forceinline__ bool swap(uint32_t* p, uint32_t& seen, uint32_t v) {
        return __hip_atomic_compare_exchange_strong(p, &seen, v, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
    }
    static __device__ __forceinline__ long long ticks() { return wall_clock64(); }
    static __device__ __forceinline__ bool leader() { return threadIdx.x == 0; }
    static __device__ __forceinline__ void settle() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
    static __device__ __forceinline__ void meet() { __syncthreads(); }
    template <class Fn> static __device__ __forceinline__ uint32_t one(Fn&& f) {
        __shared__ uint32_t v;
        if (threadIdx.x == 0) v = f();
        __syncthreads();
        return v;
    }
};

// ---- one block's group ----------------------------------------------------------------------------------------------
// Loaders of groups whose halo is not staged: exchanged values are gathered at agent scope. The staged list is read
// again in every iteration and stays in the caches (no non-temporal hint).
struct ResidentTraits {
    static constexpr int kListCache = 0;
    static constexpr bool kAlwaysSplit = true;
    template <int R> using Shape = ListShape<R>;
};
struct LoadXSr : ResidentTraits {  // {x_t, s_t}
    static constexpr int kLo = 4, kHi = 0;
    static constexpr bool kShortSqrt = LoadXS::kShortSqrt;
    const float4* __restrict__ pos;
    const float* s;
    __device__ __forceinline__ LoadXSr(const float4* p, const float* s_) : pos(p), s(s_) {}
    __device__ __forceinline__ void operator()(uint32_t t, float4& lo, float4& hi) const {
        const float4 x = pos[t];
        lo = make_float4(x.x, x.y, x.z, get_agent(s + t));
        hi = lo;
    }
};
struct LoadXVr : ResidentTraits {  // {x_t, -} {v_t, -}; kAgent: v is exchanged in this launch
    static constexpr int kLo = 3, kHi = 3;
    static constexpr bool kShortSqrt = LoadXV::kShortSqrt;
    const float4* __restrict__ pos;
    const float4* v;
    bool agent;
    __device__ __forceinline__ LoadXVr(const float4* p, const float4* v_, bool a) : pos(p), v(v_), agent(a) {}
    __device__ __forceinline__ void operator()(uint32_t t, float4& lo, float4& hi) const {
        lo = pos[t];
        hi = agent ? st4(get_agent(v + t)) : v[t];
    }
};
struct LoadXQr : ResidentTraits {  // {x_t, m / rho_t}
    static constexpr int kLo = 4, kHi = 0;
    static constexpr bool kShortSqrt = LoadXQ::kShortSqrt;
    const float4* __restrict__ pos;
    const float* __restrict__ rho;
    float m;
    __device__ __forceinline__ LoadXQr(const float4* p, const float* r, float m_) : pos(p), rho(r), m(m_) {}
    __device__ __forceinline__ void operator()(uint32_t t, float4& lo, float4& hi) const {
        const float4 x = pos[t];
        lo = make_float4(x.x, x.y, x.z, m / rho[t]);
        hi = lo;
    }
};
struct LoadXQVr : ResidentTraits {  // {x_t, m / rho_t} {u_t, -}, u_t = a_t + b_t (b null: a_t, exchanged)
    static constexpr int kLo = 4, kHi = 3;
    static constexpr bool kShortSqrt = LoadXQV::kShortSqrt;
    const float4* __restrict__ pos;
    const float* __restrict__ rho;
    const float4* a;
    const float4* b;
    float m;
    __device__ __forceinline__ LoadXQVr(const float4* p, const float* r, const float4* a_, const float4* b_, float m_)
        : pos(p), rho(r), a(a_), b(b_), m(m_) {}
    __device__ __forceinline__ void operator()(uint32_t t, float4& lo, float4& hi) const {
        const float4 x = pos[t];
        lo = make_float4(x.x, x.y, x.z, m / rho[t]);
        hi = st4(b ? ld3(a[t]) + ld3(b[t]) : get_agent(a + t));
    }
};

// v as a value of this point of the program: keeps what is formed from it - addresses, every pair's unpacked slot,
// scaled gradient or bound - from being formed once outside the iterations, in registers of its own
template <class T> __device__ __forceinline__ T here(T v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <unsigned kTiles> struct Group {
    static constexpr uint32_t kThreads = kTiles * kTile, kFill = halo_fill(kTiles);
    float* rec;         // halo records in LDS
    uint32_t m;         // halo size (0 when not staged: nothing to fill)
    uint32_t t[kFill];  // slots of this thread's halo entries threadIdx.x + u * kThreads, u < kFill
    uint32_t g, tile;
    TileCtx c;
    NbrSrc src;
    GridSync gs;
};
// The block's group (false: past the last tile, the block takes no part) and its halo's slots. Same group to block
// mapping as group_loop.
template <unsigned kTiles>
__device__ __forceinline__ bool resident_group(Group<kTiles>& r, const SceneParams* P, const uint32_t* tileScene,
                                               const Fields& F, uint32_t cap, const TileGrid& tg, uint32_t* words,
                                               uint32_t waitTicks, float* rec) {
    const uint32_t perG = tg.per / kTiles, chunk = blockIdx.x & 7u;
    r.g = chunk * perG + (blockIdx.x >> 3);
    if (r.g * kTiles >= tg.tiles) return false;
    const uint32_t blocks = (tg.tiles + kTiles - 1) / kTiles;
    r.gs = GridSync{words, blocks, chunk, min(perG, blocks - chunk * perG), (blocks + perG - 1) / perG, 0u,
                    waitTicks};
    r.tile = r.g * kTiles + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / kTile));  // (a scalar)
    r.c = tile_ctx4(r.tile, r.tile < tg.tiles, tileScene, P);
    const uint32_t m = F.haloCount[r.g];
    const bool staged = m <= kHaloMax;
    r.rec = rec;
    r.m = staged ? m : 0u;
    const uint32_t* ids = F.haloIds + (size_t)r.g * kHaloMax;
#pragma unroll
    for (uint32_t u = 0; u < r.kFill; ++u) r.t[u] = r.m ? ids[min(threadIdx.x + u * r.kThreads, r.m - 1u)] : 0u;
    r.src = NbrSrc{staged ? rec : nullptr, F.nbrLocal, F.nbrList, F.nbrCount, cap};
    return true;
}
// get(t) for every halo entry of this thread (loads together), then put(k, value)
struct PosVec {
    f3 x, v;
};
template <unsigned kTiles, class Get, class Put>
__device__ __forceinline__ void fill_halo(const Group<kTiles>& r, Get&& get, Put&& put) {
    constexpr uint32_t kFill = Group<kTiles>::kFill, kThreads = Group<kTiles>::kThreads;
    decltype(get(0u)) v[kFill];
#pragma unroll
    for (uint32_t u = 0; u < kFill; ++u)
        if (threadIdx.x + u * kThreads < r.m) v[u] = get(here(r.t[u]));
#pragma unroll
    for (uint32_t u = 0; u < kFill; ++u)
        if (threadIdx.x + u * kThreads < r.m) put(threadIdx.x + u * kThreads, v[u]);
}
// per-tile sums as tile_partials4, stored for other blocks; `first` = the first of the tile's slots written
template <unsigned kTiles, int NV>
__device__ __forceinline__ void exchange_partials(double (&v)[NV], double* partials, uint32_t tile, uint32_t first,
                                                  bool store) {
    __shared__ double sh[kTiles * kTile / kWave][NV];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
#pragma unroll
    for (int i = 0; i < NV; ++i) v[i] = wave_sum(v[i]);
    if (lane == 0)
#pragma unroll
        for (int i = 0; i < NV; ++i) sh[w][i] = v[i];
    __syncthreads();
    if ((threadIdx.x & (kTile - 1)) == 0 && store) {
        const int w0 = (threadIdx.x / kTile) * (kTile / kWave);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            double s = sh[w0][i];
            for (int j = 1; j < (int)(kTile / kWave); ++j) s += sh[w0 + j][i];
            put_agent(partials + (size_t)tile * kPartialSlots + first + i, s);
        }
    }
}

// Per-scene scalars of a solve, held by every block: each block adds up every active scene's tile partials itself (the
// tree of scene_sum over a 1024-thread block: waves of 64 tiles, then the waves in order) and evaluates the loop
// condition, so no block waits for another's decision.
struct SceneCtl {
    uint32_t active, it;
    float eta, thr, rhs2, absNew, alpha, beta, err;
    uint32_t pad;
};
// decide(s, ctl, sums) by one lane for every active scene; returns whether any scene is still active (block-uniform)
template <unsigned kTiles, int NV, class Decide>
__device__ __forceinline__ bool decide_scenes(const SceneParams* P, uint32_t sceneCount, SceneCtl* ctl,
                                              const double* partials, uint32_t first, Decide&& decide) {
    __shared__ double sh[kTiles * kTile / kWave][NV];
    __shared__ uint32_t live;
    const uint32_t lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    constexpr uint32_t kWaves = kTiles * kTile / kWave;
    auto chunk_sum = [&](uint32_t begin, uint32_t end, double (&v)[NV]) {  // tiles begin + lane, zero past the end
        const uint32_t t = begin + lane;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            v[i] = t < end ? 0.0 + get_agent(partials + (size_t)t * kPartialSlots + first + i) : 0.0;
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = wave_sum(v[i]);
    };
    if (threadIdx.x == 0) live = 0u;
    if (sceneCount == 1) {  // the block's waves take 64 tiles each: kTiles * 256 in all, as many as 256 blocks have
        if (ctl[0].active) {  // block-uniform
            double v[NV];
            chunk_sum(P[0].tileBegin + kWave * w, P[0].tileEnd, v);
            if (lane == 0)
#pragma unroll
                for (int i = 0; i < NV; ++i) sh[w][i] = v[i];
        }
        __syncthreads();
        if (threadIdx.x == 0 && ctl[0].active) {
            double s[NV];
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                s[i] = sh[0][i];
#pragma unroll
                for (uint32_t j = 1; j < kWaves; ++j) s[i] += sh[j][i];
            }
            decide(0u, ctl[0], s);
            if (ctl[0].active) live = 1u;
        }
    } else {
        __syncthreads();
        for (uint32_t s = w; s < sceneCount; s += kWaves) {
            if (!ctl[s].active) continue;  // wave-uniform
            const uint32_t b = P[s].tileBegin, e = P[s].tileEnd;
            double sum[NV], v[NV];
            chunk_sum(b, e, sum);
            for (uint32_t t = b + kWave; t < e; t += kWave) {  // (zero chunks past the scene would add nothing)
                chunk_sum(t, e, v);
#pragma unroll
                for (int i = 0; i < NV; ++i) sum[i] += v[i];
            }
            if (lane == 0) {
                decide(s, ctl[s], sum);
                if (ctl[s].active) live = 1u;
            }
        }
    }
    __syncthreads();
    return live != 0u;
}

// ---- the sums of the Jacobi solves ----------------------------------------------------------------------------------
// What a solve asks of its block's neighbour sums: the divergence of a field (begin), and per half iteration the halo's
// kappa or accelerations filled in (fill_*, then a block barrier) and the sum over the particle's own list.

// Lists and halo records in LDS, as the launched kernels have them; four waves per SIMD leave no registers for more.
static_assert(HaloRec<LoadXSr>::L == 4 && HaloRec<LoadXVr>::kSplit, "both record forms keep x in the first 12 bytes");
template <unsigned kTiles> struct ListSums {
    static constexpr size_t kLds = kLdsG + HaloRec<LoadXVr>::kBytes;
    const SceneParams& p;
    const Fields& F;
    const Group<kTiles>& r;
    float* sG;
    float* rec;
    KLds K;
    __device__ __forceinline__ ListSums(const SceneParams& p_, const Fields& F_, const Group<kTiles>& r_, float4* lds,
                                        const KTabHost& kh)
        : p(p_), F(F_), r(r_), sG(reinterpret_cast<float*>(lds)),
          rec(reinterpret_cast<float*>(lds + kLdsG / sizeof(float4))), K{sG, kh.R, kh.invStep} {
        load_table_g(sG, kh.tab);
    }
    __device__ __forceinline__ float* records() const { return rec; }
    // {x, v.x} {v.y, v.z}; afterwards the fourth word holds kappa or a.x
    __device__ __forceinline__ void begin() {
        fill_halo(r, [&](uint32_t t) { return PosVec{ld3(F.pos[t]), ld3(F.vel[t])}; },
                  [&](uint32_t k, const PosVec& q) { HaloRec<LoadXVr>::store(rec, k, st4(q.x), st4(q.v)); });
        __syncthreads();
    }
    __device__ __forceinline__ float velocity_divergence(f3 v) const {
        return field_divergence(p, K, F, r.src.cap, r.c.i, v, LoadXVr(F.pos, F.vel, false), r.src);
    }
    __device__ __forceinline__ void fill_scalar(const float* kap) const {
        fill_halo(r, [&](uint32_t t) { return get_agent(kap + t); },
                  [&](uint32_t k, float v) { rec[4 * k + 3] = v; });
    }
    __device__ __forceinline__ f3 accel(float k, const float* kap) const {
        return pressure_accel(p, K, F, r.src.cap, r.c.i, k, LoadXSr(F.pos, kap), r.src);
    }
    __device__ __forceinline__ void fill_accel() const {
        fill_halo(r, [&](uint32_t t) { return get_agent(F.ap + t); },
                  [&](uint32_t k, f3 v) {
                      rec[4 * k + 3] = v.x;
                      *reinterpret_cast<float2*>(rec + 4 * kHaloMax + 2 * k) = make_float2(v.y, v.z);
                  });
    }
    __device__ __forceinline__ float accel_divergence(f3 a) const {
        return field_divergence(p, K, F, r.src.cap, r.c.i, a, LoadXVr(F.pos, F.ap, true), r.src);
    }
};

// The pairs in registers: with one or two waves per SIMD a thread has room for gradW of its first kPairs neighbours and
// their halo slots, which do not change during a solve, so that a half iteration reads nothing but the exchanged value
// of each neighbour from LDS: no list, position or table reads. Those bound the loops of these block sizes, one list
// chunk's latency after another: an iteration of 8,000 particles took 17.3 us with ListSums and takes 9.2 us, half of it
// its two barriers. Neighbours past kPairs are looked up as they come (one-tile groups have room for every list); a
// group whose halo is not staged takes ListSums.
template <unsigned kTiles> struct PairSums {
    static constexpr uint32_t kPairs = kTiles == 1 ? 72 : 44;  // of 512 and 256 registers a thread
    static constexpr uint32_t kPairChunk = kTiles == 1 ? 8 : 4;
    static constexpr bool kRest = kPairs < kMaxNeighbors;
    static constexpr size_t kLds = (size_t)kHaloMax * 8 * sizeof(float);
    const SceneParams& p;
    const Fields& F;
    const Group<kTiles>& r;
    const float2* __restrict__ tab;
    float R, invStep;
    float4* sV;  // the vectors summed over
    float *sK, *sX;  // kappa; positions
    uint32_t n, rows;  // neighbours; the wave's longest list
    f3 q[kPairs];
    uint32_t slots[kPairs / 2];
    f3 contact[kMaxBodies];  // gradW of the boundary samples
    float vb[kMaxBodies];
    __device__ __forceinline__ PairSums(const SceneParams& p_, const Fields& F_, const Group<kTiles>& r_, float4* lds,
                                        const KTabHost& kh)
        : p(p_), F(F_), r(r_), tab(kh.tab), R(kh.R), invStep(kh.invStep), sV(lds),
          sK(reinterpret_cast<float*>(lds + kHaloMax)),
          sX(sK + kHaloMax), n(0), rows(0) {}
    __device__ __forceinline__ uint32_t slot(uint32_t j) const {
        return (here(slots[j / 2]) >> (16 * (j & 1u))) & 0xFFFFu;
    }
    // staged entries 2j, 2j + 1 (0 past the list's end, without a memory access; see each_neighbor_rec)
    __device__ __forceinline__ uint2 entries(uint32_t j) const {
        return TileLists(r.src.local, r.c.i).pair<0>(j, 2 * j < n);
    }
    __device__ __forceinline__ void begin() {
        fill_halo(r, [&](uint32_t t) { return PosVec{ld3(F.pos[t]), ld3(F.vel[t])}; },
                  [&](uint32_t k, const PosVec& h) {
                      sX[3 * k] = h.x.x;
                      sX[3 * k + 1] = h.x.y;
                      sX[3 * k + 2] = h.x.z;
                      sV[k] = st4(h.v);
                  });
        if (r.c.valid) n = F.nbrCount[r.c.i];
        rows = n;
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) rows = max(rows, (uint32_t)__shfl_xor((int)rows, o, kWave));
        rows = __builtin_amdgcn_readfirstlane(rows);
        __syncthreads();
        const f3 xi = r.c.valid ? ld3(F.pos[r.c.i]) : mk3(0.0f, 0.0f, 0.0f);
#pragma unroll
        for (uint32_t j = 0; j < kPairs; j += kPairChunk) {
            if (j < rows) {  // wave-uniform
                uint2 e[kPairChunk / 2];
                float g[kPairChunk];
#pragma unroll
                for (uint32_t u = 0; u < kPairChunk / 2; ++u) e[u] = entries(j / 2 + u);
#pragma unroll
                for (uint32_t u = 0; u < kPairChunk; ++u) g[u] = tab[(u & 1u ? e[u / 2].y : e[u / 2].x) >> 16].y;
#pragma unroll
                for (uint32_t u = 0; u < kPairChunk; ++u) {
                    const uint32_t s = (u & 1u ? e[u / 2].y : e[u / 2].x) & 0xFFFFu;
                    q[j + u] = g[u] * (xi - position(s));
                    if (u & 1u)
                        slots[(j + u) / 2] |= s << 16;
                    else
                        slots[(j + u) / 2] = s;
                }
            }
        }
        const KTab k{tab, R, 0.0f, invStep, 0.0f};
#pragma unroll
        for (uint32_t b = 0; b < kMaxBodies; ++b) {
            vb[b] = r.c.valid && b < p.bodyCount ? F.vb[(size_t)b * r.src.cap + r.c.i] : 0.0f;
            contact[b] = mk3(0.0f, 0.0f, 0.0f);
            if (vb[b] > 0.0f) contact[b] = gradW(k, xi - ld3(F.xb[(size_t)b * r.src.cap + r.c.i]));
        }
    }
    __device__ __forceinline__ f3 position(uint32_t s) const { return mk3(sX[3 * s], sX[3 * s + 1], sX[3 * s + 2]); }
    // f(slot, gradW) for the neighbours past kPairs, in list order
    template <class Fn> __device__ __forceinline__ void rest(Fn&& f) const {
        const f3 xi = ld3(F.pos[r.c.i]);
        for (uint32_t j = kPairs; j < n; ++j) {
            const uint2 e = entries(j / 2);
            const uint32_t w = j & 1u ? e.y : e.x, s = w & 0xFFFFu;
            f(s, tab[w >> 16].y * (xi - position(s)));
        }
    }
    // sum_j (u - u_j) . gradW_ij V + sum_b V_b u . gradW_ib (field_divergence), u_j in sV
    __device__ __forceinline__ float divergence(f3 ui) const {
        const uint32_t cnt = here(n);
        float d = 0.0f;
#pragma unroll
        for (uint32_t j = 0; j < kPairs; j += kPairChunk) {
            if (j < rows) {
                f3 uj[kPairChunk];
#pragma unroll
                for (uint32_t u = 0; u < kPairChunk; ++u) uj[u] = ld3(sV[slot(j + u)]);
#pragma unroll
                for (uint32_t u = 0; u < kPairChunk; ++u) {
                    const float s = d + dot3(ui - uj[u], q[j + u]);
                    d = j + u < cnt ? s : d;
                }
            }
        }
        if (kRest && n > kPairs) rest([&](uint32_t s, f3 g) { d += dot3(ui - ld3(sV[s]), g); });
        d *= p.V;
#pragma unroll
        for (uint32_t b = 0; b < kMaxBodies; ++b)
            if (vb[b] > 0.0f) d += vb[b] * dot3(ui, contact[b]);
        return d;
    }
    __device__ __forceinline__ float velocity_divergence(f3 v) const { return divergence(v); }
    __device__ __forceinline__ void fill_scalar(const float* kap) const {
        fill_halo(r, [&](uint32_t t) { return get_agent(kap + t); }, [&](uint32_t k, float v) { sK[k] = v; });
    }
    __device__ __forceinline__ f3 accel(float ki, const float*) const {  // pressure_accel
        const float negV = here(-p.V);
        const uint32_t cnt = here(n);
        f3 a = mk3(0.0f, 0.0f, 0.0f);
        auto term = [&](float kj, f3 g, bool in) {
            const float s = ki + kj;
            const f3 gj = negV * g, t = a + s * gj;
            const bool take = in && above_eps(fabsf(s));
            a = mk3(take ? t.x : a.x, take ? t.y : a.y, take ? t.z : a.z);
        };
#pragma unroll
        for (uint32_t j = 0; j < kPairs; j += kPairChunk) {
            if (j < rows) {
                float kj[kPairChunk];
#pragma unroll
                for (uint32_t u = 0; u < kPairChunk; ++u) kj[u] = sK[slot(j + u)];
#pragma unroll
                for (uint32_t u = 0; u < kPairChunk; ++u) term(kj[u], q[j + u], j + u < cnt);
            }
        }
        if (kRest && n > kPairs) rest([&](uint32_t s, f3 g) { term(sK[s], g, true); });
        if (above_eps(fabsf(ki))) {
#pragma unroll
            for (uint32_t b = 0; b < kMaxBodies; ++b)
                if (vb[b] > 0.0f) {
                    const f3 gj = (-vb[b]) * contact[b];
                    a = a + ki * gj;
                }
        }
        return a;
    }
    __device__ __forceinline__ void fill_accel() const {
        fill_halo(r, [&](uint32_t t) { return get_agent(F.ap + t); }, [&](uint32_t k, f3 v) { sV[k] = st4(v); });
    }
    __device__ __forceinline__ float accel_divergence(f3 a) const { return divergence(a); }
};

// ---- Jacobi solves ------------------------------------------------------------------------------------------------
// kPressure = false: k_div_init, the divergence iterations and k_div_final; true: k_pres_init, the pressure iterations
// and k_pres_final (dfsph.hip). A block of no particles returns; every other block passes the same barriers.
template <unsigned kTiles, bool kPressure, class Sums>
__device__ __forceinline__ void jacobi_solve(const SceneParams* __restrict__ P, const Fields& F, Group<kTiles>& r,
                                             Sums& sums, SceneCtl* ctl, uint32_t tiles, uint32_t sceneCount,
                                             int writeNext) {
    constexpr uint32_t kThreads = kTiles * kTile;
    const TileCtx c = r.c;
    const SceneParams& p = P[c.s];
    const SceneState st = F.state[c.s];  // time step (its solver fields are written below by the first group)
    float* kap = kPressure ? F.kappa : F.kappaV;
    const bool on = c.valid && (kPressure || p.enableDiv);

    // loop conditions before the first iteration (k_jacobi_begin)
    uint32_t any = 0;
    for (uint32_t s = threadIdx.x; s < sceneCount; s += kThreads) {
        const SceneParams& q = P[s];
        const float eta = kPressure ? q.presTol * 0.0001f * q.rho0 : F.state[s].dtInv * q.divTol * 0.0001f * q.rho0;
        const uint32_t minIt = kPressure ? q.minPres : q.minDiv, maxIt = kPressure ? q.maxPres : q.maxDiv;
        const bool go = (kPressure || q.enableDiv) && ((0.0f > eta || 0u < minIt) && 0u < maxIt);
        ctl[s].it = 0;
        ctl[s].eta = eta;
        ctl[s].active = go && q.count ? 1u : 0u;
        any |= ctl[s].active;
        if (r.g == 0) {
            JacobiState& J = kPressure ? F.state[s].pres : F.state[s].div;
            J.it = 0;
            J.err = 0.0f;
            J.eta = eta;
            J.active = go ? 1u : 0u;
        }
    }
    if (r.g == 0 && threadIdx.x == 0) {
        F.live[kPressure ? 1 : 0] = 0u;
        if (!kPressure) F.live[2] = 0u;
    }
    bool live = __syncthreads_or((int)any) != 0;
    sums.begin();

    float src = 0.0f, f = 0.0f, k = 0.0f, res = 0.0f;  // source term, scaled factor, kappa, residuum
    const uint32_t few = c.valid ? F.nbrCount[c.i] : 0u;
    if (on) {
        const float d = sums.velocity_divergence(ld3(F.vel[c.i]));
        if (kPressure) {
            src = F.density[c.i] / p.rho0 + st.dt * d;
            f = F.factor[c.i] * st.dt2Inv;
            k = -fminf(1.0f - src, 0.0f) * f;
        } else {
            src = few < 20u ? 0.0f : fmaxf(d, 0.0f);
            f = F.factor[c.i] * st.dtInv;
            k = src * f;
        }
        put_agent(kap + c.i, k);
    }
    uint32_t iterations = 0;
    f3 a = mk3(0.0f, 0.0f, 0.0f);
    for (;;) {
        if (!grid_sync<DeviceOps>(r.gs)) {
            grid_leave<DeviceOps>(r.gs, true);
            return;
        }
        if (iterations)
            live = decide_scenes<kTiles, 1>(P, sceneCount, ctl, F.partials, 0,
                                            [&](uint32_t s, SceneCtl& t, double (&sum)[1]) {
                const SceneParams& q = P[s];
                const uint32_t minIt = kPressure ? q.minPres : q.minDiv, maxIt = kPressure ? q.maxPres : q.maxDiv;
                const float err = (float)(-sum[0]) / (float)q.count;
                t.it += 1u;
                t.active = ((err > t.eta || t.it < minIt) && t.it < maxIt) ? 1u : 0u;
                if (r.g == 0) {
                    JacobiState& J = kPressure ? F.state[s].pres : F.state[s].div;
                    J.err = err;
                    J.it = t.it;
                    J.active = t.active;
                }
            });
        sums.fill_scalar(kap);
        __syncthreads();
        const bool act = live && ctl[c.s].active;
        if (on && (act || !live)) a = sums.accel(k, kap);
        if (!live) break;  // the accelerations of the final kappa
        if (on && act) put_agent(F.ap + c.i, a);
        if (!grid_sync<DeviceOps>(r.gs)) {
            grid_leave<DeviceOps>(r.gs, true);
            return;
        }
        sums.fill_accel();
        __syncthreads();
        double part = 0.0;
        if (on && act) {
            const float force = sums.accel_divergence(a) * (kPressure ? st.dt2 : st.dt);
            if (kPressure)
                res = fminf(1.0f - src - force, 0.0f);
            else
                res = few < 20u ? 0.0f : fminf(-src - force, 0.0f);
            k -= res * f;
            put_agent(kap + c.i, k);
            part = (double)(p.rho0 * res);
        }
        double v[1] = {part};
        exchange_partials<kTiles, 1>(v, F.partials, r.tile, 0, act && r.tile < tiles);
        ++iterations;
    }
    // the solve has passed its last barrier: results
    if (c.valid) {
        if (on) {
            F.densAdv[c.i] = src;
            if (ctl[c.s].it) F.residuum[c.i] = res;
            F.ap[c.i] = st4(a);
            const f3 v = ld3(F.vel[c.i]) + st.dt * a;
            F.vel[c.i] = st4(v);
            F.factor[c.i] = kPressure ? f : f * st.dt;
            if (kPressure) {
                const f3 x = ld3(F.pos[c.i]) + st.dt * v;
                if (writeNext) F.posNext[c.i] = st4(x);
                if (!(isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(x.x) && isfinite(x.y) &&
                      isfinite(x.z)))
                    F.state[c.s].nonfinite = 1u;  // per-step non-finite check, as k_pres_final
            }
        }
        if (!kPressure) F.acc[c.i] = make_float4(p.gx, p.gy, p.gz, 0.0f);
    }
    grid_leave<DeviceOps>(r.gs, false);
}
template <unsigned kTiles, bool kPressure>
__global__ void __launch_bounds__(kTiles * kTile, 1) k_jacobi_solve(const SceneParams* __restrict__ P,
                                                                    const uint32_t* __restrict__ tileScene, KTabHost kh,
                                                                    Fields F, uint32_t cap, TileGrid tg,
                                                                    uint32_t sceneCount, uint32_t* words,
                                                                    uint32_t waitTicks, int writeNext, long long* stamps) {
    if (!kPressure) note_time(stamps, kStampDivergence);
    extern __shared__ float4 lds[];
    __shared__ SceneCtl ctl[kResidentScenes];
    if (!solve_open<DeviceOps>(words)) return;
    Group<kTiles> r;
    if (!resident_group(r, P, tileScene, F, cap, tg, words, waitTicks, reinterpret_cast<float*>(lds))) return;
    if (kTiles < 4 && r.src.rec) {  // block-uniform
        PairSums<kTiles> sums(P[r.c.s], F, r, lds, kh);
        jacobi_solve<kTiles, kPressure>(P, F, r, sums, ctl, tg.tiles, sceneCount, writeNext);
    } else {
        ListSums<kTiles> sums(P[r.c.s], F, r, lds, kh);
        if (r.src.rec) r.src.rec = sums.records();
        jacobi_solve<kTiles, kPressure>(P, F, r, sums, ctl, tg.tiles, sceneCount, writeNext);
    }
}

// ---- viscosity solve ------------------------------------------------------------------------------------------------
// k_visc_precond, k_cg_begin, the CG iterations and k_visc_apply (dfsph.hip). The halo's second record half holds the
// search direction p of the halo's particles; what blocks exchange is z = M^-1 r: every block forms p = p beta + z of
// its halo itself, the operation the particle's own thread makes, so that an iteration needs two barriers (after the
// matrix product's partials and after the update's). With a group that is not staged the directions are exchanged too,
// behind a third.
using RecQV = HaloRec<LoadXQVr>;
static_assert(RecQV::L == 4 && HaloRec<LoadXQr>::L == 4, "both record forms keep {x, m / rho} in the first 16 bytes");
__device__ __forceinline__ float* direction(float* rec, uint32_t k) { return rec + 4 * kHaloMax + RecQV::H * k; }

template <unsigned kTiles>
__global__ void __launch_bounds__(kTiles * kTile, 1) k_visc_solve(const SceneParams* __restrict__ P,
                                                                         const uint32_t* __restrict__ tileScene,
                                                                         KTabHost kh, Fields F, uint32_t cap,
                                                                         TileGrid tg, uint32_t sceneCount,
                                                                         uint32_t* words, uint32_t waitTicks,
                                                                         const uint32_t* __restrict__ haloStats,
                                                                         long long* stamps) {
    note_time(stamps, kStampViscosity);
    __shared__ SceneCtl ctl[kResidentScenes];
    if (!solve_open<DeviceOps>(words)) return;
    VFD_HALO_KERNEL_PROLOGUE(kh)
    constexpr uint32_t kThreads = kTiles * kTile;
    Group<kTiles> r;
    if (!resident_group(r, P, tileScene, F, cap, tg, words, waitTicks, rec)) return;
    const TileCtx c = r.c;
    const SceneParams& p = P[c.s];
    const float dt = F.state[c.s].dt;
    const bool on = c.valid && p.enableVisc;
    const bool gathered = haloStats[1] != 0u;  // some group is not staged (the same in every block)
    const float m = P[0].m;                    // one particle radius per batch

    for (uint32_t s = threadIdx.x; s < sceneCount; s += kThreads) {
        ctl[s].it = 0;
        ctl[s].active = P[s].enableVisc && P[s].count ? 1u : 0u;  // takes part in the set-up
    }
    fill_halo(r,
              [&](uint32_t t) {
                  const float4 x = F.pos[t];
                  return PosVec{mk3(x.x, x.y, x.z), mk3(m / F.density[t], 0.0f, 0.0f)};
              },
              [&](uint32_t k, const PosVec& q) {
                  *reinterpret_cast<float4*>(rec + 4 * k) = make_float4(q.x.x, q.x.y, q.x.z, q.v.x);
              });
    fill_halo(r, [&](uint32_t t) { return ld3(F.vel[t]) + ld3(F.dv[t]); },
              [&](uint32_t k, f3 v) { RecQV::put(direction(rec, k), RecQV::H, st4(v)); });
    __syncthreads();
    f3 dir = mk3(0.0f, 0.0f, 0.0f), z = dir;  // p and z of this thread's particle
    double v3[3] = {0.0, 0.0, 0.0};
    if (on) {
        const M3 inv = visc_precond(p, K, F, cap, c.i, dt, LoadXQr(F.pos, F.density, m), r.src);
#pragma unroll
        for (int e = 0; e < 9; ++e) F.minv[(size_t)e * cap + c.i] = inv.m[e];
        const f3 b = ld3(F.vel[c.i]), x0 = b + ld3(F.dv[c.i]);
        F.cgX[c.i] = st4(x0);
        const f3 ax = visc_matvec(p, K, F, cap, c.i, x0, dt, LoadXQVr(F.pos, F.density, F.vel, F.dv, m), r.src);
        const f3 res = b - ax;
        z = minv_mul(F.minv, cap, c.i, res);
        F.cgR[c.i] = st4(res);
        put_agent(F.cgZ + c.i, z);
        dir = z;
        v3[0] = (double)dot3(b, b);
        v3[1] = (double)dot3(res, res);
        v3[2] = (double)dot3(res, z);
    }
    exchange_partials<kTiles, 3>(v3, F.partials, r.tile, 0, r.tile < tg.tiles && p.enableVisc);
    if (!grid_sync<DeviceOps>(r.gs)) {
        grid_leave<DeviceOps>(r.gs, true);
        return;
    }
    // k_cg_begin_finish
    bool live = decide_scenes<kTiles, 3>(P, sceneCount, ctl, F.partials, 0,
                                         [&](uint32_t s, SceneCtl& t, double (&sum)[3]) {
        const SceneParams& q = P[s];
        CgState G = F.state[s].cg;
        G.it = 0;
        G.zero = 0;
        G.active = 0;
        G.loops = 0;
        G.rhs2 = (float)sum[0];
        if (G.rhs2 == 0.0f) {
            G.zero = 1;
            G.err = 0.0f;
        } else {
            G.thr = fmaxf(q.viscTol * q.viscTol * 0.0001f * G.rhs2, FLT_MIN);
            G.res2 = (float)sum[1];
            G.err = sqrtf(G.res2 / G.rhs2);
            if (!(G.res2 < G.thr)) {
                G.absNew = fabsf((float)sum[2]);
                G.active = (0u >= q.minVisc && 0u < q.maxVisc) ? 1u : 0u;
            }
        }
        t.active = G.active;
        t.thr = G.thr;
        t.rhs2 = G.rhs2;
        t.absNew = G.absNew;
        t.pad = G.zero;
        if (r.g == 0) F.state[s].cg = G;
    });
    bool firstIteration = true;
    while (live) {
        const bool act = on && ctl[c.s].active;
        // directions: p = z at first, p beta + z afterwards (k_cg_direction); a halo entry's scene through its tile
        fill_halo(r,
                  [&](uint32_t t) {
                      return PosVec{get_agent(F.cgZ + t),
                                    mk3(__uint_as_float(sceneCount == 1 ? 0u : tileScene[t / kTile]), 0.0f, 0.0f)};
                  },
                  [&](uint32_t k, const PosVec& q) {
                      const SceneCtl& t = ctl[__float_as_uint(q.v.x)];
                      if (!t.active) return;
                      float* h = direction(rec, k);
                      const f3 d = firstIteration ? q.x : ld3(RecQV::get(h, RecQV::H)) * t.beta + q.x;
                      RecQV::put(h, RecQV::H, st4(d));
                  });
        if (act && !firstIteration) dir = dir * ctl[c.s].beta + z;
        if (gathered) {
            if (act) put_agent(F.cgP + c.i, dir);
            if (!grid_sync<DeviceOps>(r.gs)) {
                grid_leave<DeviceOps>(r.gs, true);
                return;
            }
        } else {
            __syncthreads();
        }
        firstIteration = false;
        f3 ap = mk3(0.0f, 0.0f, 0.0f);
        double v1[1] = {0.0};
        if (act) {
            ap = visc_matvec(p, K, F, cap, c.i, dir, dt, LoadXQVr(F.pos, F.density, F.cgP, nullptr, m), r.src);
            v1[0] = (double)dot3(dir, ap);
        }
        exchange_partials<kTiles, 1>(v1, F.partials, r.tile, 3, act || (r.tile < tg.tiles && ctl[c.s].active));
        if (!grid_sync<DeviceOps>(r.gs)) {
            grid_leave<DeviceOps>(r.gs, true);
            return;
        }
        // k_cg_alpha
        (void)decide_scenes<kTiles, 1>(P, sceneCount, ctl, F.partials, 3, [&](uint32_t, SceneCtl& t, double (&sum)[1]) {
            t.alpha = t.absNew / (float)sum[0];
        });
        double v2[2] = {0.0, 0.0};
        if (act) {
            const float alpha = ctl[c.s].alpha;
            F.cgX[c.i] = st4(ld3(F.cgX[c.i]) + dir * alpha);
            const f3 res = ld3(F.cgR[c.i]) - ap * alpha;
            F.cgR[c.i] = st4(res);
            z = minv_mul(F.minv, cap, c.i, res);
            put_agent(F.cgZ + c.i, z);
            v2[0] = (double)dot3(res, res);
            v2[1] = (double)dot3(res, z);
        }
        exchange_partials<kTiles, 2>(v2, F.partials, r.tile, 0, r.tile < tg.tiles && ctl[c.s].active);
        if (!grid_sync<DeviceOps>(r.gs)) {
            grid_leave<DeviceOps>(r.gs, true);
            return;
        }
        // k_cg_update_finish
        live = decide_scenes<kTiles, 2>(P, sceneCount, ctl, F.partials, 0,
                                        [&](uint32_t s, SceneCtl& t, double (&sum)[2]) {
            const SceneParams& q = P[s];
            const float res2 = (float)sum[0], err = sqrtf(res2 / t.rhs2);
            uint32_t goes = 0;
            if (!(res2 < t.thr)) {
                const float absOld = t.absNew;
                t.absNew = fabsf((float)sum[1]);
                t.beta = t.absNew / absOld;
                t.it += 1u;
                goes = (t.it >= q.minVisc && t.it < q.maxVisc) ? 1u : 0u;
            }
            t.active = goes;
            if (r.g == 0) {
                CgState& G = F.state[s].cg;
                G.loops += 1u;
                G.res2 = res2;
                G.err = err;
                G.it = t.it;
                G.absNew = t.absNew;
                G.alpha = t.alpha;
                G.beta = t.beta;
                G.active = goes;
            }
        });
    }
    // k_visc_apply
    if (on) {
        f3 x = ld3(F.cgX[c.i]);
        if (ctl[c.s].pad) {  // a zero right-hand side
            x = mk3(0.0f, 0.0f, 0.0f);
            F.cgX[c.i] = st4(x);
        }
        const f3 d = x - ld3(F.vel[c.i]);
        F.acc[c.i] = st4(ld3(F.acc[c.i]) + (1.0f / dt) * d);
        F.dv[c.i] = st4(d);
    }
    grid_leave<DeviceOps>(r.gs, false);
}

// ---- host side ----------------------------------------------------------------------------------------------------
constexpr size_t kLdsJacobi = ListSums<4>::kLds;
constexpr size_t kLdsVisc = kLdsG + RecQV::kBytes;
constexpr size_t kLdsStatic = kResidentScenes * sizeof(SceneCtl) + 2048;  // control and reduction arrays, at most
static_assert(kLdsVisc + kLdsStatic <= 160 * 1024 && PairSums<1>::kLds <= kLdsJacobi, "a resident group must fit a CU's LDS");

template <class Run> static void with_tiles(uint32_t groupTiles, Run&& run) {
    if (groupTiles == 1)
        run(std::integral_constant<unsigned, 1>());
    else if (groupTiles == 2)
        run(std::integral_constant<unsigned, 2>());
    else
        run(std::integral_constant<unsigned, 4>());
}
void launch_div_solve(const Launch& L, uint32_t groupTiles, const KTabHost& kt, const Fields& F, const Resident& r) {
    with_tiles(groupTiles, [&](auto t) {
        hipLaunchKernelGGL((k_jacobi_solve<t(), false>), dim3(L.group_count(t())), dim3(t() * kTile), kLdsJacobi,
                           L.stream, L.P, L.tileScene, kt, F, L.capacity, TileGrid(L.tg), L.sceneCount, r.words,
                           r.waitTicks, 0, L.stamps);
    });
}
void launch_pres_solve(const Launch& L, uint32_t groupTiles, const KTabHost& kt, const Fields& F, const Resident& r,
                       int writeNext) {
    with_tiles(groupTiles, [&](auto t) {
        hipLaunchKernelGGL((k_jacobi_solve<t(), true>), dim3(L.group_count(t())), dim3(t() * kTile), kLdsJacobi,
                           L.stream, L.P, L.tileScene, kt, F, L.capacity, TileGrid(L.tg), L.sceneCount, r.words,
                           r.waitTicks, writeNext, L.stamps);
    });
}
void launch_visc_solve(const Launch& L, uint32_t groupTiles, const KTabHost& kt, const Fields& F, const Resident& r,
                       const uint32_t* haloStats) {
    with_tiles(groupTiles, [&](auto t) {
        hipLaunchKernelGGL((k_visc_solve<t()>), dim3(L.group_count(t())), dim3(t() * kTile), kLdsVisc, L.stream, L.P,
                           L.tileScene, kt, F, L.capacity, TileGrid(L.tg), L.sceneCount, r.words, r.waitTicks,
                           haloStats, L.stamps);
    });
}
int configure_solve_kernels() {
    int bad = 0;
    const auto set = [&](auto kernel, size_t bytes) {
        if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) !=
            hipSuccess)
            bad = 1;
    };
    for (uint32_t g : {1u, 2u, 4u})
        with_tiles(g, [&](auto t) {
            set(k_jacobi_solve<t(), false>, kLdsJacobi);
            set(k_jacobi_solve<t(), true>, kLdsJacobi);
            set(k_visc_solve<t()>, kLdsVisc);
        });
    return bad;
}

}  // namespace vfd
