// resident.h - how the blocks of a resident solve (solve.hip) enter it, meet and leave it: the bounded grid barrier,
// written over the few operations that a block needs (Ops below), so that the same code runs on the device and, with
// threads for waves, in a program on the host.
//
// Ops:  load(p), store(p, v), add(p, v) (the new value), swap(p, seen, v) (compare-and-exchange, seen = what was there):
//       relaxed atomics that every block sees; ticks(): a clock, the same for all blocks; one(f): called by every thread
//       of the block, f() by one of them, its value to all; leader(): true in one thread of the block; settle(): waits
//       for the calling thread's own stores; meet(): the block's barrier.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define VFD_RESIDENT __device__ __forceinline__
#else
#define VFD_RESIDENT inline
#endif

namespace vfd {

// Barrier words (32-bit), zero between launches; words[kResidentAbortedAt] is set when a solve was aborted, and then
// the host clears all of them.
constexpr uint32_t kResidentWords = 1024, kResidentAbortedAt = 18 * 32;
// A 128-byte line each: arrivals (2 per block or chunk, bit 0 = aborted), arrivals per XCD chunk, release words, blocks
// that have left.
constexpr uint32_t kLine = 32;
constexpr uint32_t kWordArrive = 0, kWordChunk = kLine, kWordRelease = 9 * kLine, kWordLeft = 17 * kLine;
static_assert(kWordLeft + kLine <= kResidentAbortedAt && kResidentAbortedAt < kResidentWords, "barrier words");
constexpr uint32_t kAbortBit = 1u, kReleaseAbort = 0xFFFFFFFFu;
// Up to this many blocks poll the arrival word itself (1.5 us at 8 blocks, 2.1 at 64); more arrive through their XCD
// chunk's word and poll a release word per chunk (2.5 us at 121 blocks, 2.9 at 248, where one polled word takes 5.8).
constexpr uint32_t kFlatBlocks = 64;

constexpr uint32_t kResidentScenes = 64;  // most scenes of a resident solve (their scalars live in LDS)
// Tiles per group of a simulation's resident solves, the fewest of 1, 2 and 4 with which every group has a CU to itself;
// 0: no resident solves (more groups than CUs, or too many scenes). Solves, halo build and density of a step take the
// same value.
//
// The fewest tiles per group win: a group's neighbour sums are bound by its CU's LDS and VALU (1024 particles 7-8 us a
// sum, 256 particles about 2), and more blocks cost a barrier at most 1.4 us.
//
// Scenes: every block decides for every scene, its waves (4 a tile) taking the scenes in turn, one after the other about
// 1.5 us each. Where a wave has more than 12 that is more than the launches saved. ms a step, launched -> resident, with up
// to 100 CG iterations and with 2: 48 scenes of 200 particles (12 a wave) 7.54 -> 7.42 and 4.09 -> 3.80, 56 scenes 8.10 ->
// 8.42 and 4.80 -> 4.46, 128 scenes 13.8 -> 17.3 and 10.3 -> 10.2, 256 scenes 23.1 -> 32.5; larger groups, whose blocks
// wait for the few scenes that go on: 64 scenes of 1,900 (8 a wave) 9.41 -> 8.83 and 4.61 -> 3.83, 96 of them (6 a wave)
// 12.3 -> 13.0 and 6.32 -> 5.84.
inline uint32_t resident_tiles(uint32_t tiles, uint32_t scenes, uint32_t numCU) {
    if (tiles == 0 || scenes > kResidentScenes) return 0;
    const uint32_t most = numCU < 256u ? numCU : 256u;
    for (uint32_t t = 1; t <= 4; t *= 2)
        if ((tiles + t - 1) / t <= most) return scenes <= 12u * 4u * t ? t : 0u;
    return 0;
}

// Tiles per group of a recorded step, whose Jacobi solves are launched, over groups of groupTiles, with the viscosity solve
// resident over the same groups if those fit the CUs; 0: they do not. fitting: resident_tiles.
inline uint32_t recorded_tiles(uint32_t fitting, uint32_t groupTiles) {
    return fitting && fitting <= groupTiles ? groupTiles : 0;
}

// Longest wait at a barrier, in ticks of the 100 MHz wall clock: 3 ms. A barrier takes 2-3 us and a whole solve 0.03 to 2
// ms, so what is waited for longer is a block that other work keeps from its CU - another simulation's resident solve
// among it, dispatched in the same microseconds, each holding CUs that the other waits for.
constexpr uint32_t kResidentWait = 300000;
// Steps taken with launched iterations after an aborted solve: twice as many after each abort, until a step's resident
// solves have passed. What an abort costs (the limit, and the step begun) stays a few percent of the steps between.
struct ResidentPause {
    static constexpr uint32_t kFirst = 64, kMost = 4096;
    uint32_t left = 0, next = kFirst;
    bool over() const { return left == 0; }
    void aborted() {
        left = next;
        next = next < kMost ? 2 * next : kMost;
    }
    void stepped(bool resident) {  // a step has been completed, with resident solves or without
        if (resident)
            next = kFirst;
        else if (left)
            --left;
    }
};

struct GridSync {
    uint32_t* w;
    uint32_t blocks, chunk, chunkBlocks, chunks, epoch;
    uint32_t waitTicks;  // of the 100 MHz wall clock
};

// Whether no solve of this step has been aborted, the same answer in every thread of the block: the mark is read once,
// since blocks of this very launch may set it (a block that starts after the others' limit), and a block of which only
// some waves went on would pass barriers that nobody has completed.
template <class Ops> VFD_RESIDENT bool solve_open(const uint32_t* words) {
    return Ops::one([&] { return Ops::load(words + kResidentAbortedAt); }) == 0u;
}
template <class Ops> VFD_RESIDENT void release_chunks(const GridSync& g, uint32_t v) {
    for (uint32_t c = 0; c < g.chunks; ++c) Ops::store(g.w + kWordRelease + kLine * c, v);
}
// Arrivals are counted on through a solve and may pass 2^32 (64 blocks: after 16 million Jacobi iterations), as may the
// target; they are never farther apart than a barrier's arrivals.
VFD_RESIDENT bool short_of(uint32_t arrivals, uint32_t target) { return (int32_t)(arrivals - target) < 0; }
// the wait of one thread; target = arrivals (times 2) that complete the barrier
template <class Ops> VFD_RESIDENT bool sync_thread(const GridSync& g) {
    const long long t0 = Ops::ticks();
    uint32_t* arrive = g.w + kWordArrive;
    if (g.blocks <= kFlatBlocks) {
        const uint32_t target = 2u * g.blocks * g.epoch;
        uint32_t v = Ops::add(arrive, 2u);
        while (!(v & kAbortBit) && short_of(v, target)) {
            if ((uint64_t)(Ops::ticks() - t0) > g.waitTicks) {  // only a barrier that is still open can be aborted
                uint32_t seen = v;
                if (Ops::swap(arrive, seen, v | kAbortBit)) return false;
                v = seen;
            } else {
                v = Ops::load(arrive);
            }
        }
        return !(v & kAbortBit);
    }
    const uint32_t target = 2u * g.chunks * g.epoch;
    uint32_t* mine = g.w + kWordRelease + kLine * g.chunk;
    if (Ops::add(g.w + kWordChunk + kLine * g.chunk, 1u) == g.chunkBlocks * g.epoch) {
        const uint32_t v = Ops::add(arrive, 2u);
        if (v & kAbortBit) {
            release_chunks<Ops>(g, kReleaseAbort);
            return false;
        }
        if (v == target) {
            release_chunks<Ops>(g, g.epoch);
            return true;
        }
    }
    for (;;) {
        const uint32_t r = Ops::load(mine);
        if (r == kReleaseAbort) return false;
        if (r >= g.epoch) return true;
        if ((uint64_t)(Ops::ticks() - t0) > g.waitTicks) {
            uint32_t v = Ops::load(arrive);
            if (v & kAbortBit) return false;
            if (!short_of(v, target)) continue;  // complete: its release is being written
            if (Ops::swap(arrive, v, v | kAbortBit)) {
                release_chunks<Ops>(g, kReleaseAbort);
                return false;
            }
        }
    }
}
// Barrier over the launch's blocks, called by every thread; false: the solve is aborted (the same answer in every
// block). Every wave waits for its own stores before its block arrives.
template <class Ops> VFD_RESIDENT bool grid_sync(GridSync& g) {
    Ops::settle();
    Ops::meet();
    g.epoch += 1;
    return Ops::one([&] { return sync_thread<Ops>(g) ? 1u : 0u; }) != 0u;
}
// The last block to leave clears the words for the next launch; an aborted solve leaves its mark. A block has waited for
// its stores to the words before it counts as having left: the one to its own chunk's release word is seen by no other
// block where it is alone in the chunk (73 blocks, for instance), and must not land after the clearing.
template <class Ops> VFD_RESIDENT void grid_leave(const GridSync& g, bool aborted) {
    if (!Ops::leader()) return;
    if (aborted) Ops::store(g.w + kResidentAbortedAt, 1u);
    Ops::settle();
    if (Ops::add(g.w + kWordLeft, 1u) != g.blocks) return;
    Ops::store(g.w + kWordArrive, 0u);
    for (uint32_t c = 0; c < 8; ++c) {
        Ops::store(g.w + kWordChunk + kLine * c, 0u);
        Ops::store(g.w + kWordRelease + kLine * c, 0u);
    }
    Ops::store(g.w + kWordLeft, 0u);
}

}  // namespace vfd
