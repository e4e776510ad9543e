// The blocks of a resident solve (vfd_amd/csrc/resident.h) as threads of a host program: a thread per wave, the barrier
// words in one lock-protected array. argv[1] names a scenario; the program prints "ok" or what was wrong.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "resident.h"

using namespace vfd;

static std::mutex mu;
static uint32_t words[kResidentWords];
static std::atomic<long long> now{0};

[[noreturn]] static void wrong(const char* what) {
    std::printf("wrong: %s\n", what);
    std::fflush(stdout);
    std::_Exit(1);
}

// A block: the waves still in the launch, their barrier, and the value its leader hands to all (at first what the
// memory happens to hold).
struct Block {
    std::mutex m;
    std::condition_variable cv;
    uint32_t waves = 0, waiting = 0, generation = 0, shared = 0xDEADBEEFu;
    void meet() {
        std::unique_lock<std::mutex> lk(m);
        const uint32_t g = generation;
        if (++waiting == waves) {
            next();
            return;
        }
        if (!cv.wait_for(lk, std::chrono::seconds(30), [&] { return generation != g; })) wrong("a wave never left");
    }
    void next() {
        waiting = 0;
        ++generation;
        cv.notify_all();
    }
    void wave_ends() {  // as on the device, a wave that has ended is not waited for
        std::lock_guard<std::mutex> lk(m);
        --waves;
        if (waves && waiting == waves) next();
    }
};

struct Wave {
    Block* block = nullptr;
    uint32_t wave = 0;
    std::function<void()> afterMark;             // called between a read of the abort mark and its use
    std::function<void()> beforeLeave;           // called before the block leaves
    uint32_t* slow = nullptr;                    // a word to which this wave's stores take their time, as long as it
    std::vector<uint32_t> underway;              // does not wait for them
    void land();
};
static thread_local Wave self;

void Wave::land() {
    std::lock_guard<std::mutex> lk(mu);
    if (!underway.empty()) *slow = underway.back();
    underway.clear();
}

struct Ops {
    static uint32_t load(const uint32_t* p) {
        uint32_t v;
        {
            std::lock_guard<std::mutex> lk(mu);
            v = *p;
        }
        if (p == words + kResidentAbortedAt && self.afterMark) self.afterMark();
        std::this_thread::yield();
        return v;
    }
    static void store(uint32_t* p, uint32_t v) {
        if (p == self.slow) {
            self.underway.push_back(v);
            return;
        }
        std::lock_guard<std::mutex> lk(mu);
        *p = v;
    }
    static uint32_t add(uint32_t* p, uint32_t v) {
        std::lock_guard<std::mutex> lk(mu);
        return *p += v;
    }
    static bool swap(uint32_t* p, uint32_t& seen, uint32_t v) {
        std::lock_guard<std::mutex> lk(mu);
        if (*p != seen) {
            seen = *p;
            return false;
        }
        *p = v;
        return true;
    }
    static long long ticks() { return ++now; }
    static bool leader() { return self.wave == 0; }
    static void settle() { self.land(); }
    static void meet() { self.block->meet(); }
    template <class Fn> static uint32_t one(Fn&& f) {
        if (leader()) self.block->shared = f();
        meet();
        return self.block->shared;
    }
};

static GridSync grid_of(uint32_t block, uint32_t blocks, uint32_t limit) {  // as resident_group lays the blocks out
    const uint32_t per = ((blocks + 7) / 8 + 3) / 4 * 4, chunk = block / per;
    return GridSync{words, blocks, chunk, std::min(per, blocks - chunk * per), (blocks + per - 1) / per, 0u, limit};
}

struct Outcome {
    bool open = false;
    uint32_t passed = 0;
};
// a wave of a solve with `barriers` barriers; `arrived` counts the blocks that have come to each
static void solve(GridSync g, uint32_t barriers, std::atomic<uint32_t>* arrived, Outcome& out) {
    out.open = solve_open<Ops>(words);
    if (!out.open) return;
    for (uint32_t k = 0; k < barriers; ++k) {
        if (arrived && Ops::leader()) ++arrived[k];
        if (!grid_sync<Ops>(g)) {
            grid_leave<Ops>(g, true);
            return;
        }
        if (arrived && arrived[k] != g.blocks) wrong("a barrier was passed before every block had come to it");
        ++out.passed;
    }
    if (self.beforeLeave) self.beforeLeave();
    grid_leave<Ops>(g, false);
}

static void run(Block& b, uint32_t waves, std::vector<std::thread>& threads, const std::function<void(uint32_t)>& body) {
    b.waves = waves;
    for (uint32_t w = 0; w < waves; ++w)
        threads.emplace_back([&b, w, body] {
            self.block = &b;
            self.wave = w;
            body(w);
            self.land();
            b.wave_ends();
        });
}
static void join(std::vector<std::thread>& threads) {
    for (auto& t : threads) t.join();
    threads.clear();
}

// Every block there: all barriers are passed, and the words are zero again.
static void all_pass(uint32_t blocks) {
    constexpr uint32_t kBarriers = 4, kWaves = 2;
    std::vector<Block> b(blocks);
    std::vector<Outcome> out(blocks * kWaves);
    std::vector<std::thread> threads;
    std::atomic<uint32_t> arrived[kBarriers] = {};
    for (uint32_t k = 0; k < blocks; ++k)
        run(b[k], kWaves, threads, [&, k](uint32_t w) {
            solve(grid_of(k, blocks, 0xFFFFFFFFu), kBarriers, arrived, out[k * kWaves + w]);
        });
    join(threads);
    for (const Outcome& o : out)
        if (!o.open || o.passed != kBarriers) wrong("a block did not pass every barrier");
    for (uint32_t w : words)
        if (w) wrong("a word was left behind");
}
// A solve so long that the arrivals no longer fit 32 bits between two of its barriers: all of them hold.
static void wrap(uint32_t blocks) {
    constexpr uint32_t kBarriers = 8;
    const uint32_t chunks = grid_of(0, blocks, 0u).chunks, perBarrier = blocks <= kFlatBlocks ? blocks : chunks;
    const uint32_t before = (uint32_t)((1ull << 32) / (2u * perBarrier)) - kBarriers / 2;  // barriers passed so far
    words[kWordArrive] = 2u * perBarrier * before;
    for (uint32_t k = 0; k < blocks; ++k) {
        const GridSync g = grid_of(k, blocks, 0u);
        words[kWordChunk + kLine * g.chunk] = g.chunkBlocks * before;
        words[kWordRelease + kLine * g.chunk] = before;
    }
    std::vector<Block> b(blocks);
    std::vector<Outcome> out(blocks);
    std::vector<std::thread> threads;
    std::atomic<uint32_t> arrived[kBarriers] = {};
    for (uint32_t k = 0; k < blocks; ++k)
        run(b[k], 1, threads, [&, k](uint32_t) {
            GridSync g = grid_of(k, blocks, 0xFFFFFFFFu);
            g.epoch = before;
            solve(g, kBarriers, arrived, out[k]);
        });
    join(threads);
    for (const Outcome& o : out)
        if (o.passed != kBarriers) wrong("a block did not pass every barrier");
}
// No time to wait: blocks give up at barriers that are still open; every wave leaves.
static void no_time(uint32_t blocks) {
    constexpr uint32_t kBarriers = 3, kWaves = 2;
    std::vector<Block> b(blocks);
    std::vector<Outcome> out(blocks * kWaves);
    std::vector<std::thread> threads;
    std::atomic<uint32_t> arrived[kBarriers] = {};
    for (uint32_t k = 0; k < blocks; ++k)
        run(b[k], kWaves, threads, [&, k](uint32_t w) {
            solve(grid_of(k, blocks, 0u), kBarriers, arrived, out[k * kWaves + w]);
        });
    join(threads);
    uint32_t all = 0;
    for (uint32_t k = 0; k < blocks; ++k) {
        if (out[2 * k].open != out[2 * k + 1].open || out[2 * k].passed != out[2 * k + 1].passed)
            wrong("waves of a block went different ways");
        all += out[2 * k].passed == kBarriers;
    }
    if (all && all != blocks) wrong("some blocks passed the last barrier and some did not");
    if ((all == 0) != (words[kResidentAbortedAt] != 0)) wrong("the mark and the outcome differ");
}
// The last block starts when the others have given up: its first look at the mark falls before they set it, every later
// one after.
static void late(uint32_t blocks) {
    constexpr uint32_t kWaves = 4;
    std::vector<Block> b(blocks);
    std::vector<Outcome> out(blocks * kWaves);
    std::vector<std::thread> punctual, last;
    std::mutex m;
    std::condition_variable cv;
    int looks = 0;
    bool others = false;
    const uint32_t k = blocks - 1;
    run(b[k], kWaves, last, [&](uint32_t w) {
        self.afterMark = [&] {
            std::unique_lock<std::mutex> lk(m);
            if (looks++ == 0) {
                cv.notify_all();
                cv.wait(lk, [&] { return others; });
            }
        };
        if (w != 0) {  // another wave looks after wave 0 at the earliest (if it looks at all)
            std::unique_lock<std::mutex> lk(m);
            cv.wait(lk, [&] { return looks > 0; });
        }
        if (w > 1) {
            std::unique_lock<std::mutex> lk(m);
            cv.wait(lk, [&] { return others; });
        }
        solve(grid_of(k, blocks, 2000u), 2, nullptr, out[k * kWaves + w]);
    });
    {
        std::unique_lock<std::mutex> lk(m);
        cv.wait(lk, [&] { return looks > 0; });
    }
    for (uint32_t q = 0; q < k; ++q)
        run(b[q], 1, punctual, [&, q](uint32_t) { solve(grid_of(q, blocks, 2000u), 2, nullptr, out[q * kWaves]); });
    join(punctual);
    {
        std::lock_guard<std::mutex> lk(m);
        others = true;
    }
    cv.notify_all();
    join(last);
    if (!words[kResidentAbortedAt]) wrong("the solve was not marked as aborted");
    for (uint32_t w = 0; w < kWaves; ++w) {
        if (out[k * kWaves + w].open != out[k * kWaves].open) wrong("waves of a block went different ways");
        if (out[k * kWaves + w].passed) wrong("a barrier was passed that nobody had completed");
    }
}

// The block that completes the last barrier is alone in its chunk, so nobody waits for its store to the chunk's release
// word; another block is the last to leave and clears the words.
static void slow_store() {
    constexpr uint32_t kBlocks = 73, kAlone = 72;
    if (grid_of(kAlone, kBlocks, 0u).chunkBlocks != 1u) wrong("the scenario's last chunk has more than one block");
    std::vector<Block> b(kBlocks);
    std::vector<Outcome> out(kBlocks);
    std::vector<std::thread> threads;
    const auto until = [](uint32_t word, uint32_t value) {
        for (;; std::this_thread::yield()) {
            std::lock_guard<std::mutex> lk(mu);
            if (words[word] == value) return;
        }
    };
    for (uint32_t k = 0; k < kBlocks; ++k)
        run(b[k], 1, threads, [&, k](uint32_t) {
            const GridSync g = grid_of(k, kBlocks, 0xFFFFFFFFu);
            if (k == kAlone) {
                until(kWordArrive, 2u * (g.chunks - 1u));
                self.slow = words + kWordRelease + kLine * g.chunk;
            }
            if (k == 0) self.beforeLeave = [&] { until(kWordLeft, kBlocks - 1u); };
            solve(g, 1, nullptr, out[k]);
            if (k == kAlone) until(kWordLeft, 0u);  // and only then its store lands
        });
    join(threads);
    for (uint32_t w : words)
        if (w) wrong("a word was left behind");
}

// Two simulations that keep aborting each other's solves: the limit costs them little of their time.
static void pause() {
    ResidentPause p;
    uint32_t aborts = 0, steps = 0;
    for (; steps < 10000; ++steps) {
        if (p.over()) {
            ++aborts;
            p.aborted();
        } else {
            p.stepped(false);
        }
    }
    if (aborts > 9) wrong("every attempt fails and they are not far enough apart");
    if (aborts * (double)kResidentWait / 100.0 > 0.02 * steps * 300.0)  // us; a launched step takes 300 us and more
        wrong("the barrier's limit costs more than 2% of the steps");
    while (!p.over()) p.stepped(false);
    p.stepped(true);  // one that passes: the next abort is followed by a short pause again
    p.aborted();
    for (uint32_t k = 0; k < ResidentPause::kFirst; ++k) {
        if (p.over()) wrong("a pause shorter than the first");
        p.stepped(false);
    }
    if (!p.over()) wrong("a pause longer than the first");
}

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    const uint32_t blocks = argc > 2 ? (uint32_t)std::atoi(argv[2]) : 1u;
    if (!std::strcmp(what, "all_pass"))
        all_pass(blocks);
    else if (!std::strcmp(what, "no_time"))
        no_time(blocks);
    else if (!std::strcmp(what, "late"))
        late(blocks);
    else if (!std::strcmp(what, "wrap"))
        wrap(blocks);
    else if (!std::strcmp(what, "pause"))
        pause();
    else if (!std::strcmp(what, "recorded")) {  // groups of groupTiles have a CU each wherever they are taken
        for (uint32_t tiles = 0; tiles < 2000; ++tiles)
            for (uint32_t cus : {32u, 64u, 256u, 304u})
                for (uint32_t groupTiles : {1u, 2u, 4u}) {
                    const uint32_t fitting = resident_tiles(tiles, 1, cus), t = recorded_tiles(fitting, groupTiles);
                    const uint32_t most = std::min(cus, 256u);
                    if (t && (t != groupTiles || (tiles + t - 1) / t > most)) wrong("groups that do not fit the CUs");
                    if (!t && tiles && (tiles + groupTiles - 1) / groupTiles <= most) wrong("groups that fit are refused");
                }
    } else if (!std::strcmp(what, "rule")) {  // tiles, scenes, CUs, tiles per group
        if (argc != 6 || resident_tiles(blocks, std::atoi(argv[3]), std::atoi(argv[4])) != (uint32_t)std::atoi(argv[5]))
            wrong("the rule for the groups");
    } else if (!std::strcmp(what, "slow_store"))
        slow_store();
    else
        wrong("unknown scenario");
    std::printf("ok\n");
    return 0;
}
