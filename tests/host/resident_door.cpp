// The protocol by which the workgroups of a resident launch agree (resident_door.h), by threads of the CPU: one thread per
// workgroup, each arriving when it likes or not at all. Whatever the order, everyone comes back, everyone that takes part
// agrees on who does, and nobody waits for one that has not arrived.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

#define __host__
#define __device__
#define __forceinline__ inline
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) __atomic_load_n(p, order)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)
#define __hip_atomic_fetch_add(p, v, order, scope) __atomic_fetch_add(p, v, order)
#define __hip_atomic_fetch_or(p, v, order, scope) __atomic_fetch_or(p, v, order)
#define __hip_atomic_compare_exchange_strong(p, e, v, ok, no, scope) __atomic_compare_exchange_n(p, e, v, false, ok, no)
static unsigned long long wall_clock64() {   // 10 ns
    std::this_thread::yield();
    return (unsigned long long)(std::chrono::steady_clock::now().time_since_epoch().count() / 10);
}
#include "resident_door.h"

using namespace hipc;
namespace {

constexpr int kThreads = 24;
constexpr unsigned long long kTicks = 200000;   // 2 ms: the threads of a loaded machine

void expect(bool ok, const char *what, int trial) {
    if (ok) return;
    std::printf("FAILED: trial %d: %s\n", trial, what);
    std::exit(1);
}

// when[g]: microseconds until workgroup g arrives, < 0: only when everyone else has left
template <typename Body>
void arrive(const std::vector<int> &when, Body &&body) {
    std::vector<std::thread> pool;
    std::atomic<int> left{0};
    int early = 0;
    for (int w : when) early += w >= 0;
    for (int g = 0; g < (int)when.size(); g++)
        pool.emplace_back([&, g] {
            if (when[g] >= 0) std::this_thread::sleep_for(std::chrono::microseconds(when[g]));
            else while (left < early) std::this_thread::yield();
            body(g);
            left++;
        });
    for (std::thread &t : pool) t.join();
}

// the launch of all: `begins` where everyone comes in time
void all(const std::vector<int> &when, bool begins, int trial) {
    const unsigned long long ticks = begins ? 1000 * kTicks : kTicks;
    std::vector<uint32_t> words(kResSyncWords, 0), got(when.size(), 0);
    arrive(when, [&](int g) {
        __atomic_store_n(&words[kResFlags + g], 1u, __ATOMIC_RELAXED);
        if (g) {
            int tries = 1 << 30;
            got[g] = res_await(words.data(), 2 * ticks, tries);
            return;
        }
        const unsigned long long t0 = wall_clock64();
        const bool taken = res_take(words.data());
        bool here;
        do {
            here = true;
            for (size_t i = 0; i < when.size(); i++) here &= res_look(&words[kResFlags + i]) == 1u;
        } while (!here && wall_clock64() - t0 < ticks);
        got[g] = here && taken ? res_decision(kResGroups, true) : res_decision(0, false);
        if (taken) __atomic_store_n(&words[kResDecision], got[g], __ATOMIC_RELAXED);
    });
    for (uint32_t d : got) {
        expect(d & kResDecided, "no decision", trial);
        expect(d == got[0], "two decisions", trial);
    }
    expect(res_decided_for(got[0]) == (begins ? kResGroups : 0u), begins ? "everyone came and it did not begin" : "it began without one", trial);
}

// the stand-in: at least `least` take part
void some(const std::vector<int> &when, int least, int trial) {
    std::vector<uint32_t> words(kResSyncWords, 0), rank(when.size(), 0), n(when.size(), 0);
    arrive(when, [&](int g) {
        int tries = 1 << 30;
        rank[g] = res_join(words.data(), (uint32_t)when.size(), kTicks, &n[g], tries);
    });
    uint32_t in = 0;
    for (size_t g = 0; g < when.size(); g++) {
        if (rank[g] == kResNoRank) continue;
        in++;
        for (size_t o = 0; o < g; o++) expect(rank[o] != rank[g], "one rank twice", trial);
    }
    expect((int)in >= least, "too few take part", trial);
    for (size_t g = 0; g < when.size(); g++) {
        if (rank[g] == kResNoRank) continue;
        expect(n[g] == in, "not as many as were told", trial);
        expect(rank[g] < in, "a rank past the last", trial);
    }
}

}  // namespace

int main() {
    std::mt19937 rng(5);
    auto soon = [&] {
        std::vector<int> w(kThreads);
        for (int &v : w) v = (int)(rng() % 50);
        return w;
    };
    for (int trial = 0; trial < 40; trial++) {
        some(soon(), 1, trial);
        std::vector<int> w = soon();
        w[0] = -1;                      // workgroup 0 finds no room until the others have left
        all(w, false, trial);
        some(w, 1, trial);
        w = soon();
        w[1 + rng() % (kThreads - 1)] = -1;   // another one
        all(w, false, trial);
        for (int &v : w)
            if (rng() % 2) v = -1;
        w[rng() % kThreads] = 0;
        some(w, 1, trial);
        all(soon(), true, trial);
    }
    std::vector<int> alone(kThreads, -1);
    alone[7] = 0;
    some(alone, 1, 100);
    std::printf("ok\n");
    return 0;
}
