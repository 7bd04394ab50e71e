// How the workgroups of a resident launch (decode_resident.hip) agree whether it begins and who takes part.
//
// Nobody waits for a workgroup that has not started. The launch of all workgroups begins if workgroup 0, which takes the
// decision when it arrives, sees all of them in time; any other that has waited long enough for workgroup 0 itself settles that
// it does not begin. The launch that stands in for it takes whom it gets: a workgroup draws a ticket, the holder of the first
// (which is on the chip, whichever workgroup that is) closes the door, and a ticket drawn behind a closed door is worth nothing.
// (No other header is needed here: the protocol is also run on the CPU, by threads.)
#pragma once

#include <cstdint>

namespace hipc {

constexpr uint32_t kResXcds = 8, kResRanks = 32, kResGroups = kResXcds * kResRanks;
constexpr uint32_t kResSets = 3;   // sets of exchange words, taken in turn by the layers
// The words: [0] the step's number, then, for the launch of all workgroups and for the one that stands in for it, the decision
// (0: none yet), the tickets drawn and one flag per workgroup, all on lines of their own. The token pick closes the step: it
// counts the number up and takes decisions and tickets back, so no launch finds any that are not its own, however long ago
// that form last ran. (A flag carries the step's number and needs no clearing; no step has the number 0 that flags begin with.)
constexpr uint32_t kResDecision = 0, kResTickets = 32, kResFlags = 64, kResSyncWords = kResFlags + kResGroups;
constexpr uint32_t kResAll = 32, kResSome = kResAll + kResSyncWords, kResSync = kResSome + kResSyncWords;
constexpr uint32_t kResLaunches = kResSets << 26;   // behind the largest number: a multiple of the sets, so that they go on in turn, and 28 bits
constexpr uint32_t kResDecided = 0x80000000u;       // a decision: this, the workgroups that take part, and (bit 0) whether each group of them shares an L2
constexpr uint32_t kResTaken = 1;                   // none yet, but workgroup 0 is there to make it
constexpr uint32_t kResClosed = 0x80000000u;        // of the tickets: none is worth anything any more
constexpr uint32_t kResNoRank = 0xffffu;

__host__ __device__ inline uint32_t res_decision(uint32_t workgroups, bool one_l2) { return kResDecided | (workgroups << 1) | (one_l2 ? 1u : 0u); }
__host__ __device__ inline uint32_t res_decided_for(uint32_t decision) { return (decision & ~kResDecided) >> 1; }
// behind a step: the next one's words
__host__ __device__ inline void res_next_step(uint32_t *sync) {
    sync[0] = sync[0] + 1 == kResLaunches ? kResSets : sync[0] + 1;
    sync[kResAll + kResDecision] = sync[kResSome + kResDecision] = sync[kResSome + kResTickets] = 0;
}

#ifndef HIPC_HOST_MODEL   // (threads of the address model run one after the other: nobody waits)
__device__ __forceinline__ uint32_t res_look(uint32_t *word) { return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// Workgroup 0, when it arrives: whether the decision is its to make (else there is one: the launch does not begin).
__device__ __forceinline__ bool res_take(uint32_t *words) {
    uint32_t none = 0;
    return __hip_atomic_compare_exchange_strong(words + kResDecision, &none, kResTaken, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The other workgroups of the launch of all: the decision. Where workgroup 0 has not arrived within `ticks`, it is that the
// launch does not begin; once it has, it makes one in a time of its own (`tries` polls at most).
__device__ __forceinline__ uint32_t res_await(uint32_t *words, unsigned long long ticks, int &tries) {
    const unsigned long long t0 = wall_clock64();
    uint32_t d;
    bool wait = true;   // for workgroup 0 to arrive
    while (!((d = res_look(words + kResDecision)) & kResDecided)) {
        if (--tries <= 0) return res_decision(0, false);
        if (!wait || d == kResTaken || (tries & 15) || wall_clock64() - t0 < ticks) continue;   // (the clock is as far away as the word)
        uint32_t found = 0;
        if (__hip_atomic_compare_exchange_strong(words + kResDecision, &found, res_decision(0, false), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return res_decision(0, false);
        wait = false;
    }
    return d;
}
// Workgroups of the stand-in: the rank among the *n that take part, kResNoRank for one that comes too late. The first waits
// for `groups`, until nobody has come for `ticks`; the others wait for the first, `tries` times at most.
__device__ __forceinline__ uint32_t res_join(uint32_t *words, uint32_t groups, unsigned long long ticks, uint32_t *n, int &tries) {
    const uint32_t ticket = __hip_atomic_fetch_add(words + kResTickets, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (ticket & kResClosed) return kResNoRank;
    uint32_t d;
    if (ticket == 0) {
        unsigned long long last = wall_clock64();   // when the last one came
        uint32_t here, before = 1;
        while ((here = res_look(words + kResTickets)) < groups) {
            const unsigned long long now = wall_clock64();
            if (here != before) before = here, last = now;
            else if (now - last >= ticks) break;
        }
        d = res_decision(__hip_atomic_fetch_or(words + kResTickets, kResClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), false);
        __hip_atomic_store(words + kResDecision, d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        while (!((d = res_look(words + kResDecision)) & kResDecided))
            if (--tries <= 0) return kResNoRank;
    }
    *n = res_decided_for(d);
    return ticket;
}
#endif

}  // namespace hipc
